"""What the ensemble says of its packing is what its launches have: every column
in one of them, in enough waves to hold its lanes and not twice as many; and the
autotuner keeps plans that differ (0, 1 and 2 pack every ensemble alike, and 4
and 6; of shallow columns 3 as 4)."""
import re

import numpy as np
import pytest

from oceanbiome import workloads
from oceanbiome.runtime import HIPBatch

pytestmark = pytest.mark.gpu


def _launches(text):
    head, tail = text.split(" launches: ")
    plan = int(re.fullmatch(r"plan (\d) steps_per_launch \d+", head).group(1))
    found = [re.fullmatch(r"(\d) per lane, (\d+) columns in (\d+) waves( by rows)?", x) for x in tail.split("; ")]
    return plan, [tuple(int(v) for v in m.groups()[:3]) for m in found]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("deepest", [16, 64, 128])
def test_describe_and_autotune(deepest, precision):
    import torch
    print("case batch describe", deepest, precision, flush=True)
    wl = workloads.npzd_columns(n_columns=3000, nz_min=1, nz_max=deepest, nsteps=4)
    off = wl.extra["offsets"]
    nz = np.diff(off)
    b = HIPBatch(wl.bgc, off, wl.extra["params"], wl.extra["dz"], wl.extra["T"], precision)
    for plan in range(7):
        b.configure(plan, 0)
        got, launches = _launches(b.describe())
        assert got == plan
        assert sum(n for _, n, _ in launches) == 3000
        for L, n, waves in launches:
            assert n <= 64 * waves <= 64 * (2 * n + 4)
        lanes = sum(-(-nz // min(L for L, _, _ in launches)))
        assert 64 * sum(w for _, _, w in launches) <= 2 * lanes + 1024
    tr = [torch.from_numpy(a).to(device="cuda", dtype=b.dtype) for a in wl.tracers]
    for _ in range(4):
        b.autotune(tr, 2, wl.dt)
        assert _launches(b.describe())[0] in ((0, 3, 5) if deepest == 16 else (0, 3, 4, 5))
