"""The packing of the ensemble's columns into waves at its edges: columns of
one level, odd depths, columns that fill a wave exactly or one lane less,
more small ones than a workgroup takes, in every plan (one, two and four
levels per lane), against the oracle's column runs; the bounds are those of
the other ensemble tests (FP64 1e-12, FP32-mixed 1e-5, per column too), and
formulations other than the defaults."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2
from oceanbiome import InstantRemineralisationSediment, abi, workloads
from oceanbiome.models import Quadratic
from oceanbiome.runtime import HIPBatch

pytestmark = pytest.mark.gpu

DEPTHS = {
    "one column": [1],
    "small": [1, 2, 3] * 90,
    "full waves": [64, 63, 62, 1, 33, 32, 31],
    "deep": [128, 127, 126, 125, 1, 2, 3, 65, 64, 63, 97, 31],
}
TOL = {"fp64": 1e-12, "fp32": 1e-5}


def _ensemble(depths, seed=3):
    wl = workloads.npzd_columns(n_columns=len(depths), nz_min=128, nz_max=128, nsteps=4, seed=seed)
    keep = np.concatenate([128 * c + np.arange(128 - n, 128) for c, n in enumerate(depths)])
    wl.tracers = [np.ascontiguousarray(t[keep]) for t in wl.tracers]
    wl.extra["offsets"] = np.concatenate([[0], np.cumsum(depths)]).astype(np.int64)
    return wl


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("forms", ["default", "other"])
@pytest.mark.parametrize("name", DEPTHS)
def test_packing(name, forms, precision):
    import torch
    print("case batch packing", name, forms, precision, flush=True)
    depths = DEPTHS[name]
    wl = _ensemble(depths)
    if forms == "other":
        wl.bgc.plankton.phytoplankton_mortality_formulation = Quadratic
    sediment = precision == "fp64" and name == "deep"
    if sediment:
        wl.bgc.sediment = InstantRemineralisationSediment(sinking_tracers=("P", "D"), remineralisation_reciever="N")
    off = wl.extra["offsets"]
    ref = [a.copy() for a in wl.tracers]
    state = O.SedimentState(len(depths), 1) if sediment else None
    O.batch_run(wl.bgc.config(abi.OBME_FP64), off, list(wl.extra["params"]), wl.extra["dz"], wl.extra["T"], ref,
                wl.nsteps, wl.dt, sediment=state)
    ran = 0
    for plan in range(7):
        b = HIPBatch(wl.bgc, off, wl.extra["params"], wl.extra["dz"], wl.extra["T"], precision)
        try:
            b.configure(plan, 0)
        except Exception:          # a plan without a tile for the deepest column
            assert max(depths) > 64
            continue
        tr = [torch.from_numpy(a).to(device="cuda", dtype=b.dtype) for a in wl.tracers]
        if sediment:
            b.step(tr, wl.nsteps, wl.dt)
            assert rel_l2(b.sediment_storage.cpu().numpy().ravel(), state.storage.ravel()) <= TOL[precision]
        else:
            b.step(tr, wl.nsteps, wl.dt)
        for a, r in zip(tr, ref):
            a = a.double().cpu().numpy()
            assert rel_l2(a, r) <= TOL[precision], plan
            for c in range(len(depths)):
                s = slice(off[c], off[c + 1])
                assert rel_l2(a[s], r[s]) <= 10 * TOL[precision], (plan, c)
        ran += 1
    assert ran
