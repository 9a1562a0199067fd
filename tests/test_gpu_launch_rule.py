"""A call of several steps of a large grid takes the kernel with several steps per
launch only where a launch has room for several: with the scratch of
obme_step_noalloc filled up by T and S of 360000 columns (FP64: 313600) a launch takes one
step, which is the column sweep's.

In the dark (PAR0 = 0) a negative chlorophyll attenuation, whose logarithm the
other kernel would need, leaves a handle to the sweep and changes nothing else:
the results are the same to the bit."""
import numpy as np
import pytest

from helpers import to_device
from oceanbiome import workloads
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, Nx, Ny", [("fp32", 600, 600), ("fp64", 560, 560)])
def test_one_record_takes_the_sweep(precision, Nx, Ny):
    import torch
    print("case launch rule", precision, flush=True)
    wl = workloads.lobster_3d(Nx, Ny, 3, surface_PAR=0.0)
    g = wl.grid
    T = torch.full(g.parent_shape, 15.0, dtype=torch.float64 if precision == "fp64" else torch.float32, device="cuda")
    S = torch.full_like(T, 35.0)
    out = []
    for sweep in (False, True):
        wl.bgc.light_attenuation.chlorophyll_red_attenuation = -0.037 if sweep else 0.037
        dev = HIPBiogeochemistry(wl.bgc, precision)
        tr = to_device(wl.tracers, dev.dtype)
        dev.step_noalloc(tr, 3, 600.0, T=T, S=S)
        torch.cuda.synchronize()
        out.append([t.cpu().numpy() for t in tr])
    for n, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), n
