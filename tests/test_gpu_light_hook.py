"""The light hook at the edges of its blocks of columns and chunks of levels,
and on both sides of the line between its kernel and the sweep's (FP64, 65536
columns), on uniform and stretched grids, against the oracle; the bounds are
those of the other PAR tests, 1e-13 in FP64 and 1e-5 in FP32-mixed, and
nothing outside the interior is written."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device
from oceanbiome import NPZD, RectilinearGrid, abi
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 2), (5, 1, 8), (31, 3, 9), (64, 1, 64), (33, 2, 65), (3, 5, 130), (257, 256, 5), (256, 256, 5)]
TOL = {"fp64": 1e-13, "fp32": 1e-5}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("stretched", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_light_hook(shape, stretched, precision):
    import torch
    print("case light hook", shape, stretched, precision, flush=True)
    Nx, Ny, Nz = shape
    z = [-100.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)] if stretched else (-100.0, 0.0)
    g = RectilinearGrid(size=shape, x=(0.0, 1.0 * Nx), y=(0.0, 1.0 * Ny), z=z)
    bgc = NPZD(g)
    rng = np.random.default_rng(Nx + Nz)
    tracers = []
    for _ in range(5):
        f = g.new_field()
        g.interior(f)[...] = rng.uniform(0.01, 2.0, (Nz, Ny, Nx))
        tracers.append(f)
    ref = g.new_field()
    O.grid_update_state(bgc.config(abi.OBME_FP64), tracers, ref, 0.0)
    dev = HIPBiogeochemistry(bgc, precision)
    tr = to_device(tracers, dev.dtype)
    PAR = torch.full(g.parent_shape, -7.0, dtype=dev.dtype, device="cuda")
    dev.update_biogeochemical_state(tr, PAR, 0.0)
    torch.cuda.synchronize()
    out = PAR.double().cpu().numpy()
    assert rel_l2(g.interior(out), g.interior(ref)) <= TOL[precision]
    assert np.count_nonzero(out == -7.0) == out.size - Nx * Ny * Nz
