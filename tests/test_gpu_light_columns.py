"""FP32 light hook of more columns than its kernel takes (163 840), where the
column sweep writes the PAR: workgroups in whole and in part, uniform and
stretched grids, against the oracle on the same tracers; nothing outside the
interior is written.  The bound is that of the other PAR tests, 1e-5."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device
from oceanbiome import NPZD, RectilinearGrid, abi
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stretched", [False, True])
@pytest.mark.parametrize("Nx, Ny", [(512, 321), (409, 401)])
def test_light_hook_of_many_columns(Nx, Ny, stretched):
    import torch
    print("case light columns", Nx, Ny, stretched, flush=True)
    Nz = 9
    z = [-100.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)] if stretched else (-100.0, 0.0)
    g = RectilinearGrid(size=(Nx, Ny, Nz), x=(0.0, 1.0 * Nx), y=(0.0, 1.0 * Ny), z=z)
    bgc = NPZD(g)
    rng = np.random.default_rng(Nx)
    fields = []
    for m in (2.0, 0.5, 0.05, 12.0, 0.05):
        f = g.new_field()
        g.interior(f)[...] = np.float32(m * np.exp(0.3 * rng.standard_normal((Nz, Ny, Nx))))
        fields.append(f)
    dev = HIPBiogeochemistry(bgc, "fp32")
    PAR = torch.full(g.parent_shape, -7.0, dtype=dev.dtype, device="cuda")
    dev.update_biogeochemical_state(to_device(fields, dev.dtype), PAR, 3600.0)
    torch.cuda.synchronize()
    got = PAR.double().cpu().numpy()
    ref = np.full(g.parent_shape, -7.0)
    O.grid_update_state(bgc.config(abi.OBME_FP64), fields, ref, 3600.0)
    assert rel_l2(g.interior(got), g.interior(ref)) <= 1e-5
    g.interior(got)[...] = -7.0
    assert np.all(got == -7.0)
