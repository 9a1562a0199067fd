"""The NPZD / LOBSTER step with a column's levels along the lanes of a wave:
column heights around the lane and level counts a wave holds (1, 2 or 4
levels per lane, columns that fill a wave, share one or leave lanes over),
column counts that leave a workgroup part-filled, more steps than one launch
takes, every sinking scheme, the scaling with the CO2 flux and the sediment;
against the oracle.  And a NaN stays in its column."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device, to_host
from oceanbiome import abi, workloads
from oceanbiome.grid import RectilinearGrid
from oceanbiome.models import (LOBSTER, NPZD, CarbonateSystem, CarbonDioxideGasExchangeBoundaryCondition, Oxygen,
                               TwoBandPhotosyntheticallyActiveRadiation)
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}
# (Nx, Ny, Nz): lanes per column 1 .. 64, the sweep beyond
SHAPES = [(3, 2, 2), (7, 5, 16), (5, 3, 17), (130, 1, 32), (9, 7, 33), (3, 3, 63), (11, 6, 64), (5, 4, 65), (4, 3, 75),
          (3, 2, 128), (2, 3, 129), (2, 2, 256), (2, 1, 257)]


def _model(kind, shape):
    Nx, Ny, Nz = shape
    z = (-200.0, 0.0)
    if kind == "stretched":
        z = [-200.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)]
    grid = RectilinearGrid(size=shape, x=(0.0, 10.0 * Nx), y=(0.0, 10.0 * Ny), z=z, halo=(3, 3, 3))
    light = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR="default" if kind == "stretched" else 100.0)
    rng = np.random.Generator(np.random.PCG64(Nx + 100 * Ny + 10000 * Nz))
    if kind == "npzd":
        bgc = NPZD(grid, light_attenuation=light, oxygen=Oxygen())
        medians = (2.5, 0.1, 0.05, 12.0, 0.05, 250.0)
    else:
        scheme = kind if kind in ("weno5", "centered") else "upwind"
        bgc = LOBSTER(grid, carbonate_system=CarbonateSystem(), light_attenuation=light, sinking_scheme=scheme,
                      gas_exchange=CarbonDioxideGasExchangeBoundaryCondition(), temperature=20 - 0.05 * np.abs(grid.zc),
                      salinity=35.0, scale_negatives=kind == "scaled")
        medians = (10.0, 0.1, 0.1, 0.1, 0.05, 0.05, 0.05, 2100.0, 2320.0)
    fields = []
    for q, m in enumerate(medians):
        f = grid.new_field()
        grid.interior(f)[...] = m * np.exp((0.02 if m > 1000 else 0.3) * rng.standard_normal((Nz, Ny, Nx)))
        if kind == "scaled" and q == 3:
            grid.interior(f)[rng.random((Nz, Ny, Nx)) < 0.05] *= -0.01
        fields.append(f)
    return bgc, grid, fields


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["upwind", "stretched", "weno5", "centered", "scaled", "npzd"])
def test_step_against_the_oracle(kind, precision):
    import torch
    for shape in SHAPES:
        print("case wave step", kind, precision, shape, flush=True)
        bgc, grid, fields = _model(kind, shape)
        nsteps, dt = (18 if shape == (7, 5, 16) else 3), 60.0
        ref = [f.copy() for f in fields]
        O.grid_run(bgc.config(abi.OBME_FP64), ref, nsteps, dt, nthreads=4)
        dev = HIPBiogeochemistry(bgc, precision)
        tr = to_device(fields, dev.dtype)
        dev.step(tr, nsteps, dt)
        torch.cuda.synchronize()
        for name, x, r, f in zip(bgc.required_biogeochemical_tracers(), to_host(tr), ref, fields):
            e = rel_l2(grid.interior(x), grid.interior(r))
            assert e <= TOL[precision], (shape, name, e)
            x, f = x.copy(), f.astype(np.float32 if precision == "fp32" else np.float64).astype(np.float64)
            grid.interior(x)[...] = grid.interior(f)
            assert np.array_equal(x, f), "a halo was written"


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_nan_stays_in_its_column(precision):
    """Columns share waves (and a wave's prefix sums): a NaN in one leaves the
    bits of the others as they are without it."""
    import torch
    for kind, shape in (("upwind", (9, 3, 17)), ("weno5", (9, 3, 20)), ("upwind", (9, 3, 64))):
        print("case wave nan", kind, precision, shape, flush=True)
        bgc, grid, fields = _model(kind, shape)
        out = []
        for bad in (False, True):
            fs = [f.copy() for f in fields]
            if bad:
                for f in fs:
                    grid.interior(f)[shape[2] // 2, 1, 4] = np.nan
            dev = HIPBiogeochemistry(bgc, precision)
            tr = to_device(fs, dev.dtype)
            dev.step(tr, 2, 60.0)
            torch.cuda.synchronize()
            out.append(to_host(tr))
        for x, y in zip(*out):
            a, b = grid.interior(x).copy(), grid.interior(y).copy()
            assert np.isnan(b[:, 1, 4]).any()
            a[:, 1, 4] = b[:, 1, 4] = 0.0
            assert np.array_equal(a, b)
