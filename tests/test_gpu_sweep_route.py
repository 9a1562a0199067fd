"""The column sweep where the dispatch keeps it: single steps of more than 40960
columns, the tendency hook of more than 32768, and every step of formulations
other than the defaults.  Rows that end inside a wave and column counts that fill
the last workgroup of every width or do not, against the oracle, with the same
bits from 1, 2, 4 and 8 waves per workgroup, and nothing outside the interior
written."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device, to_host
from oceanbiome import abi
from oceanbiome.grid import RectilinearGrid
from oceanbiome.models import (LOBSTER, NPZD, CarbonateSystem, CarbonDioxideGasExchangeBoundaryCondition, Linear, Oxygen,
                               OxygenGasExchangeBoundaryCondition, TwoBandPhotosyntheticallyActiveRadiation)
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}
# (Nx, Ny, Nz): columns that leave the last workgroup part-filled (a row of 333
# ends inside a wave), that fill it for every width, one level, two
SHAPES = [(333, 127, 5), (320, 160, 6), (257, 161, 2), (4096, 12, 1)]
KINDS = ["lobster", "full", "npzd", "forms"]


def _model(kind, shape):
    Nx, Ny, Nz = shape
    z = (-60.0, 0.0)
    if kind == "full":
        z = [-60.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)]
    grid = RectilinearGrid(size=shape, x=(0.0, 10.0 * Nx), y=(0.0, 10.0 * Ny), z=z, halo=(3, 3, 3))
    rng = np.random.default_rng(Nx + Nz)
    T = S = None
    if kind == "npzd":
        bgc = NPZD(grid, light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0))
        medians = (2.5, 0.1, 0.05, 12.0, 0.05)
    elif kind == "full":
        # every component, the daily cycle, a stretched grid, T and S of the host
        bgc = LOBSTER(grid, carbonate_system=CarbonateSystem(), oxygen=Oxygen(),
                      gas_exchange=(CarbonDioxideGasExchangeBoundaryCondition(), OxygenGasExchangeBoundaryCondition()))
        medians = (10.0, 0.1, 0.1, 0.1, 0.05, 0.05, 0.05, 2100.0, 2320.0, 250.0)
        T, S = grid.new_field(), grid.new_field()
        grid.interior(T)[...] = rng.uniform(5.0, 25.0, (Nz, Ny, Nx))
        grid.interior(S)[...] = rng.uniform(33.0, 37.0, (Nz, Ny, Nx))
    else:
        bgc = LOBSTER(grid, carbonate_system=CarbonateSystem(), temperature=15.0, salinity=35.0,
                      gas_exchange=CarbonDioxideGasExchangeBoundaryCondition(),
                      light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0))
        if kind == "forms":
            bgc.plankton.phytoplankton_mortality_formulation = Linear
        medians = (10.0, 0.1, 0.1, 0.1, 0.05, 0.05, 0.05, 2100.0, 2320.0)
    fields = []
    for m in medians:
        f = grid.new_field()
        grid.interior(f)[...] = m * np.exp((0.02 if m > 1000 else 0.3) * rng.standard_normal((Nz, Ny, Nx)))
        fields.append(f)
    return bgc, grid, fields, T, S


def _untouched(grid, x, f, precision):
    x, f = x.copy(), f.astype(np.float32 if precision == "fp32" else np.float64).astype(np.float64)
    grid.interior(x)[...] = grid.interior(f)
    assert np.array_equal(x, f), "a halo was written"


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("kind", KINDS)
def test_single_steps(kind, shape, precision):
    import torch
    print("case sweep route step", kind, shape, precision, flush=True)
    bgc, grid, fields, T, S = _model(kind, shape)
    cfg = bgc.config(abi.OBME_FP64)
    ref = [f.copy() for f in fields]
    for s in range(2):
        O.grid_run(cfg, ref, 1, 300.0, t0=300.0 * s, T3=T, S3=S)
    first = None
    for waves in (1, 2, 4, 8):
        dev = HIPBiogeochemistry(bgc, precision)
        dev.configure_sweep(waves)
        tr = to_device(fields, dev.dtype)
        TS = [None if x is None else to_device([x], dev.dtype)[0] for x in (T, S)]
        for s in range(2):
            dev.step(tr, 1, 300.0, t0=300.0 * s, T=TS[0], S=TS[1])
        torch.cuda.synchronize()
        out = to_host(tr)
        if first is None:
            first = out
            for name, x, r, f in zip(bgc.required_biogeochemical_tracers(), out, ref, fields):
                e = rel_l2(grid.interior(x), grid.interior(r))
                assert e <= TOL[precision], (name, e)
                _untouched(grid, x, f, precision)
        for n, (x, y) in enumerate(zip(first, out)):
            assert np.array_equal(x, y), (waves, n)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("kind", KINDS)
def test_tendency_hook(kind, shape, precision):
    import torch
    print("case sweep route hook", kind, shape, precision, flush=True)
    bgc, grid, fields, T, S = _model(kind, shape)
    rng = np.random.default_rng(3)
    G0 = [rng.standard_normal(grid.parent_shape) * 1e-6 for _ in fields]
    want = [a.copy() for a in G0]
    PAR_ref = grid.new_field()
    O.grid_tendencies(bgc.config(abi.OBME_FP64), fields, want, 40000.0, T3=T, S3=S, PAR=PAR_ref)
    first = None
    for waves in (1, 2, 4, 8):
        dev = HIPBiogeochemistry(bgc, precision)
        dev.configure_sweep(waves)
        tr, G = to_device(fields, dev.dtype), to_device(G0, dev.dtype)
        G0r = to_host(G)
        TS = [None if x is None else to_device([x], dev.dtype)[0] for x in (T, S)]
        PAR = torch.full(grid.parent_shape, -7.0, dtype=dev.dtype, device="cuda")
        dev.update_tendencies(tr, G, PAR, T=TS[0], S=TS[1], t=40000.0)
        torch.cuda.synchronize()
        out = to_host(G + [PAR])
        if first is None:
            first = out
            for name, a, b, a0, a0r in zip(bgc.required_biogeochemical_tracers(), out, want, G0, G0r):
                e = rel_l2(grid.interior(a - a0r), grid.interior(b - a0))
                assert e <= TOL[precision], (name, e)
                _untouched(grid, a, a0r, precision)
            assert rel_l2(grid.interior(out[-1]), grid.interior(PAR_ref)) <= (1e-13 if precision == "fp64" else 1e-5)
            assert np.count_nonzero(out[-1] == -7.0) == out[-1].size - np.prod(shape)
        for n, (x, y) in enumerate(zip(first, out)):
            assert np.array_equal(x, y), (waves, n)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_several_steps_of_other_formulations(precision):
    """Five steps in a call and one by one after it: the residuals and the warm
    starts from launch to launch."""
    import torch
    print("case sweep route forms", precision, flush=True)
    bgc, grid, fields, _, _ = _model("forms", (45, 20, 33))
    ref = [f.copy() for f in fields]
    O.grid_run(bgc.config(abi.OBME_FP64), ref, 7, 300.0)
    dev = HIPBiogeochemistry(bgc, precision)
    tr = to_device(fields, dev.dtype)
    dev.step(tr, 5, 300.0)
    for s in (5, 6):
        dev.step(tr, 1, 300.0, t0=300.0 * s)
    torch.cuda.synchronize()
    for name, x, r in zip(bgc.required_biogeochemical_tracers(), to_host(tr), ref):
        assert rel_l2(grid.interior(x), grid.interior(r)) <= TOL[precision], name
