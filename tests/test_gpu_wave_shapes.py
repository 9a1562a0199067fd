"""The kernels with a column's levels along the lanes where a lane holds two or
four levels and a wave several columns, which wave_shape chooses on grids of
some thousand columns: FP32 of 40 levels (two per lane, three columns per wave)
and 75 (four, three), FP64 of 40 and 47 (two per lane), in the last wave part
filled; the schemes, the scaling with the CO2 flux and the sediment with two
levels per lane (its bottom level the first or the second of a lane); against the
oracle, on every 37th column.  And a NaN stays in its column."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device
from oceanbiome import abi
from oceanbiome.grid import RectilinearGrid
from oceanbiome.models import (LOBSTER, NPZD, CarbonateSystem, CarbonDioxideGasExchangeBoundaryCondition,
                               InstantRemineralisationSediment, Oxygen, TwoBandPhotosyntheticallyActiveRadiation)
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}
LIGHT = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0)


def _model(kind, shape, sediment=False):
    Nx, Ny, Nz = shape
    z = (-200.0, 0.0)
    if kind == "stretched":
        z = [-200.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)]
    grid = RectilinearGrid(size=shape, x=(0.0, 10.0 * Nx), y=(0.0, 10.0 * Ny), z=z, halo=(1, 1, 3))
    if kind == "npzd":
        sed = InstantRemineralisationSediment(grid) if sediment else None
        bgc = NPZD(grid, light_attenuation=LIGHT, oxygen=Oxygen(), sediment_model=sed)
        medians = (2.5, 0.1, 0.05, 12.0, 0.5, 250.0)
    else:
        sed = InstantRemineralisationSediment(sinking_tracers=("sPOM", "bPOM"),
                                              remineralisation_reciever="NH₄") if sediment else None
        bgc = LOBSTER(grid, carbonate_system=None if kind == "plain" else CarbonateSystem(), light_attenuation=LIGHT,
                      sinking_scheme=kind if kind in ("weno5", "centered") else "upwind",
                      gas_exchange=None if kind == "plain" else CarbonDioxideGasExchangeBoundaryCondition(),
                      temperature=12.0, salinity=35.0, scale_negatives=kind == "scaled", sediment_model=sed)
        medians = (10.0, 0.1, 0.1, 0.1, 0.5, 0.5, 0.05) + (() if kind == "plain" else (2100.0, 2320.0))
    rng = np.random.default_rng(Nx + Nz)
    fields = []
    for q, m in enumerate(medians):
        f = grid.new_field()
        grid.interior(f)[...] = m * np.exp((0.02 if m > 1000 else 0.3) * rng.standard_normal((Nz, Ny, Nx)))
        if kind == "scaled" and q == 3:
            grid.interior(f)[rng.random((Nz, Ny, Nx)) < 0.05] *= -0.01
        fields.append(f)
    return bgc, grid, fields


def _columns(shape, every):
    at = np.arange(0, shape[0] * shape[1], every)
    return (at % shape[0]).astype(np.int32), (at // shape[0]).astype(np.int32)


def _compare(bgc, grid, shape, tr, ref, ci, cj, precision, what):
    for name, x, r in zip(bgc.required_biogeochemical_tracers(), tr, ref):
        a = grid.interior(x.double().cpu().numpy())
        b = grid.interior(r)
        e = rel_l2(a[:, cj, ci], b[:, cj, ci])
        assert e <= TOL[precision], (what, shape, name, e)


# 9011 columns: no multiple of the columns of a wave or a workgroup
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["upwind", "stretched", "weno5", "centered", "scaled", "npzd"])
def test_several_levels_per_lane_and_columns_per_wave(kind, precision):
    import torch
    for Nz in ((40, 47) if precision == "fp64" else (40, 75)):
        shape = (9011, 1, Nz)
        print("case wave shapes", kind, precision, shape, flush=True)
        bgc, grid, fields = _model(kind, shape)
        ci, cj = _columns(shape, 37)
        ref = [f.copy() for f in fields]
        O.grid_run_columns(bgc.config(abi.OBME_FP64), ref, ci, cj, 3, 60.0)
        dev = HIPBiogeochemistry(bgc, precision)
        tr = to_device(fields, dev.dtype)
        dev.step(tr, 3, 60.0)
        torch.cuda.synchronize()
        _compare(bgc, grid, shape, tr, ref, ci, cj, precision, kind)


@pytest.mark.parametrize("kind, precision", [("plain", "fp64"), ("upwind", "fp64"), ("scaled", "fp64"),
                                             ("npzd", "fp64"), ("plain", "fp32"), ("upwind", "fp32"),
                                             ("scaled", "fp32")])
def test_sediment(kind, precision):
    import torch
    # FP64: two levels per lane, the bottom level the second (even) or the first (odd) of its lane
    for shape in ((5, 3, 65), (4, 3, 66), (3, 2, 127), (2, 2, 128), (9011, 1, 40)) if precision == "fp64" else \
            ((5, 3, 33), (9, 5, 64), (701, 13, 20)):
        print("case wave shapes sediment", kind, precision, shape, flush=True)
        bgc, grid, fields = _model(kind, shape, sediment=True)
        ref = [f.copy() for f in fields]
        state = O.SedimentState(grid.Nx, grid.Ny)
        dev = HIPBiogeochemistry(bgc, precision)
        tr = to_device(fields, dev.dtype)
        for call in range(2):
            O.grid_run_sediment(bgc.config(abi.OBME_FP64), ref, state, 2, 300.0, t0=600.0 * call)
            dev.step(tr, 2, 300.0, t0=600.0 * call)
        torch.cuda.synchronize()
        ci, cj = _columns(shape, 1)
        _compare(bgc, grid, shape, tr, ref, ci, cj, precision, kind)
        e = rel_l2(dev.sediment_storage.cpu().numpy(), state.storage)
        assert np.all(state.storage > 0) and e <= TOL[precision], (shape, e)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["upwind", "weno5", "scaled"])
def test_nan_stays_in_its_column(kind, precision):
    import torch
    for Nz in ((40,) if precision == "fp64" else (40, 75)):
        shape = (9011, 1, Nz)
        print("case wave shapes nan", kind, precision, shape, flush=True)
        bgc, grid, fields = _model(kind, shape)
        bad = [100, 4567, 9010]
        out = []
        for plant in (False, True):
            fs = [f.copy() for f in fields]
            if plant:
                for f in fs:
                    for q, c in enumerate(bad):
                        grid.interior(f)[(0, Nz // 2, Nz - 1)[q], 0, c] = np.nan
            dev = HIPBiogeochemistry(bgc, precision)
            tr = to_device(fs, dev.dtype)
            dev.step(tr, 2, 60.0)
            torch.cuda.synchronize()
            out.append([grid.interior(t.double().cpu().numpy()).copy() for t in tr])
        for a, b in zip(*out):
            assert np.isnan(b[:, 0, bad]).any()
            a[:, 0, bad] = b[:, 0, bad] = 0.0
            assert np.array_equal(a, b)
