"""The carbonate solve at the edges of its dispatch: the reference's solver
settings (an FP32 guess refined in FP64) with carbon and alkalinity from none
to far above the ocean's, no salt, cold and warm water; a carbon below zero
and other settings (the damped Newton); against the oracle's damped Newton,
whose steps onto 0 end in NaN at some of the alkalinities without salt, as
the last bits fall: points where it or a last-bit neighbour does are left out.

Bounds: H is the root of a sum whose terms are rounded to 2^-53 of the
alkalinity, and away from the endpoints' buffer minima its relative error is
below a hundred of those: 1e-12 in pH.  The flux is k (pCO2 - pCO2_air), so
its error is measured against |F| + k pCO2_air (the flux at DIC = 0)."""
import itertools

import numpy as np
import pytest

import oracle as O

from oceanbiome import abi, workloads
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

CARBON = [0.0, 5.0, 2000.0, 8000.0]
ALKALINITY = [10.0, 300.0, 2400.0, 9000.0]
WATER = [(-1.8, 35.0), (5.0, 0.0), (18.0, 1e-3), (33.0, 41.0)]
SOLVERS = {"reference": {}, "other damping": dict(damping=0.7), "other start": dict(initial_pH_guess=7.25),
           "other descent": dict(armijo_constant=0.1)}


def points(settings):
    q = list(itertools.product(CARBON, ALKALINITY, WATER))
    q += [(-10.0, 2400.0, (10.0, 35.0))]
    DIC, Alk, T, S = (np.array(v, dtype=np.float64) for v in
                      ([x[0] for x in q], [x[1] for x in q], [x[2][0] for x in q], [x[2][1] for x in q]))
    cfg = workloads.lobster_3d(4, 4, 4, nsteps=1).bgc.config(abi.OBME_FP64)
    for k, v in settings.items():
        assert getattr(cfg.solver, k) != v
        setattr(cfg.solver, k, v)
    return cfg, DIC, Alk, T, S, np.full(DIC.size, 7.0)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("solver", SOLVERS)
def test_carbonate_edges(solver, mode):
    import torch
    print("case carbonate edges", solver, mode, flush=True)
    cfg, *pts = points(SOLVERS[solver])
    air = 413.0
    pH_ref, F_ref = O.co2_flux_batch(cfg.co2, cfg.solver, *pts, air)
    none = [np.zeros_like(pts[0]), np.full_like(pts[1], 10.0)] + pts[2:]
    scale = np.abs(F_ref) + np.abs(O.co2_flux_batch(cfg.co2, cfg.solver, *none, air)[1])
    wl = workloads.lobster_3d(4, 4, 4, nsteps=1)
    real = wl.bgc.config
    wl.bgc.config = lambda *a, **k: _with(real(*a, **k), SOLVERS[solver])
    dev = HIPBiogeochemistry(wl.bgc, "fp64")
    pH, F = dev.co2_flux(*[torch.from_numpy(p).cuda() for p in pts], pCO2_air=air, mode=mode)
    pH, F = pH.cpu().numpy(), F.cpu().numpy()
    ok = np.isfinite(pH_ref)
    for e in (1 + 4e-16, 1 - 4e-16):
        ok &= np.isfinite(O.co2_flux_batch(cfg.co2, cfg.solver, pts[0] * e, pts[1] * (2 - e), *pts[2:], air)[0])
    assert ok.sum() > 50
    print("pH", np.nanmax(np.abs(pH - pH_ref)), "flux", np.nanmax(np.abs(F - F_ref) / scale), flush=True)
    assert np.max(np.abs(pH - pH_ref)[ok]) <= 1e-12
    assert np.max((np.abs(F - F_ref) / scale)[ok]) <= 1e-11


def _with(cfg, settings):
    for k, v in settings.items():
        setattr(cfg.solver, k, v)
    return cfg
