"""The fused FP32-mixed PISCES step on columns of two waves (65 to 128 levels)
against the numpy FP64 oracle at its edges (one level in the lower wave, all of
them, an odd number of columns a row; grids so deep that the euphotic depth and
the mixed layer end in the upper wave, the lower one or between them), with the
gas exchange and the negative scaling; several steps per launch against one, bit
for bit; and the per-stage kernels above 128 levels.  Bar: that of the fused
step, relative L2 <= 1e-5 per tracer, inputs around the reference's test values."""
import numpy as np
import pytest

import pisces as OP
from helpers import rel_l2
from oceanbiome import pisces as HP
from oceanbiome import workloads
from test_gpu_pisces_fused import TOL, _device_run, _oracle_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nz,Lz,gas,scale", [(65, 1000.0, False, False), (66, 300.0, True, False),
                                             (97, 200.0, True, True), (128, 150.0, False, True),
                                             (128, 260.0, True, False), (127, 60.0, False, False), (120, 400.0, False, False),
                                             (129, 1000.0, False, False)])
def test_deep_fused_step_against_oracle(Nz, Lz, gas, scale):
    print("case pisces fused deep", Nz, Lz, "gas", gas, "scale", scale, flush=True)
    wl = workloads.pisces_3d(7, 3, Nz, nsteps=2, dt=300.0, seed=17, Lz=Lz, medians="test")
    wl.bgc = HP.PISCES(wl.grid, co2_exchange=gas, o2_exchange=gas, scale_negatives=scale)
    q, light, F, zc, zf, dz, solver = _oracle_inputs(wl)
    cfg = wl.bgc.config(0)
    kw = {}
    if gas:
        kw["gas"] = {"co2": cfg.co2, "o2": cfg.o2}
    if scale:
        kw["scaling"] = OP.conserved_groups(q)
    for c in range(2):
        OP.step(q, light, F, zc, zf, dz, wl.nsteps, wl.dt, c * wl.nsteps * wl.dt, solver, **kw)
    out = _device_run(wl, 2, wl.nsteps)
    g = wl.grid
    errs = {name: rel_l2(g.interior(out[n]), F[name]) for n, name in enumerate(OP.WRITTEN)}
    print("errors", {k: float(v) for k, v in errs.items()}, flush=True)
    assert all(e <= TOL for e in errs.values()), errs
    for n in range(len(OP.WRITTEN)):
        np.testing.assert_array_equal(out[n][0], wl.tracers[n][0].astype(np.float32).astype(np.float64))


def test_deep_fused_matches_per_stage_and_one_step_per_launch():
    print("case pisces fused deep launches", flush=True)
    wl = workloads.pisces_3d(33, 9, 100, nsteps=18, dt=300.0, seed=41, Lz=180.0, medians="test")
    wl.bgc = HP.PISCES(wl.grid, co2_exchange=True, o2_exchange=True, surface_PAR="default")
    a = _device_run(wl, 1, wl.nsteps, t_start=36000.0)
    b = _device_run(wl, 1, wl.nsteps, steps_per_launch=1, t_start=36000.0)
    c = _device_run(wl, 1, wl.nsteps, fused=False, t_start=36000.0)
    g = wl.grid
    for n, name in enumerate(OP.WRITTEN):
        assert np.array_equal(a[n], b[n], equal_nan=True), name
        x, y = g.interior(a[n]), g.interior(c[n])
        ok = np.isfinite(y)
        assert np.array_equal(np.isfinite(x), ok) and rel_l2(x[ok], y[ok]) <= TOL, name
