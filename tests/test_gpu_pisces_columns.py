"""The column pass of PISCES (light, euphotic depth, mixed-layer light) and its
saturation state at the edges of the pass's blocks of 16 columns and chunks of
64 levels, against the oracle: written into the interiors of the caller's
parent arrays, all of them and one at a time.  Bounds: those of the light
fields elsewhere, 1e-13 in FP64 and 1e-5 in FP32-mixed, and 1e-12 for Ω."""
import ctypes as C

import numpy as np
import pytest

import pisces as OP
from helpers import rel_l2
from oceanbiome import workloads
from oceanbiome.runtime import HIPPISCES, library

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 2), (7, 3, 63), (16, 1, 64), (17, 2, 65), (5, 5, 129)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_column_pass(precision, shape):
    import torch
    print("case pisces columns", precision, shape, flush=True)
    wl = workloads.pisces_3d(*shape, nsteps=1, seed=4, medians="test")
    g, m = wl.grid, wl.bgc
    light = dict(surface_PAR=m.surface_PAR, kw=m.kw, e=m.e, chi=m.chi, division=m.division)
    F = {n: g.interior(a).copy() for n, a in zip(OP.TRACERS, wl.tracers)}
    solver = m.carbon_chemistry.solver.struct(m.carbon_chemistry.initial_pH_guess)
    A = OP.update_state(OP.params_from_vector(m.param_vector()), light, F, np.asarray(g.zc), np.asarray(g.zf), 0.0, solver)
    want = [A["PAR"], A["PAR1"], A["PAR2"], A["PAR3"], A["Omega"], A["zeu"][0], A["mlPAR"][0]]
    if precision == "fp32":
        # below FP32's least normal number (the red band over two levels of
        # kilometres) the output type holds no digits to compare
        want = [np.where(np.abs(w) < np.finfo(np.float32).tiny, 0.0, w) for w in want]
    dev = HIPPISCES(m, precision)
    tr = [torch.from_numpy(a).to(device="cuda", dtype=dev.dtype) for a in wl.tracers]
    ptrs = (C.c_void_p * 26)(*[t.data_ptr() for t in tr])

    def run(wanted):
        out = [torch.full(g.parent_shape if q < 5 else (g.Ny, g.Nx), -7.0, dtype=dev.dtype, device="cuda")
               for q in range(7)]
        at = [o.data_ptr() if q in wanted else None for q, o in enumerate(out)]
        bands = (C.c_void_p * 3)(*at[1:4])
        assert library().obme_pisces_update_state(dev.handle, ptrs, C.c_void_p(at[0]), bands, C.c_void_p(at[4]),
                                                  C.c_void_p(at[5]), C.c_void_p(at[6]), C.c_double(0.0), None) == 0
        torch.cuda.synchronize()
        return [o.double().cpu().numpy() for o in out]

    every = run(range(7))
    for q in range(7):
        tol = (1e-12 if q == 4 else 1e-13) if precision == "fp64" else 1e-5
        got = g.interior(every[q]) if q < 5 else every[q]
        assert rel_l2(got, want[q]) <= tol if np.any(want[q]) else not np.any(got), q
        if q < 5:
            assert np.count_nonzero(every[q] == -7.0) == every[q].size - got.size
    for q in range(7):
        one = run([q])
        for r in range(7):
            if r == q:
                np.testing.assert_array_equal(one[r], every[r])
            else:
                assert np.all(one[r] == -7.0)
