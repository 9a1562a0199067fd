"""Device memory of a handle with the CO2 exchange: the records of several steps
(up to 128 MB) are there once a call has taken several steps, not before;
obme_step_noalloc has none of the library's.  And a first call under graph capture
goes without them."""
import numpy as np
import pytest

from helpers import rel_l2, to_device, to_host
from oceanbiome import workloads
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


def _workload(scaling, *shape):
    wl = workloads.lobster_3d(*shape)
    wl.bgc.scale_negatives = scaling
    return wl


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("scaling", [False, True])
def test_records_of_several_steps(scaling, precision):
    import torch
    print("case memory", scaling, precision, flush=True)
    wl = _workload(scaling, 512, 512, 2)
    dtype = torch.float64 if precision == "fp64" else torch.float32
    tr = to_device(wl.tracers, dtype)
    G = [torch.zeros_like(t) for t in tr]
    PAR = torch.zeros_like(tr[0])
    # (the library's own first use: its code and its static scratch)
    small = _workload(scaling, 8, 8, 2)
    first = HIPBiogeochemistry(small.bgc, precision)
    ts = to_device(small.tracers, dtype)
    first.step_noalloc(ts, 3, 10.0)
    first.step(ts, 1, 10.0)
    first.update_biogeochemical_state(ts, torch.zeros_like(ts[0]), 0.0)
    first.update_tendencies(ts, [torch.zeros_like(t) for t in ts])
    first.close()
    torch.cuda.synchronize()

    def held():
        torch.cuda.synchronize()
        return before - torch.cuda.mem_get_info()[0]

    before = torch.cuda.mem_get_info()[0]
    dev = HIPBiogeochemistry(wl.bgc, precision)
    dev.update_biogeochemical_state(tr, PAR, 0.0)
    dev.update_tendencies(tr, G, PAR)
    dev.step_noalloc(tr, 3, 10.0)
    if not scaling:
        dev.step(tr, 1, 10.0)
    # one step's scratch per column: 6 record values, the warm start, the residuals, the stage's flux
    one = 512 * 512 * (6 * (8 if precision == "fp64" else 4) + 8 + 8 + 8)
    print("held", held(), "one step's", one, flush=True)
    assert held() <= one + (8 << 20)
    dev.step(tr, 3, 10.0)
    assert held() > one + (8 << 20)
    dev.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("scaling, nsteps", [(False, 1), (True, 3)])
def test_first_call_under_capture(scaling, nsteps, precision):
    import torch
    print("case capture", scaling, precision, flush=True)
    wl = _workload(scaling, 20, 6, 12)
    eager = HIPBiogeochemistry(wl.bgc, precision)
    want = to_device(wl.tracers, eager.dtype)
    dev = HIPBiogeochemistry(wl.bgc, precision)
    tr = to_device(wl.tracers, dev.dtype)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        dev.step(tr, nsteps, 60.0)
    for replay in range(3):
        graph.replay()
        torch.cuda.synchronize()
        eager.step(want, nsteps, 60.0)
        torch.cuda.synchronize()
        for name, a, b in zip(wl.bgc.required_biogeochemical_tracers(), to_host(tr), to_host(want)):
            e = rel_l2(wl.grid.interior(a), wl.grid.interior(b))
            assert e <= (1e-12 if precision == "fp64" else 1e-5), (replay, name, e)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_noalloc_with_scaling(precision):
    """The top cells' records in the static array: two calls, the second on a
    smaller grid, as obme_step on a fresh handle."""
    import torch
    for shape in ((48, 20, 24), (10, 6, 8)):
        print("case noalloc scaling", precision, shape, flush=True)
        wl = _workload(True, *shape)
        out = []
        for noalloc in (False, True):
            dev = HIPBiogeochemistry(wl.bgc, precision)
            tr = to_device(wl.tracers, dev.dtype)
            (dev.step_noalloc if noalloc else dev.step)(tr, 18, 60.0)
            torch.cuda.synchronize()
            out.append(to_host(tr))
        for a, b in zip(*out):
            if precision == "fp64":
                assert np.array_equal(a, b)
            else:
                assert rel_l2(wl.grid.interior(a), wl.grid.interior(b)) <= 1e-5
