"""FP32 ensembles with a sediment: the default formulations (compiled in) and
others (chosen at run time), in every plan and at the depths where the packing
has its edges, in whole rows of lanes and, with many short columns, lane by
lane, against the oracle's column runs; the bounds are those of the other FP32
ensemble tests (1e-5, ten times that per column), and the storage's is the
tracers'."""
import pytest

import oracle as O
from helpers import rel_l2
from oceanbiome import InstantRemineralisationSediment, abi
from oceanbiome.models import Quadratic
from oceanbiome.runtime import HIPBatch
from test_gpu_batch_packing import DEPTHS, _ensemble

pytestmark = pytest.mark.gpu
TOL = 1e-5
# (in whole rows: over 1024 waves; lane by lane: far fewer)
CASES = dict(DEPTHS, many=[1, 2, 3, 5, 8, 13, 21] * 650 + [128, 127, 97, 65, 64, 63, 62, 33, 31])


@pytest.mark.parametrize("forms", ["default", "other"])
@pytest.mark.parametrize("name", CASES)
def test_forms(name, forms):
    import torch
    print("case batch sediment", name, forms, flush=True)
    depths = CASES[name]
    wl = _ensemble(depths, seed=5)
    if forms == "other":
        wl.bgc.plankton.phytoplankton_mortality_formulation = Quadratic
    wl.bgc.sediment = InstantRemineralisationSediment(sinking_tracers=("P", "D"), remineralisation_reciever="N")
    off = wl.extra["offsets"]
    ref = [a.copy() for a in wl.tracers]
    state = O.SedimentState(len(depths), 1)
    O.batch_run(wl.bgc.config(abi.OBME_FP64), off, list(wl.extra["params"]), wl.extra["dz"], wl.extra["T"], ref,
                wl.nsteps, wl.dt, sediment=state)
    ran = 0
    for plan in range(7):
        b = HIPBatch(wl.bgc, off, wl.extra["params"], wl.extra["dz"], wl.extra["T"], "fp32")
        try:
            b.configure(plan, 0)
        except Exception:          # a plan without a tile for the deepest column
            assert max(depths) > 64
            continue
        tr = [torch.from_numpy(a).to(device="cuda", dtype=b.dtype) for a in wl.tracers]
        b.step(tr, wl.nsteps, wl.dt)
        assert rel_l2(b.sediment_storage.cpu().numpy().ravel(), state.storage.ravel()) <= TOL, plan
        for a, r in zip(tr, ref):
            a = a.double().cpu().numpy()
            assert rel_l2(a, r) <= TOL, plan
            for c in range(len(depths)):
                s = slice(off[c], off[c + 1])
                assert rel_l2(a[s], r[s]) <= 10 * TOL, (plan, c)
        ran += 1
    assert ran
