"""Grids of many columns: a launch of few steps is the column sweep's where that
is the faster, with a sediment from fewer columns on.

In the dark (PAR0 = 0) a negative chlorophyll attenuation, whose logarithm the
levels-along-the-lanes kernel would need, leaves a handle to the sweep and
changes nothing else: the results are the same to the bit."""
import numpy as np
import pytest

from helpers import to_device
from oceanbiome import InstantRemineralisationSediment, workloads
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, n, steps, sediment", [("fp32", 512, 2, False), ("fp32", 256, 1, True),
                                                           ("fp64", 320, 1, True)])
def test_sweep_of_many_columns(precision, n, steps, sediment):
    import torch
    print("case many columns", precision, n, steps, sediment, flush=True)
    wl = workloads.lobster_3d(n, n, 5, surface_PAR=0.0)
    if sediment:
        wl.bgc.sediment = InstantRemineralisationSediment(sinking_tracers=("sPOM", "bPOM"),
                                                          remineralisation_reciever="NH₄")
    out = []
    for sweep in (False, True):
        wl.bgc.light_attenuation.chlorophyll_red_attenuation = -0.037 if sweep else 0.037
        dev = HIPBiogeochemistry(wl.bgc, precision)
        tr = to_device(wl.tracers, dev.dtype)
        dev.step(tr, steps, 600.0)
        torch.cuda.synchronize()
        out.append([t.cpu().numpy() for t in tr])
    for m, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), m
