"""FP32 with a sediment: the FP64 storage is the same to the bit from the kernel
with a column's levels along the lanes and from the column sweep, for every
combination of the components that changes the kernels.

In the dark (PAR0 = 0) the light does not matter, and a negative chlorophyll
attenuation, whose logarithm the first kernel would need, leaves a handle to the
sweep."""
import itertools

import numpy as np
import pytest

from helpers import to_device
from oceanbiome import (LOBSTER, CarbonateSystem, CarbonDioxideGasExchangeBoundaryCondition,
                        InstantRemineralisationSediment, RectilinearGrid, TwoBandPhotosyntheticallyActiveRadiation)
from oceanbiome.models import Oxygen
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu

RANGES = ((5.0, 12.0), (0.1, 1.0), (0.05, 0.5), (0.05, 0.3), (0.5, 3.0), (0.5, 3.0), (0.1, 1.0))
CARBONATE = ((2000.0, 2200.0), (2300.0, 2400.0))


@pytest.mark.parametrize("Nz", [2, 8, 50, 64])
def test_storage_of_both_kernels(Nz):
    import torch
    for carbonate, oxygen, scaling, stretched in itertools.product((False, True), repeat=4):
        print("case sediment order", Nz, carbonate, oxygen, scaling, stretched, flush=True)
        z = [-4.0 * Nz * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)] if stretched else (-4.0 * Nz, 0.0)
        g = RectilinearGrid(size=(9, 7, Nz), x=(0.0, 90.0), y=(0.0, 70.0), z=z)
        ranges = RANGES + (CARBONATE if carbonate else ()) + (((200.0, 300.0),) if oxygen else ())
        rng = np.random.default_rng(Nz)
        fields = []
        for lo, hi in ranges:
            f = g.new_field()
            g.interior(f)[...] = rng.uniform(lo, hi, (Nz, 7, 9))
            fields.append(f)
        if scaling:
            g.interior(fields[3])[rng.random((Nz, 7, 9)) < 0.05] *= -0.01
        out = []
        for attenuation in (0.037, -0.037):
            bgc = LOBSTER(g, carbonate_system=CarbonateSystem() if carbonate else None,
                          oxygen=Oxygen() if oxygen else None, scale_negatives=scaling, temperature=12.0, salinity=35.0,
                          gas_exchange=CarbonDioxideGasExchangeBoundaryCondition() if carbonate else None,
                          light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(
                              surface_PAR=0.0, chlorophyll_red_attenuation=attenuation),
                          sediment_model=InstantRemineralisationSediment(sinking_tracers=("sPOM", "bPOM"),
                                                                         remineralisation_reciever="NH₄"))
            dev = HIPBiogeochemistry(bgc, "fp32")
            tr = to_device(fields, dev.dtype)
            dev.step(tr, 3, 60.0)
            dev.step(tr, 4, 300.0, t0=180.0)
            torch.cuda.synchronize()
            out.append(dev.sediment_storage.cpu().numpy())
        assert np.all(out[0] > 0)
        assert np.array_equal(out[0], out[1])
