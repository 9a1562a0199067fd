"""Negative scaling with a factor below 0 (a sum that is negative where no member
is): FP64 rescales such cells as the reference does, in the step of columns along
the lanes, of deeper ones in the sweep, and with the CO2 flux at the top."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device, to_host
from oceanbiome import (LOBSTER, NPZD, CarbonateSystem, CarbonDioxideGasExchangeBoundaryCondition, RectilinearGrid,
                        TwoBandPhotosyntheticallyActiveRadiation, abi)
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nz", [20, 150])
@pytest.mark.parametrize("model", ["npzd", "lobster"])
def test_factor_below_zero(model, Nz):
    import torch
    print("case scaling factor", model, Nz, flush=True)
    g = RectilinearGrid(size=(7, 3, Nz), x=(0.0, 7.0), y=(0.0, 3.0), z=(-100.0, 0.0))
    light = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0)
    if model == "npzd":
        bgc = NPZD(g, light_attenuation=light, scale_negatives=True, invalid_fill_value=0.5)
        medians = (2.5, 0.1, 0.05, 12.0, 0.05)
    else:
        bgc = LOBSTER(g, carbonate_system=CarbonateSystem(), light_attenuation=light, scale_negatives=True,
                      invalid_fill_value=0.5, gas_exchange=CarbonDioxideGasExchangeBoundaryCondition(),
                      temperature=12.0, salinity=35.0)
        medians = (10.0, 0.1, 0.1, 0.1, 0.05, 0.05, 0.05, 2100.0, 2320.0)
    plain = bgc.config

    def config(precision):
        c = plain(precision)
        c.scaling.scalefactor[0][1] = -(60.0 if model == "npzd" else 120.0)   # the sums are about 0
        return c

    bgc.config = config
    rng = np.random.default_rng(4)
    fields = []
    for m in medians:
        f = g.new_field()
        g.interior(f)[...] = m * np.exp((0.02 if m > 1000 else 0.3) * rng.standard_normal((Nz, 3, 7)))
        fields.append(f)
    ref = [f.copy() for f in fields]
    O.grid_run(bgc.config(abi.OBME_FP64), ref, 2, 60.0)
    assert any(not np.allclose(g.interior(r), g.interior(f), rtol=0.1) for r, f in zip(ref, fields))
    dev = HIPBiogeochemistry(bgc, "fp64")
    tr = to_device(fields, dev.dtype)
    dev.step(tr, 2, 60.0)
    torch.cuda.synchronize()
    for name, x, r in zip(bgc.required_biogeochemical_tracers(), to_host(tr), ref):
        a, b = g.interior(x), g.interior(r)
        assert np.array_equal(np.isnan(a), np.isnan(b)), name
        ok = ~np.isnan(b)
        assert rel_l2(a[ok], b[ok]) <= 1e-10, name
