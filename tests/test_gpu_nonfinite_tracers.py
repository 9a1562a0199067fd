"""Tracers that are not finite, and denominators of 0, in the LOBSTER tendencies:
the same tendencies are NaN as in the oracle and the others agree with it, from
the levels-along-the-lanes kernel and from the column sweep (300 levels)."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device
from oceanbiome import LOBSTER, CarbonateSystem, RectilinearGrid, TwoBandPhotosyntheticallyActiveRadiation, abi
from oceanbiome.models import AnalyticalLightLimitation, MondoLightLimitation, Oxygen
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-12, "fp32": 1e-4}
MEDIANS = (10.0, 0.1, 0.1, 0.1, 0.05, 0.05, 0.05, 2100.0, 2320.0, 250.0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("Nz", [24, 300])
@pytest.mark.parametrize("light", [MondoLightLimitation, AnalyticalLightLimitation])
def test_ammonia_that_is_not_finite(light, Nz, precision):
    import torch
    for value in (np.inf, np.nan, "-k"):
        if value == "-k" and precision == "fp32":
            continue    # (the FP32 transitions share one reciprocal: NaN)
        print("case ammonia", light, Nz, precision, value, flush=True)
        g = RectilinearGrid(size=(6, 2, Nz), x=(0.0, 6.0), y=(0.0, 2.0), z=(-100.0, 0.0))
        bgc = LOBSTER(g, carbonate_system=CarbonateSystem(), oxygen=Oxygen(), temperature=12.0, salinity=35.0,
                      light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0))
        bgc.plankton.light_limitation = light
        rng = np.random.default_rng(5)
        fields = []
        for m in MEDIANS:
            f = g.new_field()
            g.interior(f)[...] = m * np.exp(0.2 * rng.standard_normal((Nz, 2, 6)))
            fields.append(f)
        k = bgc.config(abi.OBME_FP64).npd.ammonia_half_saturation
        g.interior(fields[1])[Nz // 2, 1, 2] = -k if value == "-k" else value
        want = [g.new_field() for _ in fields]
        O.grid_tendencies(bgc.config(abi.OBME_FP64), fields, want)
        dev = HIPBiogeochemistry(bgc, precision)
        tr = to_device(fields, dev.dtype)
        G = [torch.zeros_like(t) for t in tr]
        dev.update_tendencies(tr, G)
        torch.cuda.synchronize()
        for name, x, y in zip(bgc.required_biogeochemical_tracers(), G, want):
            a, b = g.interior(x.double().cpu().numpy()), g.interior(y)
            assert np.array_equal(np.isnan(a), np.isnan(b)), name
            ok = np.isfinite(b)
            assert np.array_equal(a[~ok & ~np.isnan(b)], b[~ok & ~np.isnan(b)]), name
            assert rel_l2(a[ok], b[ok]) <= TOL[precision], name
