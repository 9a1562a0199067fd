"""FP32 tendency hook on a uniform grid: the sinking of nearly uniform particle
tracers is rounded against their differences, not against their fluxes (from the
kernel of small grids and from the sweep).

Every term of the tendency is a product of at most eight rounded factors and the
terms are added one by one: 16 roundings of 2^-24 against the sum of the terms'
sizes.  A flux w c itself, 1e3 times the differences here, would leave 2^-24 w c
of rounding."""
import numpy as np
import pytest

import oracle as O
from helpers import to_device
from oceanbiome import LOBSTER, NPZD, RectilinearGrid, TwoBandPhotosyntheticallyActiveRadiation, abi
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nz", [30, 64, 150])
@pytest.mark.parametrize("model", ["npzd", "lobster"])
def test_sinking_of_nearly_uniform_particles(model, Nz):
    import torch
    print("case hook sinking", model, Nz, flush=True)
    g = RectilinearGrid(size=(12, 5, Nz), x=(0.0, 12.0), y=(0.0, 5.0), z=(-2.0 * Nz, 0.0))
    light = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0)
    bgc = NPZD(g, light_attenuation=light) if model == "npzd" else LOBSTER(g, light_attenuation=light)
    names = bgc.required_biogeochemical_tracers()
    sinking = {"npzd": ("D",), "lobster": ("sPOM", "bPOM")}[model]
    rng = np.random.default_rng(1)
    fields = []
    for n in names:
        f = g.new_field()
        if n in sinking:
            f[...] = 10.0
            g.interior(f)[...] += 0.01 * rng.standard_normal((Nz, 5, 12))
        elif n == "T":
            f[...] = 12.0
        else:
            g.interior(f)[...] = 1e-4 if n in ("P", "Z") else 1.0
        fields.append(f.astype(np.float32).astype(np.float64))
    cfg = bgc.config(abi.OBME_FP64)
    want = [g.new_field() for _ in fields]
    O.grid_tendencies(cfg, fields, want)
    dev = HIPBiogeochemistry(bgc, "fp32")
    tr = to_device(fields, dev.dtype)
    G = [torch.zeros_like(t) for t in tr]
    dev.update_tendencies(tr, G)
    torch.cuda.synchronize()
    for q, n in enumerate(names):
        if n not in sinking:
            continue
        c = g.interior(fields[q])
        w = cfg.sinking.speed[q] / 2.0
        differences = w * np.abs(np.diff(c, axis=0))
        got, ref = g.interior(G[q].double().cpu().numpy())[:-1], g.interior(want[q])[:-1]
        size = differences + np.abs(ref) + np.abs(ref + w * np.diff(c, axis=0))
        size += {"D": bgc.config(abi.OBME_FP64).npd.remineralisation_rate,
                 "sPOM": cfg.npd.small_remineralisation_rate, "bPOM": cfg.npd.large_remineralisation_rate}[n] * c[:-1]
        worst = np.max(np.abs(got - ref) / size)
        print(n, "error in roundings", worst * 2.0 ** 24, flush=True)
        assert worst <= 16 * 2.0 ** -24, n
