"""FP64 powers past the range of doubles: the chlorophyll power of the light
with exponents that take it to infinity (no light is left) or to 0 (the water's
light is left), in the light hook, the tendencies and the step; and the
temperature factor Q10^(T/10) where it overflows, underflows and for a Q10 of 0
or less; against the oracle's pow."""
import numpy as np
import pytest

import oracle as O
from helpers import rel_l2, to_device, to_host
from oceanbiome import NPZD, RectilinearGrid, TwoBandPhotosyntheticallyActiveRadiation, abi
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


def _npzd(Nz, e, stretched):
    z = [-100.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)] if stretched else (-100.0, 0.0)
    g = RectilinearGrid(size=(5, 2, Nz), x=(0.0, 5.0), y=(0.0, 2.0), z=z)
    light = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0, chlorophyll_red_exponent=e,
                                                     chlorophyll_blue_exponent=0.5 * e)
    rng = np.random.default_rng(3)
    fields = []
    for lo, hi in ((1.0, 10.0), (0.05, 0.5), (0.05, 0.3), (8.0, 20.0), (0.5, 3.0)):
        f = g.new_field()
        g.interior(f)[...] = rng.uniform(lo, hi, (Nz, 2, 5))
        fields.append(f)
    return NPZD(g, light_attenuation=light), g, fields


# (exponent of the red band, P of one cell in the middle of every column)
POWERS = [(4.0, 1e100), (4.0, 1e-100), (-3.0, 1e-120), (-3.0, 1e120), (300.0, 20.0)]


@pytest.mark.parametrize("Nz", [6, 300])
@pytest.mark.parametrize("e, P", POWERS, ids=str)
def test_chlorophyll_power_past_the_range(e, P, Nz):
    import torch
    for stretched in (False, True):
        print("case power limits", e, P, Nz, stretched, flush=True)
        bgc, g, fields = _npzd(Nz, e, stretched)
        g.interior(fields[1])[...] = 0.5 if e < 10 else 0.9 * 0.7 / 1.31
        g.interior(fields[1])[Nz // 2] = P
        cfg = bgc.config(abi.OBME_FP64)
        ref = g.new_field()
        O.grid_update_state(cfg, fields, ref, 0.0)
        dev = HIPBiogeochemistry(bgc, "fp64")
        tr = to_device(fields, dev.dtype)
        PAR = torch.zeros(g.parent_shape, dtype=dev.dtype, device="cuda")
        dev.update_biogeochemical_state(tr, PAR, 0.0)
        G = [torch.zeros_like(PAR) for _ in tr]
        PAR2 = torch.zeros_like(PAR)
        dev.update_tendencies(tr, G, PAR2)
        torch.cuda.synchronize()
        want = g.interior(ref)
        assert np.isfinite(want).all()
        for x in (PAR, PAR2):
            got = g.interior(x.cpu().numpy())
            assert np.isfinite(got).all()
            assert rel_l2(got, want) <= 1e-13
        if P > 1e30:
            continue    # (P^2 times Z of such a cell is past any tolerance of the step)
        step = [f.copy() for f in fields]
        O.grid_run(cfg, step, 2, 60.0)
        dev.step(tr, 2, 60.0)
        torch.cuda.synchronize()
        for a, b in zip(to_host(tr), step):
            assert rel_l2(g.interior(a), g.interior(b)) <= 1e-12


# T = 0 and a multiple of 10 among the levels
@pytest.mark.parametrize("Q10, T", [(0.0, 12.0), (0.0, 0.0), (-2.0, 10.0), (-2.0, 20.0), (-2.0, 12.0), (1.88, -2e5),
                                    (1.88, 12.0)], ids=str)
@pytest.mark.parametrize("Nz", [6, 300])
def test_temperature_factor(Q10, T, Nz):
    import torch
    print("case Q10", Q10, T, Nz, flush=True)
    bgc, g, fields = _npzd(Nz, 0.629, True)
    bgc.plankton.temperature_coefficient = Q10
    g.interior(fields[3])[...] = T
    cfg = bgc.config(abi.OBME_FP64)
    dev = HIPBiogeochemistry(bgc, "fp64")
    tr = to_device(fields, dev.dtype)
    G = [torch.zeros_like(t) for t in tr]
    dev.update_tendencies(tr, G)
    want = [g.new_field() for _ in fields]
    O.grid_tendencies(cfg, fields, want)
    torch.cuda.synchronize()
    for n in (0, 1, 2, 4):
        a, b = g.interior(G[n].cpu().numpy()), g.interior(want[n])
        assert np.array_equal(np.isnan(a), np.isnan(b)), n
        ok = ~np.isnan(b)
        assert rel_l2(a[ok], b[ok]) <= 1e-12, n
    step = [f.copy() for f in fields]
    O.grid_run(cfg, step, 2, 60.0)
    dev.step(tr, 2, 60.0)
    torch.cuda.synchronize()
    for n, (x, y) in enumerate(zip(to_host(tr), step)):
        a, b = g.interior(x), g.interior(y)
        assert np.array_equal(np.isnan(a), np.isnan(b)), n
        ok = ~np.isnan(b)
        assert rel_l2(a[ok], b[ok]) <= 1e-12, n
