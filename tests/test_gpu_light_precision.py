"""FP32 PAR of the hooks against 64 bits on the same FP32 tracers: no further off
than the column sweep's, whose integral is a compensated sum.  The sweep writes
the PAR of the tendency hook above 32768 columns and above 128 levels; the
light hook's kernel and, below that, the tendency hook's own take other sums.
All three round the exponent once and take the same powers: their rms errors
are alike, a quarter more is the room for another order of the roundings."""
import numpy as np
import pytest

from helpers import to_device
from oceanbiome import NPZD, RectilinearGrid, TwoBandPhotosyntheticallyActiveRadiation
from oceanbiome.runtime import HIPBiogeochemistry

pytestmark = pytest.mark.gpu


def _par(light, zc, zf, P):
    Rr = light.phytoplankton_chlorophyll_ratio / light.pigment_ratio
    out = 0.0
    for kw, chi, e in ((light.water_red_attenuation, light.chlorophyll_red_attenuation, light.chlorophyll_red_exponent),
                       (light.water_blue_attenuation, light.chlorophyll_blue_attenuation,
                        light.chlorophyll_blue_exponent)):
        p = (P * Rr) ** e
        above = (zf[1:] - zc)[:, None, None] * p                        # the half cell above a level's centre
        below = np.zeros_like(p)
        below[:-1] = (zc[1:] - zf[1:-1])[:, None, None] * p[1:]         # of the level above, under its centre
        J = np.cumsum((above + below)[::-1], axis=0)[::-1]
        out = out + 0.5 * np.exp(kw * zc[:, None, None] - chi * J)
    return out


def _hooks(light, z, shape, fields):
    """PAR of the light hook and of the tendency hook."""
    import torch
    Nx, Ny, Nz = shape
    g = RectilinearGrid(size=shape, x=(0.0, 1.0 * Nx), y=(0.0, 1.0 * Ny), z=z)
    dev = HIPBiogeochemistry(NPZD(g, light_attenuation=light), "fp32")
    parents = []
    for f in fields:
        p = g.new_field()
        g.interior(p)[...] = f
        parents.append(p)
    tr = to_device(parents, dev.dtype)
    PAR = [torch.zeros(g.parent_shape, dtype=dev.dtype, device="cuda") for _ in range(2)]
    dev.update_biogeochemical_state(tr, PAR[0], 0.0)
    dev.update_tendencies(tr, [torch.zeros_like(t) for t in tr], PAR[1])
    torch.cuda.synchronize()
    return [g.interior(x.double().cpu().numpy()) for x in PAR]


@pytest.mark.parametrize("median", [0.1, 3.0])
@pytest.mark.parametrize("stretched", [False, True])
@pytest.mark.parametrize("Nx, Ny, Nz", [(256, 130, 10), (256, 130, 64), (256, 130, 100), (96, 40, 400)])
def test_par_of_the_hooks(Nx, Ny, Nz, stretched, median):
    print("case light precision", Nz, stretched, median, flush=True)
    z = [-400.0 * (1 - k / Nz) ** 1.5 for k in range(Nz + 1)] if stretched else (-400.0, 0.0)
    light = TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0)
    rng = np.random.default_rng(Nz)
    fields = [np.float32(m * np.exp(0.5 * rng.standard_normal((Nz, Ny, Nx)))).astype(np.float64)
              for m in (2.0, median, 0.05, 12.0, 0.05)]
    g = RectilinearGrid(size=(1, 1, Nz), x=(0.0, 1.0), y=(0.0, 1.0), z=z)
    want = 100.0 * _par(light, np.asarray(g.zc), np.asarray(g.zf), fields[1])
    ok = want > 1e-30

    def rms(x, rows):
        k = ok[:, rows]
        return np.sqrt(np.mean((x[k] / want[:, rows][k] - 1) ** 2))

    every, some = slice(None), slice(0, 40)
    hook, sweep = _hooks(light, z, (Nx, Ny, Nz), fields)
    errors = [rms(hook, every), rms(sweep, every)]
    if Nz <= 128:
        errors.insert(1, rms(_hooks(light, z, (Nx, 40, Nz), [f[:, some] for f in fields])[1], some))
    print("rms errors", errors, flush=True)
    assert max(errors[:-1]) <= 1.25 * errors[-1]
