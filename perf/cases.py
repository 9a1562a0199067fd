"""Timed cases of the biogeochemistry step: what a program that uses this
package has it do, through the package's public entry points.

A case is a dict of plain values; its "kind" says which entry points it
takes:

 - "npd":      HIPBiogeochemistry (NPZD or LOBSTER): step(), or the two hooks
               of a coupled ocean model, update_biogeochemical_state() and
               update_tendencies(), which it calls at every Runge-Kutta stage;
 - "pisces":   HIPPISCES: step(), or its two hooks;
 - "ensemble": HIPBatch: independent NPZD columns of ragged depth, each with
               its own parameters (parameter estimation);
 - "points":   HIPBiogeochemistry.co2_flux(): pH and CO2 flux of point sets.

listed() are the cases, draw() makes more of the same ranges, prepare() makes
what a program holds before the call, run() is one pass, work() the bytes and
operations a pass cannot do without, and exact() the same values from plain
torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oceanbiome.jl_amd"))

from oceanbiome.grid import RectilinearGrid                                     # noqa: E402
from oceanbiome.models import (LOBSTER, NPZD, CarbonateSystem,                  # noqa: E402
                               CarbonDioxideGasExchangeBoundaryCondition, InstantRemineralisationSediment, Oxygen,
                               OxygenGasExchangeBoundaryCondition, TwoBandPhotosyntheticallyActiveRadiation)
from oceanbiome.pisces import PISCES                                            # noqa: E402
from oceanbiome.runtime import HIPPISCES, HIPBatch, HIPBiogeochemistry          # noqa: E402

DAY = 86400.0
HALO = 3
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


# ---------------------------------------------------------------- the cases

def _npd(name, model, precision, nx, ny, nz, call="step", steps=1, dt=60.0, carbonate=False, oxygen=False, gas=False,
         light="constant", sinking="upwind", stretched=False, fields=False, scale=False, sediment=False):
    return dict(name=name, kind="npd", model=model, precision=precision, nx=nx, ny=ny, nz=nz, call=call, steps=steps,
                dt=dt, carbonate=carbonate, oxygen=oxygen, gas=gas, light=light, sinking=sinking,
                stretched=stretched, fields=fields, scale=scale, sediment=sediment)


def _pisces(name, precision, nx, ny, nz, call="step", steps=1, dt=300.0, gas=False, light="constant"):
    return dict(name=name, kind="pisces", precision=precision, nx=nx, ny=ny, nz=nz, call=call, steps=steps, dt=dt,
                gas=gas, light=light)


def _ensemble(name, precision, columns, nz_min, nz_max, steps, sediment=False):
    return dict(name=name, kind="ensemble", precision=precision, columns=columns, nz_min=nz_min, nz_max=nz_max,
                steps=steps, dt=60.0, sediment=sediment)


def _points(name, n, mode):
    return dict(name=name, kind="points", n=n, mode=mode)


def listed():
    return [
        # one step of the smallest model configuration, the 2-D NPZD front of
        # 160 x 32 cells: a call's own latency
        _npd("npzd_slice", "npzd", "fp64", 160, 1, 32, dt=50.0),
        # the standalone stepper on the headline configuration
        _npd("lobster_fp32", "lobster", "fp32", 512, 512, 64, steps=10, carbonate=True, gas=True),
        # the same model in double precision on a regional grid
        _npd("lobster_fp64", "lobster", "fp64", 256, 256, 64, steps=4, carbonate=True, gas=True),
        # one step at a time between the steps of a host model that holds T
        # and S: every component, the daily cycle of light, a stretched
        # vertical grid and a horizontal size that is no multiple of anything
        _npd("lobster_o2_ragged", "lobster", "fp32", 333, 187, 75, carbonate=True, oxygen=True, gas=True,
             light="diurnal", stretched=True, fields=True),
        # fifth-order WENO sinking, the advection scheme of the usual setups
        _npd("lobster_weno5", "lobster", "fp32", 256, 256, 64, steps=4, carbonate=True, gas=True, sinking="weno5"),
        # the safe options together: negative tracers rescaled, a sediment
        # under every column, light from a 2-D surface field
        _npd("lobster_safe", "lobster", "fp32", 240, 180, 50, steps=4, carbonate=True, gas=True, light="array",
             scale=True, sediment=True),
        # the hooks of a coupled model, one Runge-Kutta stage
        _npd("lobster_hooks", "lobster", "fp32", 384, 384, 64, call="hooks", carbonate=True, gas=True),
        # PISCES: the standalone stepper on its benchmark grid
        _pisces("pisces_fp32", "fp32", 256, 256, 64, steps=10),
        # PISCES in double precision with its gas exchange and daily light
        _pisces("pisces_fp64", "fp64", 120, 100, 48, steps=2, gas=True, light="diurnal"),
        # PISCES's hooks, one Runge-Kutta stage of a coupled model
        _pisces("pisces_hooks", "fp32", 128, 96, 64, call="hooks"),
        # the ensemble of the parameter studies
        _ensemble("ensemble_fp32", "fp32", 8192, 16, 128, 50),
        # pH and CO2 flux of a global surface data set, the default solve
        _points("carbonate_points", 4000037, 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(nx, ny, nz, steps, most):
    """(ny, steps) with nx ny nz steps <= most."""
    steps = max(1, min(steps, most // (nx * nz)))
    return max(1, min(ny, most // (nx * nz * steps))), steps


def draw(rng):
    kind = rng.choice(("npd", "npd", "npd_hooks", "pisces", "pisces_hooks", "ensemble", "points"))
    precision = rng.choice(("fp32", "fp32", "fp64"))
    wide = 1 if precision == "fp32" else 3
    light = rng.choice(("constant", "diurnal", "array"))
    if kind in ("npd", "npd_hooks"):
        nx, ny, nz = _log_int(rng, 16, 512), _log_int(rng, 8, 512), rng.randint(10, 100)
        steps = rng.randint(1, 10) if kind == "npd" else 1
        model = rng.choice(("npzd", "lobster", "lobster"))
        lobster = model == "lobster"
        sinking = rng.choice(("upwind", "upwind", "centered", "weno5"))
        carbonate = lobster and rng.random() < 0.7
        scale = sinking == "upwind" and rng.random() < 0.25
        sediment = sinking == "upwind" and rng.random() < 0.25
        heavy = 1 if sinking == "upwind" and not scale else 4
        ny, steps = _fit(nx, ny, nz, steps, 512 * 512 * 64 * 10 // (wide * heavy))
        c = _npd("", model, precision, nx, ny, nz, "hooks" if kind == "npd_hooks" else "step", steps, 60.0, carbonate,
                 lobster and rng.random() < 0.3, carbonate and rng.random() < 0.8, light, sinking,
                 rng.random() < 0.3, lobster and rng.random() < 0.4, scale, sediment)
    elif kind in ("pisces", "pisces_hooks"):
        nx, ny, nz = _log_int(rng, 8, 256), _log_int(rng, 8, 256), rng.randint(20, 100)
        steps = rng.randint(1, 10) if kind == "pisces" else 1
        heavy = 2 if kind == "pisces" and precision == "fp32" and nz <= 64 else 10
        ny, steps = _fit(nx, ny, nz, steps, 256 * 256 * 64 * 10 // heavy)
        c = _pisces("", precision, nx, ny, nz, "hooks" if kind == "pisces_hooks" else "step", steps, 300.0,
                    kind == "pisces" and rng.random() < 0.5, light)
    elif kind == "ensemble":
        columns = _log_int(rng, 100, 8192)
        nz_min = rng.randint(4, 40)
        c = _ensemble("", precision, columns, nz_min, rng.randint(nz_min + 1, 128), rng.randint(5, 50),
                      rng.random() < 0.4)
    else:
        c = _points("", _log_int(rng, 1000, 4000000), rng.choice((0, 0, 1)))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs

# medians of the lognormal tracers
LOBSTER_MEDIANS = {"NO₃": 10.0, "NH₄": 0.1, "P": 0.1, "Z": 0.1, "sPOM": 0.05, "bPOM": 0.05, "DOM": 0.05}
NPZD_MEDIANS = {"N": 2.5, "P": 0.1, "Z": 0.05, "D": 0.05}
PISCES_MEDIANS = {"P": 0.5, "PChl": 0.02, "PFe": 0.005, "D": 0.1, "DChl": 0.004, "DFe": 0.001, "DSi": 0.01, "Z": 0.1,
                  "M": 0.7, "DOC": 2.1, "POC": 7.8, "GOC": 38.0, "SFe": 0.206, "BFe": 1.1, "PSi": 0.1, "CaCO₃": 0.1,
                  "NO₃": 2.3, "NH₄": 0.9, "PO₄": 0.6, "Fe": 0.13, "Si": 8.5, "DIC": 2205.0, "Alk": 2566.0,
                  "O₂": 317.0}
UNIFORM = {"DIC": (2000.0, 2200.0), "Alk": (2250.0, 2400.0), "O₂": (180.0, 320.0), "T": (2.0, 28.0)}
# NPZD parameters in the order of the per-column parameter table; the ones
# at FIXED are fractions, which the studies leave alone
NPZD_DEFAULTS = (2.3868, 0.6989 / 0.1953, 0.6989 / DAY, 0.0, 0.75, 1.88, (0.066 + 0.0101) / DAY, 0.3395 / DAY,
                 0.0102 / DAY, 0.0101 / (0.066 + 0.0101), 1.0, 1.0, 2.1522 / DAY, 0.5573, 0.9116, 0.1213 / DAY, 0.5,
                 0.2551 / DAY, 2.7489 / DAY, 100.0)
FIXED = (3, 4, 9, 10, 11, 14, 16)
ENSEMBLE_DZ, ENSEMBLE_T = 2.0, 10.0


def _dtype(case):
    return torch.float64 if case["precision"] == "fp64" else torch.float32


def _grid(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    depth = {"npd": 200.0, "pisces": 1000.0}[case["kind"]]
    if case.get("model") == "npzd" and ny == 1:
        return RectilinearGrid(size=(nx, nz), extent=(10000.0, 500.0), halo=(HALO,) * 3,
                               topology=("Bounded", "Flat", "Bounded"))
    z = (-depth, 0.0)
    if case.get("stretched"):
        z = [-depth * (1 - k / nz) ** 1.5 for k in range(nz + 1)]
    return RectilinearGrid(size=(nx, ny, nz), x=(0.0, 500.0 * nx), y=(0.0, 500.0 * ny), z=z, halo=(HALO,) * 3)


def _tracers(case):
    if case["kind"] == "pisces":
        return list(PISCES_MEDIANS) + ["T", "S"]
    if case["model"] == "npzd":
        names = ["N", "P", "Z", "T", "D"]
    else:
        names = list(LOBSTER_MEDIANS) + (["DIC", "Alk"] if case["carbonate"] else [])
    return names + (["O₂"] if case["oxygen"] else [])


def _temperature_profile(grid):
    return 20 - 0.05 * np.abs(grid.zc)


def _fields(case, grid, seed):
    """The inputs of a grid case on DEVICE: the tracers, what the hooks add
    to (G) and fill (PAR), the 3-D T and S, the surface light."""
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    dt = _dtype(case)
    shape = (grid.Nz, grid.Ny, grid.Nx)

    def parent(v):
        f = torch.zeros(grid.parent_shape, dtype=dt, device=DEVICE)
        _interior(grid, f).copy_(v)
        return f

    def normal(s=shape):
        return torch.randn(s, generator=gen, device=DEVICE, dtype=torch.float32).double()

    def uniform(lo, hi, s=shape):
        return lo + (hi - lo) * torch.rand(s, generator=gen, device=DEVICE, dtype=torch.float32).double()

    zc = torch.as_tensor(grid.zc, device=DEVICE)[:, None, None]
    st = {"tracers": [], "T": None, "S": None, "surface": None}
    if case["kind"] == "pisces":
        rows = (torch.arange(grid.Ny, device=DEVICE, dtype=torch.float64) + 0.5) / grid.Ny
        for name, m in PISCES_MEDIANS.items():
            st["tracers"].append(parent(m * torch.exp((0.02 if name in ("DIC", "Alk") else 0.3) * normal())))
        st["tracers"].append(parent((2 + 26 * rows)[None, :, None] * torch.exp(zc / 500) + 0.0 * zc))
        st["tracers"].append(parent(35.0 + 0.3 * normal()))
    else:
        medians = NPZD_MEDIANS if case["model"] == "npzd" else LOBSTER_MEDIANS
        for name in _tracers(case):
            v = uniform(*UNIFORM[name]) if name in UNIFORM else medians[name] * torch.exp(0.5 * normal())
            if case["scale"] and name in ("P", "Z"):
                # the small undershoots an advection scheme leaves
                v = torch.where(uniform(0, 1) < 0.002, -0.01 * v, v)
            st["tracers"].append(parent(v))
        if case["fields"]:
            st["T"] = parent(18 + 0.04 * zc + 2 * normal())
            st["S"] = parent(35.0 + 0.3 * normal())
    if case["light"] == "array":
        st["surface"] = uniform(20.0, 180.0, (grid.Ny, grid.Nx)).to(dt)
    if case["call"] == "hooks":
        written = [t for n, t in zip(_tracers(case), st["tracers"]) if n not in ("T", "S")]
        st["G"] = [parent(1e-6 * _interior(grid, t).double() * normal()) for t in written]
        if case["kind"] == "npd":
            st["PAR"] = torch.zeros(grid.parent_shape, dtype=dt, device=DEVICE)
            if case["model"] == "npzd":   # T has a slot too (its tendency is not written)
                st["G"].insert(3, torch.zeros(grid.parent_shape, dtype=dt, device=DEVICE))
    return st


def _interior(grid, f):
    return f[grid.Hz:grid.Hz + grid.Nz, grid.Hy:grid.Hy + grid.Ny, grid.Hx:grid.Hx + grid.Nx]


def _ensemble_inputs(case, seed):
    # the columns' depths are the case's (the sites of a study), what is in
    # them the seed's
    n = case["columns"]
    offsets = np.zeros(n + 1, dtype=np.int64)
    offsets[1:] = np.cumsum(np.random.Generator(np.random.PCG64(n)).integers(case["nz_min"], case["nz_max"] + 1, n))
    rng = np.random.Generator(np.random.PCG64(int(seed)))
    params = np.tile(np.array(NPZD_DEFAULTS)[:, None], (1, n))
    factor = np.exp(0.2 * rng.standard_normal(params.shape))
    for k in range(len(params)):
        if k not in FIXED:
            params[k] *= factor[k]
    params[19] = rng.uniform(50.0, 200.0, n)
    cells = int(offsets[-1])
    lo_hi = ((1.0, 10.0), (0.01, 0.1), (0.01, 0.1), (0.005, 0.05))
    tracers = [torch.from_numpy(rng.uniform(a, b, cells)).to(DEVICE, _dtype(case)) for a, b in lo_hi]
    return offsets, params, tracers


def _point_inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def uniform(lo, hi):
        return lo + (hi - lo) * torch.rand(case["n"], generator=gen, device=DEVICE, dtype=torch.float64)

    u10 = 10 * torch.exp(0.3 * torch.randn(case["n"], generator=gen, device=DEVICE, dtype=torch.float64))
    return dict(DIC=uniform(1900.0, 2300.0), Alk=uniform(2100.0, 2500.0), T=uniform(-2.0, 32.0),
                S=uniform(30.0, 38.0), u10=u10)


# ---------------------------------------------------------------- prepare and run

def _npd_model(case, grid):
    surface = {"constant": 100.0, "diurnal": "default", "array": 100.0}[case["light"]]
    kw = dict(light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=surface),
              sinking_scheme=case["sinking"], scale_negatives=case["scale"],
              oxygen=Oxygen() if case["oxygen"] else None)
    if case["sediment"]:
        kw["sediment_model"] = (InstantRemineralisationSediment(grid) if case["model"] == "npzd" else
                                InstantRemineralisationSediment(grid, sinking_tracers=("sPOM", "bPOM"),
                                                                remineralisation_reciever="NH₄"))
    if case["model"] == "npzd":
        return NPZD(grid, **kw)
    gas = []
    if case["gas"] and case["carbonate"]:
        gas.append(CarbonDioxideGasExchangeBoundaryCondition())
    if case["gas"] and case["oxygen"]:
        gas.append(OxygenGasExchangeBoundaryCondition())
    return LOBSTER(grid, carbonate_system=CarbonateSystem() if case["carbonate"] else None, gas_exchange=tuple(gas),
                   temperature=_temperature_profile(grid), salinity=35.0, **kw)


def prepare(case, seed):
    if case["kind"] == "points":
        grid = RectilinearGrid(size=(1, 1, 8), extent=(1.0, 1.0, 8.0))
        bgc = LOBSTER(grid, carbonate_system=CarbonateSystem(),
                      gas_exchange=CarbonDioxideGasExchangeBoundaryCondition(), temperature=15.0, salinity=35.0)
        return dict(case=case, dev=HIPBiogeochemistry(bgc, "fp64"), points=_point_inputs(case, seed))
    if case["kind"] == "ensemble":
        offsets, params, tracers = _ensemble_inputs(case, seed)
        grid = RectilinearGrid(size=(1, 1, 128), z=(-128 * ENSEMBLE_DZ, 0.0))
        bgc = NPZD(grid, light_attenuation=TwoBandPhotosyntheticallyActiveRadiation(surface_PAR=100.0),
                   sediment_model=InstantRemineralisationSediment(grid) if case["sediment"] else None)
        dev = HIPBatch(bgc, offsets, params, ENSEMBLE_DZ, ENSEMBLE_T, case["precision"])
        return dict(case=case, dev=dev, tracers=tracers)
    grid = _grid(case)
    st = _fields(case, grid, seed)
    if case["kind"] == "pisces":
        light = {"constant": 100.0, "diurnal": "default", "array": None}[case["light"]]
        if light is None:
            light = st["surface"].double().cpu().numpy()
        st["dev"] = HIPPISCES(PISCES(grid, surface_PAR=light, co2_exchange=case["gas"], o2_exchange=case["gas"]),
                              case["precision"])
    else:
        st["dev"] = HIPBiogeochemistry(_npd_model(case, grid), case["precision"], surface_array=st["surface"])
    st["case"] = case
    return st


def run(state):
    case, dev = state["case"], state["dev"]
    if case["kind"] == "points":
        p = state["points"]
        return dev.co2_flux(p["DIC"], p["Alk"], p["T"], p["S"], p["u10"], pCO2_air=420.0, mode=case["mode"])
    if case["kind"] == "ensemble":
        dev.step(state["tracers"], case["steps"], case["dt"])
        return state["tracers"], dev.sediment_storage
    tracers = state["tracers"]
    if case["kind"] == "pisces":
        if case["call"] == "hooks":
            aux = dev.update_biogeochemical_state(tracers, t=_clock(case))
            dev.update_tendencies(tracers, state["G"], t=_clock(case))
            return aux, state["G"]
        dev.step(tracers, case["steps"], case["dt"], t0=_clock(case))
        return tracers[:24]
    if case["call"] == "hooks":
        dev.update_biogeochemical_state(tracers, state["PAR"], t=_clock(case))
        dev.update_tendencies(tracers, state["G"], PAR=state["PAR"], T=state["T"], S=state["S"], t=_clock(case))
        return state["PAR"], state["G"], tracers if case["scale"] else None
    dev.step(tracers, case["steps"], case["dt"], t0=_clock(case), T=state["T"], S=state["S"])
    return tracers, dev.sediment_storage


def _clock(case):
    return 3 * 3600.0 if case["light"] == "diurnal" else 0.0


def work(case):
    """Bytes: every input read once, every output written once.  Operations:
    multiplications, additions, quotients and elementary functions counted
    one each."""
    if case["kind"] == "points":
        return {"bytes": 56.0 * case["n"], "flops": 900.0 * case["n"]}
    size = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "ensemble":
        cells = case["columns"] * (case["nz_min"] + case["nz_max"]) / 2
        return {"bytes": 8.0 * size * cells + 160.0 * case["columns"], "flops": 3.0 * 110 * cells * case["steps"]}
    columns = case["nx"] * case["ny"]
    cells = columns * case["nz"]
    if case["kind"] == "pisces":
        if case["call"] == "hooks":
            return {"bytes": (26.0 + 2 * 24 + 5) * size * cells, "flops": 1100.0 * cells}
        return {"bytes": (26.0 + 24) * size * cells, "flops": 3 * 1100.0 * cells * case["steps"]}
    n = len(_tracers(case))
    npzd = case["model"] == "npzd"
    written = n - 1 if npzd else n
    flops = (110.0 if npzd else 150.0) + (60.0 if case["sinking"] == "weno5" else 0.0)
    surface = columns * (1500.0 if case["gas"] and case["carbonate"] else 0.0)
    if case["call"] == "hooks":
        # DIC and Alk enter the top cells' flux alone
        read = n - (2 if case["carbonate"] and not case["scale"] else 0) - (1 if case["oxygen"] else 0)
        return {"bytes": (read + 2.0 * written + 1) * size * cells, "flops": flops * cells + surface}
    return {"bytes": 1.0 * (n + written) * size * cells, "flops": 3.0 * case["steps"] * (flops * cells + surface)}


# ---------------------------------------------------------------- the same values in 64 bits

GAMMA, ZETA = (8 / 15, 5 / 12, 3 / 4), (0.0, -17 / 60, -5 / 12)
CLOCK = (0.0, 8 / 15, 2 / 3)
TINY = 5e-324


def _dev64(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device=DEVICE)


def _daylight(t):
    return 100 * max(0.0, math.cos(t * math.pi / (12 * 3600.0)))


def _density(T, S, bar):
    """Sea water density, the 55-term polynomial of Roquet et al. (2015)."""
    t, s, z = T / 40, torch.sqrt((S + 32) / (40 * 35.16504 / 35)), -(10 * bar) / 1e4
    r0 = (((((-1.7243708991e-03 * z + 1.5616995503e-02) * z + 6.4326772569e-02) * z + 2.2601900708e-01) * z
           - 5.2099962525) * z + 4.6494977072e+01) * z
    r3 = 3.7969820455e-01 * t - 1.8507636718e-02 * s - 2.3342758797e-02
    r2 = ((-1.2419983026 * t - 2.1311365518e-01 * s + 2.0564311499) * t + (2.5019633244 * s - 4.9527603989) * s
          + 2.0660924175)
    r1 = (((5.5927935970e-01 * t - 5.5077101279e-01 * s - 2.4649669534) * t + (-1.8795372996 * s + 3.5063081279) * s
           + 6.7080479603) * t + ((-6.5399043664e-01 * s + 5.0042598061) * s - 4.4870114575) * s - 1.3336301113e+01) * t
    r1 = r1 + ((6.6051753097 * s - 3.0938076334e+01) * s + 5.0774768218e+01) * s * s - 4.2549998214e+01 * s
    r1 = r1 + 1.9681925209e+01
    a = ((-1.9083568888e-01 * t + 4.8169980163e-01 * s + 5.4048723791e-01) * t
         + (-5.3563304045 * s + 1.1311538584e+01) * s - 8.3627885467) * t
    a = (a + ((-3.1742946532 * s + 1.9717078466e+01) * s - 3.3449108469e+01) * s + 2.1661789529e+01) * t
    a = (a + (((-5.4723692739 * s + 2.9130021253e+01) * s - 6.0362551501e+01) * s + 6.1548258127e+01) * s
         - 3.7074170417e+01) * t
    a = (a + ((((-1.9193502195 * s + 1.7681814114e+01) * s - 5.6888046321e+01) * s + 8.1770425108e+01) * s
              - 6.5281885265e+01) * s + 2.6010145068e+01) * t
    a = a + (((((-6.0579916612e+01 * s + 4.3227585684e+02) * s - 1.2849161071e+03) * s + 2.0375295546e+03) * s
              - 1.7864682637e+03) * s + 8.6672408165e+02) * s + 8.0189615746e+02
    return r0 + ((r3 * z + r2) * z + r1) * z + a


def _equilibrium(T, S):
    """The carbonate system's equilibrium constants at the surface."""
    K, lT, q = T + 273.15, torch.log(T + 273.15), torch.sqrt(S)
    ion = 19.924 * S / (1000 - 1.005 * S)
    qi, dilution = torch.sqrt(ion), torch.log(1 - 0.001005 * S)
    c = dict(K=K)
    c["K0"] = torch.exp(-60.2409 + 9345.17 / K + 23.3585 * (lT - math.log(100.0))
                        + (0.023517 - 0.00023656 * K + 4.7036e-7 * K * K) * S)
    c["K1"] = 10 ** (61.2172 - 3633.86 / K - 9.67770 * lT + 0.011555 * S - 0.0001152 * S * S)
    c["K2"] = 10 ** (-25.9290 - 471.78 / K + 0.01781 * S - 0.0001122 * S * S + 3.16967 * lT)
    c["KB"] = torch.exp(148.0248 + (-8966.90 - 2890.53 * q - 77.942 * S + 1.728 * S * q - 0.0996 * S * S) / K
                        + 137.1942 * q + 1.62142 * S + (-24.4344 - 25.085 * q - 0.2474 * S) * lT + 0.053105 * q * K)
    c["KW"] = torch.exp(148.9652 - 13847.26 / K - 23.6521 * lT + (-5.977 + 118.67 / K + 1.0495 * lT) * q - 0.01615 * S)
    c["KS"] = torch.exp(141.328 - 4276.1 / K - 23.093 * lT + (324.57 - 13856.0 / K - 47.986 * lT) * qi
                        + (-771.54 + 35474.0 / K + 114.723 * lT) * ion - 2698.0 * ion * qi / K
                        + 1776.0 * ion * ion / K + dilution)
    c["KF"] = torch.exp(-9.68 + 874.0 / K + 0.111 * q)
    c["KSi"] = torch.exp(117.385 - 8904.2 / K - 19.334 * lT + (3.5913 - 458.79 / K) * qi + (-1.5998 + 188.74 / K) * ion
                         + (0.07871 - 12.1652 / K) * ion * ion + dilution)
    c["boron"] = 0.000232 / 10.811 * S / 1.80655
    c["sulfate"] = 0.14 / 96.06 * S / 1.80655
    c["fluoride"] = 0.000067 / 18.9984 * S / 1.80655
    return c


def _hydrogen(c, DIC, Alk, Si=0.0):
    """[H+] where the alkalinity of the species is Alk: Newton from pH 8."""
    sd = 1 + c["sulfate"] / c["KS"]
    x = torch.full_like(DIC + Alk, 1e-8)
    for _ in range(30):
        d = x * x + c["K1"] * x + c["K1"] * c["K2"]
        n = c["K1"] * DIC * (x + 2 * c["K2"])
        bor, so4, hf, sil = (c["boron"] * c["KB"] / (c["KB"] + x), c["sulfate"] * x / (x + c["KS"] * sd),
                             c["fluoride"] * x / (x + c["KF"]), Si * c["KSi"] / (c["KSi"] + x))
        f = n / d + bor + c["KW"] / x + sil - x / sd - so4 - hf - Alk
        df = (c["K1"] * DIC / d - n * (2 * x + c["K1"]) / (d * d) - bor / (c["KB"] + x) - c["KW"] / (x * x)
              - sil / (c["KSi"] + x) - 1 / sd - so4 / x * c["KS"] * sd / (x + c["KS"] * sd)
              - hf / x * c["KF"] / (x + c["KF"]))
        x = torch.maximum(x - f / df, x / 4)
    return x


def _schmidt_velocity(coefficients, u10, T):
    a, b, c, d, e = coefficients
    return 0.266 / 3600 / 100 * u10 * u10 / torch.sqrt((a + b * T + c * T ** 2 + d * T ** 3 + e * T ** 4) / 660)


def _co2_exchange(DIC, Alk, T, S, u10=2.0, air=413.0):
    """(pH, F): F = k (pCO2 of the water - air), positive out of the water."""
    c = _equilibrium(T, S)
    unit = 1e-3 / _density(T, S, 1.0)
    DIC, Alk = DIC * unit, Alk * unit
    x, K = _hydrogen(c, DIC, Alk), c["K"]
    f = DIC * x * x / (x * x + c["K1"] * x + c["K1"] * c["K2"]) / c["K0"] * 1e6 * 0.09807
    virial = (-1636.75 + 12.0408 * K - 3.27957e-2 * K ** 2 + 3.16528e-5 * K ** 3) * 1e-6
    cross = (57.7 - 0.118 * K) * 1e-6
    phi = torch.ones_like(f)
    for _ in range(3):
        phi = torch.exp((virial + 2 * (1 - f / (phi * 101325)) ** 2 * cross) * 101325 / (8.31446261815324 * K))
    k = _schmidt_velocity((2116.8, -136.25, 4.7353, -0.092307, 0.0007555), u10, T)
    return -torch.log10(x), k * c["K0"] * _density(T, S, 0.0) / 1000 * (f / phi / 0.09807 - air)


def _o2_exchange(O2, T, S):
    K = T + 273.15
    h = K / 100
    beta = torch.exp(-58.3877 + 85.8079 / h + 23.8439 * torch.log(h)
                     + S * (-0.034892 + 0.015578 * h + 0.015578 * h * h))
    return _schmidt_velocity((1920.4, -135.6, 5.2122, -0.10939, 0.00093777), 2.0, T) * (O2 - 9352.7 * beta / K)


def _two_band(P, zc, zf, PAR0):
    """The two-band light at the centres of a column's cells."""
    def integral(e):
        p = (P * (1.31 / 0.7)) ** e
        inc = (zf[1:] - zc).view(-1, 1, 1) * p
        inc[:-1] += (zc[1:] - zf[1:-1]).view(-1, 1, 1) * p[1:]
        return inc.flip(0).cumsum(0).flip(0)
    z = zc.view(-1, 1, 1)
    return PAR0 * (torch.exp(0.225 * z - 0.037 * integral(0.629)) + torch.exp(0.0232 * z - 0.074 * integral(0.674))) / 2


def _grazing(P, Z, S, pref, rate, half):
    p = pref * P / (pref * P + (1 - pref) * S + TINY)
    food = p * P + (1 - p) * S
    L = food * food / (food * food + half * half)
    den = food + TINY
    return rate * L * Z, rate * p * L * P / den * Z, rate * (1 - p) * L * S / den * Z


def _npzd(X, PAR, oxygen, q, Lt):
    """q: the parameters in the order of NPZD_DEFAULTS."""
    N, P, Z, D = X["N"], X["P"], X["Z"], X["D"]
    mu = q[2] * PAR / torch.sqrt(PAR * PAR + q[1] * q[1]) * (N / (N + q[0])) * Lt * P
    G, onP, onS = _grazing(P, Z, q[16] * D, q[11], q[12], q[13])
    dead = q[6] * P
    waste = q[10] * q[8] * Z + (1 - q[9]) * dead
    out = dict(N=waste + q[15] * D - mu * (1 - q[4] * q[3]), P=(1 - q[3]) * mu - onP - dead,
               Z=q[14] * G - q[7] * Z * Z - q[8] * Z,
               D=((1 - q[4]) * q[3] * mu + (1 - q[10]) * q[8] * Z + (1 - q[14]) * G + q[9] * dead + q[7] * Z * Z
                  - onS - q[15] * D))
    if oxygen:
        out["O₂"] = 10.75 * mu - 8.75 * waste
    return out


def _lobster(X, PAR, carbonate, oxygen):
    NO3, NH4, P, Z, s, b, DOM = (X[n] for n in LOBSTER_MEDIANS)
    nl, al = NO3 * torch.exp(-3.0 * NH4) / (NO3 + 0.7), (NH4 / (0.001 + NH4)).clamp_min(0)
    base = 2.42e-5 * PAR / (33.0 + PAR) * P / 2
    mu, nitrification = base * (nl + al), 5.8e-7 * NH4
    G, onP, onS = _grazing(P, Z, s, 0.5, 9.26e-6, 1.0)
    dead = 5.8e-7 * P * P
    waste, rem = 0.5 * 5.8e-7 * Z, 3.86e-7 * DOM
    solid = 0.3 * G + dead + 2.31e-6 * Z * Z
    out = {"NO₃": nitrification - base * nl, "NH₄": waste + rem - nitrification - base * al + 0.0375 * mu,
           "P": 0.95 * mu - onP - dead, "Z": 0.7 * G - 2.31e-6 * Z * Z - 5.8e-7 * Z,
           "sPOM": 0.5 * solid - onS - 5.88e-7 * s, "bPOM": 0.5 * solid - 5.88e-7 * b,
           "DOM": 0.0125 * mu + waste + 5.88e-7 * (s + b) - rem}
    if carbonate:
        calcite = (onP + dead) * 0.656
        out["DIC"] = -(1 + 0.095 - 0.0375) * 6.56 * mu + 6.56 * (waste + rem) + calcite
        out["Alk"] = out["NH₄"] * 0.9375 - out["NO₃"] * 1.0625 - 4 * 0.656 * mu + 2 * calcite
    if oxygen:
        out["O₂"] = 10.75 * mu - 8.75 * out["NH₄"] - 10.75 * nitrification
    return out


def _face_values(c, scheme):
    """The values of a sinking tracer at the bottom faces of its cells."""
    f, n = c.clone(), len(c)
    if scheme == "centered":
        f[1:] = (c[:-1] + c[1:]) / 2
    if scheme == "weno5" and n > 3:
        def weights(b, d):
            a = [w * (1 + ((b[0] - b[-1]).abs() / (x + 1e-8)) ** 2) for x, w in zip(b, d)]
            return a, sum(a)
        for k in {2, n - 2}:
            m, o, p = c[k - 1], c[k], c[k + 1]
            a, s = weights([(o - p) ** 2, (m - o) ** 2], (1 / 3, 2 / 3))
            f[k] = (a[0] * (3 * o - p) / 2 + a[1] * (o + m) / 2) / s
        if n > 5:
            i = torch.arange(3, n - 2, device=c.device)
            mm, m, o, p, pp = (c[i + j] for j in (-2, -1, 0, 1, 2))
            b = [13 / 12 * (pp - 2 * p + o) ** 2 + (pp - 4 * p + 3 * o) ** 2 / 4,
                 13 / 12 * (p - 2 * o + m) ** 2 + (p - m) ** 2 / 4,
                 13 / 12 * (o - 2 * m + mm) ** 2 + (3 * o - 4 * m + mm) ** 2 / 4]
            a, s = weights(b, (0.1, 0.6, 0.3))
            f[i] = (a[0] * (2 * pp - 7 * p + 11 * o) / 6 + a[1] * (-p + 5 * o + 2 * m) / 6
                    + a[2] * (2 * o + 5 * m - mm) / 6) / s
    return f


def _sink(G, X, name, w, dz, scheme="upwind"):
    """G[name] minus the flux divergence of the face velocities w <= 0."""
    flux = w[:-1].view(-1, 1, 1) * _face_values(X[name], scheme)
    G[name] = G[name] + flux / dz.view(-1, 1, 1)
    G[name][:-1] -= flux[1:] / dz[:-1].view(-1, 1, 1)


def _rescale(X, group):
    """Negative members of a conserved group to zero, the others scaled."""
    total = sum(s * X[n] for n, s in group.items())
    positive = sum(s * X[n].clamp_min(0) for n, s in group.items())
    for n in group:
        X[n] = torch.where(X[n] > 0, X[n] * total / positive, torch.zeros_like(total))


def _burial(f):
    return 0.013 + 0.53 * (f / (7.0 / 6.56 + f)) ** 2


def _runge_kutta(X, names, tendencies, steps, dt, t0):
    """steps of the three-stage scheme in place; tendencies(X, t, dt of the
    stage's sediment step, step, stage)."""
    for step in range(steps):
        before = None
        for st in range(3):
            G = tendencies(X, t0 + (step + CLOCK[st]) * dt, dt, step, st)
            for n in names:
                X[n] = X[n] + dt * (GAMMA[st] * G[n] + (ZETA[st] * before[n] if st else 0.0))
            before = G


def _sediment(storage, f, step, st, dt):
    """The storage's step by a stage's flux f: forward Euler of the stage's
    length, the very first one with the second stage's tendency."""
    g = _burial(f) * f
    first = step == 0
    if st == 0:
        return storage if first else storage + GAMMA[0] * dt * g
    if st == 1 and first:
        storage = storage + GAMMA[0] * dt * g
    return storage + (GAMMA[st] + ZETA[st]) * dt * g


def _exact_npd(case, seed):
    grid = _grid(case)
    st = _fields(case, grid, seed)
    names = _tracers(case)
    X = {n: _interior(grid, t).double() for n, t in zip(names, st["tracers"])}
    zc, zf, dz = _dev64(grid.zc), _dev64(grid.zf), _dev64(grid.dz)
    npzd = case["model"] == "npzd"
    sinkers = {"P": 0.2551 / DAY, "D": 2.7489 / DAY} if npzd else {"sPOM": 3.47e-5, "bPOM": 200 / DAY}
    receiver = "N" if npzd else "NH₄"
    w = {n: -v * torch.cat([torch.ones_like(zc), torch.zeros_like(zc[:1])]) for n, v in sinkers.items()}
    co2, o2 = case["gas"] and case["carbonate"], case["gas"] and case["oxygen"] and not npzd
    if st["T"] is not None:
        T, S = _interior(grid, st["T"])[-1].double(), _interior(grid, st["S"])[-1].double()
    else:
        T = torch.full_like(X["P"][-1], float(_temperature_profile(grid)[-1]))
        S = torch.full_like(T, 35.0)
    groups = [{n: 1.0 for n in (NPZD_MEDIANS if npzd else LOBSTER_MEDIANS)}]
    if case["carbonate"]:
        groups.append({"P": 1.1 * 6.56, "Z": 6.56, "DIC": 1.0, "sPOM": 6.56, "bPOM": 6.56, "DOM": 6.56})
    stored = {"s": torch.zeros_like(T)}

    def light(t):
        return {"constant": 100.0, "diurnal": _daylight(t), "array": None}[case["light"]]

    def tendencies(X, t, dt, step, stage, rescale=True):
        if case["scale"] and rescale:
            for g in groups:
                _rescale(X, g)
        PAR0 = light(t)
        PAR = _two_band(X["P"], zc, zf, st["surface"].double() if PAR0 is None else PAR0)
        if npzd:
            G = _npzd(X, PAR, case["oxygen"], NPZD_DEFAULTS, 1.88 ** (X["T"] / 10))
        else:
            G = _lobster(X, PAR, case["carbonate"], case["oxygen"])
        if co2:
            G["DIC"][-1] -= _co2_exchange(X["DIC"][-1], X["Alk"][-1], T, S)[1] / dz[-1]
        if o2:
            G["O₂"][-1] -= _o2_exchange(X["O₂"][-1], T, S) / dz[-1]
        for n in sinkers:
            _sink(G, X, n, w[n], dz, case["sinking"])
        if case["sediment"]:
            f = sum(v * X[n][0] for n, v in sinkers.items())
            G[receiver][0] += (1 - _burial(f)) * f / dz[0]
            stored["s"] = _sediment(stored["s"], f, step, stage, dt)
        G["PAR"] = PAR
        return G

    def parent(v):
        f = torch.zeros(grid.parent_shape, dtype=torch.float64, device=DEVICE)
        _interior(grid, f).copy_(v)
        return f

    written = [n for n in names if n != "T"]
    if case["call"] == "hooks":
        G = tendencies(X, _clock(case), case["dt"], 0, 0)
        out = [parent(_interior(grid, st["G"][k]).double() + G[n]) if n != "T" else None for k, n in enumerate(names)]
        scaled = [parent(X[n]) for n in names] if case["scale"] else None
        return parent(G["PAR"]), out, scaled
    _runge_kutta(X, written, tendencies, case["steps"], case["dt"], _clock(case))
    return [parent(X[n]) for n in names], stored["s"] if case["sediment"] else None


def _exact_ensemble(case, seed):
    offsets, params, tracers = _ensemble_inputs(case, seed)
    offsets, q = torch.as_tensor(offsets, device=DEVICE), _dev64(params)
    nz = offsets[1:] - offsets[:-1]
    n, depth = len(nz), int(nz.max())
    # every column padded to the deepest below its bottom, [level, column, 1]
    k = torch.arange(depth, device=DEVICE)[:, None]
    inside = (k >= depth - nz)
    at = (offsets[:-1] + k - (depth - nz)).clamp_min(0)
    X = {name: torch.where(inside, t.double()[at], torch.ones_like(at, dtype=torch.float64) * 0.01)[:, :, None]
         for name, t in zip(NPZD_MEDIANS, tracers)}
    zf = -ENSEMBLE_DZ * torch.arange(depth, -1, -1, device=DEVICE, dtype=torch.float64)
    zc = (zf[1:] + zf[:-1]) / 2
    p = [row[:, None] for row in q]
    Lt = p[5] ** (ENSEMBLE_T / 10)
    bottom = (depth - nz)
    column = torch.arange(n, device=DEVICE)
    stored = {"s": torch.zeros(n, device=DEVICE, dtype=torch.float64)}

    def tendencies(X, t, dt, step, stage):
        G = _npzd(X, _two_band(X["P"], zc, zf, p[19]), False, p, Lt)
        for name, w in (("P", p[17]), ("D", p[18])):
            G[name] = G[name] - w * X[name] / ENSEMBLE_DZ
            G[name][:-1] += (w * X[name] / ENSEMBLE_DZ)[1:]
        if case["sediment"]:
            f = (p[17] * X["P"][bottom, column] + p[18] * X["D"][bottom, column])[:, 0]
            G["N"][bottom, column, 0] += (1 - _burial(f)) * f / ENSEMBLE_DZ
            stored["s"] = _sediment(stored["s"], f, step, stage, dt)
        return G

    _runge_kutta(X, list(NPZD_MEDIANS), tendencies, case["steps"], case["dt"], 0.0)
    out = [X[name][:, :, 0].T[inside.T] for name in NPZD_MEDIANS]
    return out, stored["s"] if case["sediment"] else None


def _day_length(t, latitude):
    day = math.floor(math.fmod(t, 365 * DAY) / DAY)
    theta = 0.216310 + 2 * math.atan(0.9671396 * math.tan(0.00860 * (day - 186)))
    dec = math.asin(0.39795 * math.cos(theta))
    lat = math.radians(math.fmod(latitude, 360.0))
    L = (math.sin(math.radians(0.833)) + math.sin(lat) * math.sin(dec)) / (math.cos(lat) * math.cos(dec))
    return (24 - 24 / 180 * math.degrees(math.acos(max(-1.0, min(1.0, L))))) * 3600


NANO = dict(dark=3 * DAY, NH4=0.013, NO3=0.13, PO4=0.8, si=False, band=(2.1, 0.42, 0.4), w1=0.0, chl=0.033, fe=1.0)
DIATOM = dict(dark=4 * DAY, NH4=0.039, NO3=0.39, PO4=2.4, si=True, band=(1.6, 0.69, 0.7), w1=0.03 / DAY, chl=0.05,
              fe=3.0)
MICRO = dict(g0=3 / DAY, pref=(1.0, 0.5, 0.1), m0=0.004 / DAY, r=0.03 / DAY, e0=0.3, ff=0.0, eta=0.5, fe=0.01)
MESO = dict(g0=0.75 / DAY, pref=(0.3, 1.0, 0.3, 1.0), m0=0.03 / DAY, r=0.005 / DAY, e0=0.35, ff=2e-3, eta=0.75,
            fe=0.015)
PISCES_MLD, PISCES_LATITUDE = -50.0, 45.0
# attenuation by water, chlorophyll exponent and coefficient: the means of
# the Morel (1988) spectral table over 400-500, 500-600 and 600-700 nm
BANDS = ((0.01143, 0.0699895, 0.3737025), (0.673612, 0.649562, 0.65865), (0.09989825, 0.04361825, 0.04255))


def _phytoplankton(h, F, A, I, chl, fe):
    """Growth, limitations, losses and uptakes of one phytoplankton class."""
    zero = torch.zeros_like(I)
    theta_fe, theta_chl = fe / (I + TINY), chl / (12 * I + TINY)
    size = (torch.clamp_max(I, 1.0) + 3 * (I - 1).clamp_min(0)) / (I + TINY)
    NO3, NH4, PO4, Si = F["NO₃"], F["NH₄"], F["PO₄"], F["Si"]
    kn, kh = h["NO3"] * size, h["NH4"] * size
    d = kn * kh + kn * NH4 + kh * NO3 + TINY
    s = dict(I=I, LNO3=kh * NO3 / d, LNH4=kn * NH4 / d, LPO4=PO4 / (PO4 + h["PO4"] * size + TINY))
    s["LN"] = s["LNO3"] + s["LNH4"]
    least = 1000 * (0.0016 / 55.85 * 12 * theta_chl + 1.5 * 1.21e-5 * 14 / (55.85 * 7.625) * s["LN"]
                    + 1.15e-4 * 14 / (55.85 * 7.625) * s["LNO3"])
    s["LFe"] = ((theta_fe - least) / 0.007).clamp(0, 1)
    s["L"] = torch.minimum(torch.minimum(s["LN"], s["LPO4"]), s["LFe"])
    if h["si"]:
        s["L"] = torch.minimum(s["L"], Si / (Si + size + 7 * 7.5 ** 2 / (16.6 ** 2 + 7.5 ** 2)))
    PAR = sum(b * p for b, p in zip(h["band"], A["bands"]))
    rate = 0.6 / DAY * 1.066 ** F["T"]
    mixing = (A["zeu"] - PISCES_MLD).clamp_min(0) ** 2
    light = 1 - torch.exp(-2.0 * theta_chl * PAR / (A["dl"] * (0.033 / DAY + 1 / DAY)))
    s["mu"] = rate * (1.5 * A["dl"] / (A["dl"] + 0.5 * DAY)) * (1 - mixing / (mixing + h["dark"])) * light * s["L"]
    s["muI"] = s["mu"] * I
    s["lin"] = 0.01 / DAY * I / (I + 0.2) * I
    s["quad"] = A["shear"] * (0.01 / DAY + h["w1"] * 0.25 * (1 - s["L"] ** 2) / (0.25 + s["L"] ** 2)) * I * I
    f1 = 1.5 * A["dl2"] / (A["dl2"] + 0.5 * DAY)
    rho = 12 * s["mu"] / f1 * A["dl2"] * I / (2.0 * chl * PAR + TINY) * s["L"]
    s["chl"] = 0.95 * 12 * (0.0033 + (h["chl"] - 0.0033) * rho) * s["muI"]
    quota = theta_fe / 0.06
    s["fe"] = (0.95 * 0.06 * F["Fe"] / (F["Fe"] + h["fe"] * size + TINY) * (4 - 4.5 * s["LFe"] / (s["LFe"] + 1))
               * torch.maximum(zero, (1 - quota) / (1.05 - quota)) * rate * I)
    if h["si"]:
        L1 = Si / (Si + 2.0 + TINY)
        F1 = torch.minimum(torch.minimum(s["mu"] / (rate * s["L"] + TINY), s["LFe"]),
                           torch.minimum(s["LPO4"], s["LN"]))
        F2 = (2.2 * (L1 - 0.5).clamp_min(0)).clamp_max(1)
        s["si"] = 0.95 * 0.159 * L1 * (4.4 * torch.exp(-4.23 * F1) * F2 + 1).clamp_max(5.4) * s["muI"]
    s["theta_fe"], s["theta_chl"] = theta_fe, theta_chl
    return s


def _zooplankton(h, F, A, I, anoxia):
    tf = 1.079 ** F["T"]
    prey = [F["P"], F["D"], F["POC"], F["Z"]][:len(h["pref"])]
    iron = [F["PFe"] / (F["P"] + TINY), F["DFe"] / (F["D"] + TINY), F["SFe"] / (F["POC"] + TINY),
            MICRO["fe"]][:len(h["pref"])]
    above = [p * (x - 0.001).clamp_min(0) for p, x in zip(h["pref"], prey)]
    food, irons = sum(p * x for p, x in zip(h["pref"], prey)), sum(p * i for p, i in zip(h["pref"], iron))
    available = sum(above)
    specific = h["g0"] * tf * (available - (available / 2).clamp_max(0.3)).clamp_min(0) / (20.0 + food)
    ratio = irons / (h["fe"] * specific + TINY)
    g = dict(e=ratio.clamp_max(1) * (0.7 * ratio).clamp_max(h["e0"]), on=[a * specific / (available + TINY) * I
                                                                        for a in above])
    flux = h["ff"] * tf * I
    g["food"] = specific * I + flux * (F["POC"] * A["wP"] + F["GOC"] * A["wG"])
    g["iron"] = (sum(a * i for a, i in zip(above, iron)) * specific / (available + TINY) * I
                 + flux * (F["SFe"] * A["wP"] + F["BFe"] * A["wG"]))
    g["onPOC"], g["onGOC"] = g["on"][2] + flux * F["POC"] * A["wP"], flux * F["GOC"] * A["wG"]
    g["lin"] = tf * h["r"] * (I / (I + 0.2) + 3 * anoxia) * I
    g["dead"] = tf * h["m0"] * I * I + g["lin"]
    g["waste"], g["tf"] = (0.7 - g["e"]) * g["food"], tf
    return g


def _pisces_tendencies(F, A):
    T, O2, Fe, DOC, POC, GOC = (F[n] for n in ("T", "O₂", "Fe", "DOC", "POC", "GOC"))
    NO3, NH4, PO4, Si = (F[n] for n in ("NO₃", "NH₄", "PO₄", "Si"))
    anoxia = (0.4 * (6.0 - O2) / (1.0 + O2)).clamp(0, 1)
    p = _phytoplankton(NANO, F, A, F["P"], F["PChl"], F["PFe"])
    d = _phytoplankton(DIATOM, F, A, F["D"], F["DChl"], F["DFe"])
    z, m = _zooplankton(MICRO, F, A, F["Z"], anoxia), _zooplankton(MESO, F, A, F["M"], anoxia)
    G = {}
    for s, n, k in ((p, "P", 0), (d, "D", 1)):
        s["loss"] = s["lin"] + s["quad"] + z["on"][k] + m["on"][k]
        G[n] = 0.95 * s["muI"] - s["loss"]
        G[n + "Chl"] = s["chl"] - s["loss"] * s["theta_chl"] * 12
        G[n + "Fe"] = s["fe"] - s["loss"] * s["theta_fe"]
    theta_si = F["DSi"] / (F["D"] + TINY)
    G["DSi"] = d["si"] - d["loss"] * theta_si
    G["Z"], G["M"] = z["e"] * z["food"] - z["dead"] - m["on"][3], m["e"] * m["food"] - m["dead"]
    upper = 1 / (1 - 0.35) * 0.03 / DAY * m["tf"] * F["M"] ** 2
    inorganic, organic = 0.6 * (z["waste"] + m["waste"] + 0.35 * upper), 0.4 * (z["waste"] + m["waste"] + 0.35 * upper)
    # bacteria, dissolved organic carbon
    deep = torch.clamp_max(A["zeu"], PISCES_MLD)
    below = A["z"] < deep
    bacteria = torch.where(below, (deep / A["z"]) ** 0.684, torch.ones_like(T)) * (0.7 * F["Z"] + 1.4
                                                                                    * F["M"]).clamp_max(4)
    active = torch.minimum(torch.minimum((0.03 * NH4 + 0.003 * NO3) / (9e-5 + 0.03 * NH4 + 0.003 * NO3),
                                         PO4 / (PO4 + 0.003)), Fe / (Fe + 0.01)) * DOC / (DOC + 417)
    degraded = 0.3 / DAY * 1.066 ** T * active * bacteria * DOC
    unit = 1e-6 / DAY
    phi1 = A["shear"] * (0.37 * DOC + 102 * POC) * unit * DOC
    phi2 = A["shear"] * 3530 * unit * GOC * DOC
    phi3 = (5095 * POC + 114 * DOC) * unit * DOC
    lam = 0.025 / DAY * 1.066 ** T * (1 - 0.45 * anoxia)
    G["DOC"] = 0.05 * (p["muI"] + d["muI"]) + organic + lam * POC - degraded - phi1 - phi2 - phi3
    # particles
    aggregated = unit * (A["shear"] * (25.9 * POC ** 2 + 4452 * POC * GOC) + 3.3 * POC * GOC + 47.1 * POC ** 2)
    PAR = A["PAR"]
    rain = (0.3 * torch.minimum(torch.minimum(p["LN"], Fe / (Fe + 0.05)), p["LPO4"]) * (F["P"] / 2).clamp_min(1)
            * (PAR - 1).clamp_min(0) / (4 + PAR) * 30 / (30 + PAR) * (T / (T + 0.1)).clamp_min(0)
            * (1 + torch.exp(-(T - 10) ** 2 / 25)))
    dead = p["lin"] + p["quad"]
    small, large = (1 - rain / 2) * dead, rain / 2 * dead
    onPOC, onGOC = z["onPOC"] + m["onPOC"], z["onGOC"] + m["onGOC"]
    G["POC"] = (0.3 * z["food"] + small + d["lin"] / 2 + z["dead"] + phi1 + phi3 + lam * GOC - onPOC - aggregated
                - lam * POC)
    G["GOC"] = (0.3 * m["food"] + large + d["lin"] / 2 + d["quad"] + m["lin"] + 0.3 * upper + aggregated + phi2 - onGOC
                - lam * GOC)
    ligands = (0.09 * (DOC + 40) - 3).clamp_min(0.6)
    K = torch.exp(16.27 - 1565.7 / (T + 273.15))
    b = 1 + K * ligands - K * Fe
    free = (-b + torch.sqrt(b * b + 4 * K * Fe)) / (2 * K)
    colloid = 0.5 * (Fe - free) / (DOC + TINY)
    scavenging = 3e-5 / DAY + 0.005 / DAY * (POC + GOC + F["CaCO₃"] + F["PSi"])
    bacteria_fe = 0.6 / DAY * 1.066 ** T * active * 0.06 * Fe / (Fe + 0.3) * bacteria * 0.16
    theta_s, theta_b = F["SFe"] / (POC + TINY), F["BFe"] / (GOC + TINY)
    G["SFe"] = (0.3 * z["iron"] + small * p["theta_fe"] + d["lin"] * d["theta_fe"] / 2 + z["dead"] * MICRO["fe"]
                + lam * F["BFe"] + scavenging * POC * free + 0.12 / 0.16 * bacteria_fe + (phi1 + phi3) * colloid
                - (onPOC + aggregated) * theta_s - lam * F["SFe"])
    G["BFe"] = (0.3 * m["iron"] + large * p["theta_fe"] + (d["lin"] / 2 + d["quad"]) * d["theta_fe"]
                + (m["lin"] + 0.3 * upper) * MESO["fe"] + scavenging * GOC * free + 0.04 / 0.16 * bacteria_fe
                + phi2 * colloid + aggregated * theta_s - onGOC * theta_b - lam * F["BFe"])
    chi = 0.5 * torch.where(below, torch.exp(0.022 / DAY * (deep - A["z"]) / A["wG"]), torch.ones_like(T))
    equilibrium = 10 ** (6.44 - 968 / (T + 273.15))
    excess = (equilibrium - Si) / equilibrium
    dissolved = ((chi * 0.025 / DAY + (1 - chi) * 0.003 / DAY) * F["PSi"]
                 * (0.225 * (1 + T / 15) * excess + 0.775 * ((1 + T / 400) ** 4 * excess) ** 9))
    G["PSi"] = d["loss"] * theta_si - dissolved
    G["Si"] = dissolved - d["si"]
    calcite = rain * (0.5 * z["on"][0] + 0.75 * m["on"][0] + dead / 2)
    dissolving = 0.197 / DAY * (1 - A["Omega"]).clamp_min(0) * F["CaCO₃"]
    G["CaCO₃"] = calcite - dissolving
    # nutrients, carbon and oxygen
    thN, thP, rp, rn = 16 / 122, 1 / 122, 133 / 122, 32 / 122
    nitrified = 0.05 / DAY * NH4 / (1 + A["mlPAR"]) * (1 - anoxia)
    # (the nitrogen fixation needs a growth rate above 2.15 / s: none)
    up_no3, up_nh4 = (sum(s["muI"] * s[n] / (s["LN"] + TINY) for s in (p, d)) for n in ("LNO3", "LNH4"))
    oxic, anoxic = (1 - anoxia) * degraded, anoxia * degraded
    grown = p["muI"] + d["muI"]
    G["NO₃"] = nitrified + thN * (oxic - up_no3)
    G["NH₄"] = thN * (anoxic + inorganic - up_nh4) - nitrified
    G["PO₄"] = thP * (inorganic + degraded - grown)
    unused = sum(0.7 * g["iron"] - h["fe"] * g["e"] * g["food"] for g, h in ((z, MICRO), (m, MESO)))
    excess_fe = 1000 * scavenging * (Fe - (0.09 * DOC - 0.6).clamp_min(0.6)).clamp_min(0) * free
    G["Fe"] = (lam * F["SFe"] + unused + 0.35 * MESO["fe"] * upper - p["fe"] - d["fe"] - excess_fe
               - (phi1 + phi2 + phi3) * colloid - scavenging * (POC + GOC) * free - bacteria_fe)
    G["DIC"] = inorganic + degraded + dissolving - calcite - grown
    G["Alk"] = G["NH₄"] - G["NO₃"] - 2 * G["CaCO₃"]
    G["O₂"] = (rp * up_nh4 + (rp + rn) * up_no3 - (rp + rn) * oxic - rp * anoxic - rp * inorganic
               - rn * nitrified / thN)
    return G


MILLERO = dict(K1=(-25.50, 0.1271, 0.0, -0.00308, 0.0000877), K2=(-15.82, -0.0219, 0.0, 0.00113, -0.0001475),
               KB=(-29.48, 0.1622, -0.0026080, -0.00284, 0.0), KW=(-20.02, 0.1119, -0.001409, -0.00513, 0.0000794),
               KS=(-18.03, 0.0466, 0.000316, -0.00453, 0.00009), KF=(-9.78, -0.0090, -0.000942, -0.00391, 0.000054),
               KC=(-48.76, 0.5304, 0.0, -0.01176, 0.0003692))


def _calcite(T, S, z):
    """What the saturation state takes from T, S and the depth."""
    bar = z.abs() * 9.80665 * 1026 / 100000 + 0.0 * T
    c = _equilibrium(T, S)
    K = c["K"]
    c["KC"] = 10 ** (-171.9065 - 0.077993 * K + 2839.319 / K + 71.595 * torch.log10(K)
                     + (-0.77712 + 0.0028426 * K + 178.34 / K) * torch.sqrt(S) - 0.07711 * S + 0.0041249 * S ** 1.5)
    for n, a in MILLERO.items():
        volume, compress = a[0] + a[1] * T + a[2] * T * T, a[3] + a[4] * T
        c[n] = c[n] * torch.exp((-volume + 0.5 * compress * bar) * bar / (83.14472 * K))
    c["unit"], c["ca"] = 1e-3 / _density(T, S, bar), 0.0103 * S / 35
    return c


def _exact_pisces(case, seed):
    grid = _grid(case)
    st = _fields(case, grid, seed)
    names = _tracers(case)
    F = {n: _interior(grid, t).double() for n, t in zip(names, st["tracers"])}
    T, S = F["T"], F["S"]
    zc, zf, dz = _dev64(grid.zc), _dev64(grid.zf), _dev64(grid.dz)
    z = zc.view(-1, 1, 1)
    nothing = torch.zeros_like(zc[:1])
    wP = torch.cat([-2 / DAY * torch.ones_like(zc), nothing])
    wG = torch.cat([-30 / DAY + 170 / DAY * zc.clamp_max(0) / 5000, nothing])
    kw, e, chi = BANDS
    c = _calcite(T, S, z)
    share = (zf[1:] - zf[:-1].clamp_min(PISCES_MLD)).clamp_min(0).view(-1, 1, 1)
    share = torch.where(zf[:-1].view(-1, 1, 1) >= PISCES_MLD, dz.view(-1, 1, 1), share)

    def auxiliary(F, t):
        A = dict(z=z, shear=torch.where(z < PISCES_MLD, 0.01, 1.0))
        A["dl"], A["dl2"] = _day_length(PISCES_LATITUDE, t), _day_length(t, PISCES_LATITUDE)
        PAR0 = {"constant": 100.0, "diurnal": _daylight(t), "array": None}[case["light"]]
        PAR0 = st["surface"].double() if PAR0 is None else torch.full_like(T[0], PAR0)
        chl = F["PChl"] + F["DChl"]
        step = torch.cat([zc[:-1] - zc[1:], zc[-1:]]).view(-1, 1, 1)
        A["bands"] = [PAR0 / 3 * torch.exp((step * (kw[n] + chi[n] * chl ** e[n])).flip(0).cumsum(0).flip(0))
                      for n in range(3)]
        PAR = A["PAR"] = sum(A["bands"])
        # the first level below the top with a thousandth of the surface light
        dark = (PAR[:-1] <= 1e-3 * PAR0).double()
        k = dark * torch.arange(1, len(PAR), device=DEVICE).view(-1, 1, 1)
        k = k.max(0).values.long()[None] - 1
        j = k.clamp_min(0)
        lo, hi, zl = (v.expand_as(T).gather(0, i)[0] for v, i in ((PAR.log(), j), (PAR.log(), j + 1), (z, j)))
        depth = zl + (torch.log(1e-3 * PAR0) - lo) * (zl - z.expand_as(T).gather(0, j + 1)[0]) / (lo - hi)
        none = (k[0] < 0) | ~torch.isfinite(depth)
        A["zeu"] = torch.where(none, zc[0] - (zc[1] - zc[0]), depth)
        A["mlPAR"] = (PAR * share).sum(0) / share.sum(0)
        DIC = F["DIC"] * c["unit"]
        x = _hydrogen(c, DIC, F["Alk"] * c["unit"], F["Si"] * c["unit"])
        A["Omega"] = c["ca"] / c["KC"] * DIC * c["K1"] * c["K2"] / (x * x + c["K1"] * x + c["K1"] * c["K2"])
        A["wP"], A["wG"] = ((w[:-1] + w[1:]).view(-1, 1, 1) / 2 for w in (wP, wG))
        return A

    def tendencies(F, t, dt=0.0, step=0, stage=0):
        A = auxiliary(F, t)
        G = _pisces_tendencies(F, A)
        for n in ("POC", "SFe"):
            _sink(G, F, n, wP, dz)
        for n in ("GOC", "BFe", "PSi", "CaCO₃"):
            _sink(G, F, n, wG, dz)
        if case["gas"]:
            G["DIC"][-1] -= _co2_exchange(F["DIC"][-1], F["Alk"][-1], T[-1], S[-1])[1] / dz[-1]
            G["O₂"][-1] -= _o2_exchange(F["O₂"][-1], T[-1], S[-1]) / dz[-1]
        G["aux"] = A
        return G

    def parent(v):
        f = torch.zeros(grid.parent_shape, dtype=torch.float64, device=DEVICE)
        _interior(grid, f).copy_(v)
        return f

    if case["call"] == "hooks":
        G = tendencies(F, _clock(case))
        A = G["aux"]
        aux = (parent(A["PAR"]), [parent(b) for b in A["bands"]], parent(A["Omega"]), A["zeu"], A["mlPAR"])
        return aux, [parent(_interior(grid, g).double() + G[n]) for n, g in zip(names, st["G"])]
    _runge_kutta(F, names[:24], tendencies, case["steps"], case["dt"], _clock(case))
    return [parent(F[n]) for n in names[:24]]


def exact(case, seed):
    if case["kind"] == "points":
        p = _point_inputs(case, seed)
        return _co2_exchange(p["DIC"], p["Alk"], p["T"], p["S"], p["u10"], 420.0)
    if case["kind"] == "ensemble":
        return _exact_ensemble(case, seed)
    return _exact_pisces(case, seed) if case["kind"] == "pisces" else _exact_npd(case, seed)
