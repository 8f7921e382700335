"""The work that programs have this package do, as cases that can be timed and checked.

A case is one pass of a program: a coupled time step of one model, a step of an ensemble, the
update's phases called one by one, or the diagnostics between steps. Inputs are synthetic, made
on the GPU from a seed with the distributions of the package's own workloads (T, S, velocities,
atmosphere and radiation as in ``numericalearth_hip.generators``), and ``exact`` restates the
step in plain FP64 torch.

Bathymetry: "hills" is smoothed noise over the whole depth (the benchmark workload's, where less
than half of the cells lie above the bottom); "basins" has continents on about a third of the
area and mostly deep, stretched water columns, as the real ocean has.
"""
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "numericalearth.jl_amd"))

from numericalearth_hip import params as P  # noqa: E402
from numericalearth_hip.ensemble import Ensemble  # noqa: E402
from numericalearth_hip.generators import GridArrays, GridSpec, SourceSpec, SurfaceCase  # noqa: E402
from numericalearth_hip.generators import NE_BOUNDED, NE_FLAT, NE_PERIODIC  # noqa: E402
from numericalearth_hip.model import OceanOnlyModel, Phases  # noqa: E402

DT = 1200.0                 # the workloads' time step (s)
SNAPSHOTS = 3               # of the atmosphere and the radiation, 3 hours apart (JRA55-do's)
SNAPSHOT_INTERVAL = 10800.0
DEPTH = 3000.0
RADIUS = 6_371_000.0
LARGEST_CELLS = 1440 * 560 * 10   # listed; a drawn case has at most half of them


def _step(name, Nx, Ny, Nz, **kw):
    return _filled(dict(kw, kind="step", Nx=Nx, Ny=Ny, Nz=Nz), name)


def _filled(case, name=None):
    full = dict(kind="step", precision="fp64", Nx=1, Ny=1, Nz=10, periodic=True, bathymetry="hills", fluxes="edson",
                two_color=False, stepper="SplitRungeKutta3", members=0, sizes=0)
    full.update(case)
    return dict(full, name=name) if name else full


def listed():
    return [
        # the smallest request of a serving loop or member of an ensemble: one column, launch latency alone
        _step("column_fp64", 1, 1, 50, periodic=False),
        # a coarse global model (the CPU reference configuration): too little work to fill the chip
        _step("coarse_fp64", 90, 40, 10),
        # a ragged regional model at a quarter degree in the mixed form, continents, shortwave that penetrates
        _step("regional_mixed", 353, 137, 19, precision="mixed", periodic=False, bathymetry="basins", two_color=True),
        # a half-degree global model with the reference's other time stepper
        _step("half_ab2", 720, 280, 10, bathymetry="basins", stepper="QuasiAdamsBashforth2"),
        # bulk formulae other than similarity theory (Large & Yeager's), an odd-sized basin model
        _step("large_yeager_fp64", 481, 187, 23, bathymetry="basins", fluxes="large_yeager", two_color=True),
        # the headline workload: the quarter-degree global step, FP64 and mixed
        _step("quarter_fp64", 1440, 560, 10),
        _step("quarter_mixed", 1440, 560, 10, precision="mixed"),
        # calibration ensembles: uneven members, each with its own roughness parameters, one graph a step
        _filled(dict(kind="ensemble", members=12, sizes=5, fluxes="tuned", periodic=False), "ensemble_fp64"),
        _filled(dict(kind="ensemble", members=12, sizes=6, fluxes="tuned", periodic=False, precision="mixed"),
                "ensemble_mixed"),
        # a host program that calls the phases of the update and the tendency one by one
        _filled(dict(kind="phases", Nx=720, Ny=280, Nz=10, bathymetry="basins"), "phases_fp64"),
        # between steps: w from continuity, heat and salt content
        _filled(dict(kind="diagnostics", Nx=719, Ny=281, Nz=17, bathymetry="basins"), "diagnostics_fp64"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["ensemble", "phases", "diagnostics"])
    c = dict(kind=kind, periodic=rng.random() < 0.5, bathymetry=rng.choice(["hills", "basins"]),
             two_color=rng.random() < 0.3, fluxes=rng.choice(["edson", "edson", "tuned", "large_yeager"]))
    if kind in ("step", "ensemble"):
        c["precision"] = rng.choice(["fp64", "mixed"])
    if kind == "ensemble":
        c.update(members=rng.randint(2, 12), sizes=rng.randint(0, 10 ** 6), fluxes="tuned", two_color=False)
        return _filled(c)
    if kind == "step" and c["precision"] == "fp64" and rng.random() < 0.25:
        c["stepper"] = "QuasiAdamsBashforth2"
    while True:
        c.update(Nx=_log_int(rng, 1, 1440), Ny=_log_int(rng, 1, 560), Nz=_log_int(rng, 4, 60))
        if c["Nx"] * c["Ny"] * c["Nz"] <= LARGEST_CELLS // 2 and (c["Nx"] > 1) == (c["Ny"] > 1):
            break
    if c["Nx"] == 1:
        c["periodic"] = False
    return _filled(c)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _smooth(x, sigma_x, sigma_y):
    """Gaussian smoothing of a 2-D field by its Fourier transform (periodic)."""
    ky = torch.fft.fftfreq(x.shape[0], device=x.device, dtype=x.dtype)[:, None]
    kx = torch.fft.rfftfreq(x.shape[1], device=x.device, dtype=x.dtype)[None, :]
    f = torch.exp(-2 * math.pi ** 2 * ((sigma_x * kx) ** 2 + (sigma_y * ky) ** 2))
    return torch.fft.irfft2(torch.fft.rfft2(x) * f, s=x.shape)


def _bottom(case, gen, dev):
    Nx, Ny = case["Nx"], case["Ny"]
    if Nx == 1 and Ny == 1:
        return torch.full((1, 1), -DEPTH - 1.0, dtype=torch.float64, device=dev)
    noise = torch.randn(Ny, Nx, generator=gen, dtype=torch.float64, device=dev)
    if case["bathymetry"] == "hills":
        sigma = min(4.0, max(Nx, Ny) / 8.0) if not case["periodic"] else 4.0 * Nx / 1440.0
        s = _smooth(noise, sigma, sigma)
        D = -400.0 + (s - s.min()) / max(float(s.max() - s.min()), 1e-300) * (DEPTH + 400.0)
        land = D < 50.0
    else:
        s = _smooth(noise, Nx / 24.0, Ny / 12.0)
        rank = s.flatten().argsort().argsort().reshape(Ny, Nx).double() / max(1, Nx * Ny - 1)
        land = rank < 0.3
        D = 200.0 + 5500.0 * ((rank - 0.3).clamp(min=0) / 0.7) ** 0.6
    return torch.where(land, 0.0, -D.clamp(200.0, DEPTH))


def _inputs(case, seed):
    """Everything one model is made of, as FP64 tensors."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    f64 = dict(dtype=torch.float64, device=dev)
    randn = lambda *s: torch.randn(*s, generator=gen, **f64)  # noqa: E731
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    periodic = bool(case["periodic"])
    if periodic:
        lon, lat = (0.0, 360.0), (-70.0, 70.0)
    else:
        lon, lat = (20.0, 20.0 + 0.25 * Nx), (-0.125 * Ny, 0.125 * Ny)
        if Nx == 1:
            lat = (35.0, 35.25)
    dlon, dlat = (lon[1] - lon[0]) / Nx, (lat[1] - lat[0]) / Ny
    lam = lon[0] + (torch.arange(Nx, **f64) + 0.5) * dlon
    phi_f = lat[0] + torch.arange(Ny + 1, **f64) * dlat
    phi = lat[0] + (torch.arange(Ny, **f64) + 0.5) * dlat
    zf = torch.linspace(0.0, 1.0, Nz + 1, **f64)
    zf = -DEPTH * (1 - zf) ** (1.5 if case["bathymetry"] == "basins" else 1.0)
    dz, zc = zf[1:] - zf[:-1], 0.5 * (zf[1:] + zf[:-1])
    rlon, rlat = math.radians(dlon), math.radians(dlat)
    sin = torch.sin(torch.deg2rad(phi_f))
    g = dict(Nx=Nx, Ny=Ny, Nz=Nz, periodic=periodic, lon=lon, lat=lat, dz=dz, zc=zc, zf=zf, lam=lam, phi=phi, phi_f=phi_f,
             dyx=torch.full((Ny,), RADIUS * rlat, **f64), dxy=RADIUS * torch.cos(torch.deg2rad(phi_f)) * rlon,
             Az=RADIUS ** 2 * rlon * (sin[1:] - sin[:-1]))
    bottom = _bottom(case, gen, dev)
    kmin = (zc[:, None, None] <= bottom).sum(0)
    active = torch.arange(Nz, device=dev)[:, None, None] >= kmin
    g.update(bottom=bottom, kmin=kmin, active=active)
    cos2 = torch.cos(torch.deg2rad(phi)) ** 2
    T = 2.0 + 26.0 * cos2[None, :, None] * torch.exp(zc / 500.0)[:, None, None] + 0.1 * randn(Nz, Ny, Nx)
    S = 35.0 + 0.5 * randn(Nz, Ny, Nx)
    # velocities on open faces, without depth-mean transport; w by continuity
    pad = torch.zeros_like
    west = torch.roll(active, 1, 2) if periodic else torch.cat([pad(active[:, :, :1]), active[:, :, :-1]], 2)
    ou = torch.cat([west & active, (west & active)[:, :, :1] & periodic], 2)
    ov = torch.cat([pad(active[:, :1]), active[:, :-1] & active[:, 1:], pad(active[:, :1])], 1)
    vel = []
    for o in (ou, ov):
        x = 0.1 * randn(*o.shape)
        if periodic and o is ou:
            x[:, :, -1] = x[:, :, 0]
        h = dz[:, None, None] * o
        x = torch.where(o, x - (h * x).sum(0) / h.sum(0).clamp(min=1e-300), 0.0)
        vel.append(x * (0.0 if Nx == 1 and Ny == 1 else 1.0))
    u, v = vel
    Fu, Fv = g["dyx"][:, None] * u, g["dxy"][:, None] * v
    div = dz[:, None, None] * ((Fu[:, :, 1:] - Fu[:, :, :-1]) + (Fv[:, 1:] - Fv[:, :-1])) / g["Az"][:, None]
    w = torch.cat([torch.zeros(1, Ny, Nx, **f64), torch.where(active, -torch.cumsum(div * active, 0), 0.0)], 0)
    g.update(T=T, S=S, u=u, v=v, w=w)
    # prescribed atmosphere and radiation, twice as coarse
    Nxa, Nya = max(1, Nx // 2), max(1, Ny // 2)
    dla, dpa = (lon[1] - lon[0]) / Nxa, (lat[1] - lat[0]) / Nya
    phia = torch.deg2rad(lat[0] + (torch.arange(Nya, **f64) + 0.5) * dpa)[:, None]
    shape = (SNAPSHOTS, Nya, Nxa)
    ones = torch.ones(shape, **f64)
    Ta = 2.0 + 26.0 * torch.cos(phia) ** 2 * torch.exp(zc[-1] / 500.0) + 273.15 - 1.0 + randn(*shape)
    pa = 101325.0 * ones + 500.0 * randn(*shape)
    atmos = dict(u=8.0 * torch.sin(2.0 * phia) * ones + randn(*shape), v=2.0 * randn(*shape), T=Ta, p=pa,
                 q=0.8 * _saturation_humidity(Ta, pa, 1.0), rain=3e-5 * randn(*shape).abs(), snow=0.0 * ones)
    rad = dict(downwelling_shortwave=300.0 * torch.cos(phia) * ones, downwelling_longwave=350.0 + 10.0 * randn(*shape))
    g.update(Nxa=Nxa, Nya=Nya, dla=dla, dpa=dpa, atmos=atmos, rad=rad)
    return g


# ---------------------------------------------------------------------------
# Parameters
# ---------------------------------------------------------------------------

def _tuning(case, member):
    """(Charnock parameter, roughness factor) of a calibration member; the defaults otherwise."""
    if case["fluxes"] != "tuned":
        return 0.02, 1.0
    rng = random.Random(1000 * case["sizes"] + member)
    return rng.uniform(0.01, 0.02), rng.uniform(0.8, 1.2)


def _params(case, member=0):
    forcing = P.default_radiative_forcing() if case["two_color"] else None
    fluxes = None
    if case["fluxes"] == "large_yeager":
        fluxes = P.CoefficientBasedFluxes(P.LargeYeagerTransferCoefficients())
    p = P.to_params(fluxes, radiative_forcing=forcing)
    charnock, factor = _tuning(case, member)
    if case["fluxes"] == "tuned":
        p.charnock_parameter = charnock
        p.smooth_wall_parameter *= factor
        p.reynolds_scaling_A *= factor
    return p


def _members(case):
    """Sizes log-uniform between a column of 50 levels and a 360 x 140 x 20 region, one case each."""
    rng = random.Random(case["sizes"])
    out = []
    for _ in range(case["members"]):
        s = rng.random()
        n = [max(1, int(round(a ** (1 - s) * b ** s))) for a, b in ((1, 360), (1, 140), (50, 20))]
        if n[1] == 1:
            n[0] = 1
        out.append(dict(case, Nx=n[0], Ny=n[1], Nz=n[2]))
    return out


def _model(case, seed, member=0):
    g = _inputs(case, seed)
    np64 = lambda t: np.ascontiguousarray(t.cpu().numpy())  # noqa: E731
    tx = NE_PERIODIC if g["periodic"] else NE_BOUNDED
    spec = GridSpec(g["Nx"], g["Ny"], g["Nz"], longitude=g["lon"], latitude=g["lat"], z=(-DEPTH, 0.0), topology_x=tx)
    grid = GridArrays(spec=spec, dz=np64(g["dz"]), z_center=np64(g["zc"]), z_face=np64(g["zf"]), dy_xface=np64(g["dyx"]),
                      dx_yface=np64(g["dxy"]), Az=np64(g["Az"]), lambda_c=np64(g["lam"]), phi_c=np64(g["phi"]),
                      phi_f=np64(g["phi_f"]), bottom_height=np64(g["bottom"]), kmin=np64(g["kmin"].int()))
    src = SourceSpec(g["Nxa"], g["Nya"], tx if g["Nxa"] > 1 else NE_FLAT, NE_BOUNDED if g["Nya"] > 1 else NE_FLAT,
                     g["lon"][0], g["dla"], g["lat"][0], g["dpa"])
    times = np.arange(SNAPSHOTS) * SNAPSHOT_INTERVAL
    sc = SurfaceCase(grid=grid, T=np64(g["T"]), S=np64(g["S"]), u=np64(g["u"]), v=np64(g["v"]), w=np64(g["w"]),
                     atmos_grid=src, atmos={k: np64(x) for k, x in g["atmos"].items()}, atmos_times=times, rad_grid=src,
                     rad={k: np64(x) for k, x in g["rad"].items()}, rad_times=times.copy(), seed=int(seed))
    return OceanOnlyModel(sc, params=_params(case, member), precision=case["precision"], timestepper=case["stepper"])


def prepare(case, seed):
    case = _filled(case)
    if case["kind"] == "ensemble":
        models = [_model(c, 97 * seed + k, k) for k, c in enumerate(_members(case))]
        ensemble = Ensemble(models)
        ensemble.use_graph()
        return dict(case=case, models=models, ensemble=ensemble)
    model = _model(case, seed)
    return dict(case=case, model=model, phases=Phases(model) if case["kind"] == "phases" else None)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["kind"] == "ensemble":
        state["ensemble"].time_step(DT)
        if case["precision"] == "mixed":
            return [[m.T, m.S] for m in state["models"]]
        return [[m.T, m.S, m.net["J_T"], m.net["J_w"], m.net["tau_x"]] for m in state["models"]]
    m = state["model"]
    if case["kind"] == "diagnostics":
        m.update_vertical_velocity()
        return dict(w=m.w, heat=m.heat_content(), salt=m.budget(m.S))
    if case["kind"] == "phases":
        ph = state["phases"]
        ph.interp()
        ph.flux_solve()
        ph.freeze(DT)
        ph.assemble()
        ph.radiation()
        GT, GS = ph.tendency()
        return dict(_surface(m), G_T=GT, G_S=GS)
    m.time_step(DT)
    if case["precision"] == "mixed":
        # the FP32 state, and the heat fluxes and wind stress in the state's precision, as its output is written
        out = {k: m.fluxes[k].float() for k in ("sensible_heat", "latent_heat", "x_momentum")}
        return dict(out, T=m.T, S=m.S)
    return dict(_surface(m), T=m.T, S=m.S)


def _surface(m):
    return dict(fluxes=dict(m.fluxes), net=dict(m.net), radiative=dict(m.radiative), frazil=m.frazil_heat)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

# Share of a grid's cells above the bottom (hills 0.44 at a quarter degree; basins 0.64 of all cells, land
# included), and flops of one WENO5-Z reconstruction with its flux (about 75), 6 to a cell and stage for T and S.
ACTIVE = {"hills": 0.44, "basins": 0.64}


def work(case):
    case = _filled(case)
    if case["kind"] == "ensemble":
        each = [work(dict(c, kind="step")) for c in _members(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    columns = case["Nx"] * case["Ny"]
    share = 1.0 if columns == 1 else ACTIVE[case["bathymetry"]]
    cells = share * columns * case["Nz"]
    s = 8 if case["precision"] == "fp64" else 4
    # a stage reads u, v, w, T, S (later ones T0 and S0 too) and writes T, S; per column the coarse atmosphere in,
    # eight interface fluxes, Ts and six net fluxes out; 13 iterations of a fixed point of about 350 flops
    surface = columns * (7.25 * s + 14 * 8)
    solve = columns * (13 * 350 + 500)
    if case["kind"] == "diagnostics":
        return {"bytes": cells * 5 * s, "flops": cells * 16}
    if case["kind"] == "phases":
        return {"bytes": cells * 7 * s + 2 * surface, "flops": cells * 450 + solve}
    stages = 15 if case["stepper"] != "SplitRungeKutta3" else 25
    return {"bytes": cells * stages * s + surface, "flops": cells * (450 if stages == 15 else 1350) + solve}


# ---------------------------------------------------------------------------
# The step in plain FP64 torch
# ---------------------------------------------------------------------------

KELVIN, RHO, HEAT_CAPACITY, GRAVITY = 273.15, 1020.0, 3991.86795711963, 9.80665
GAS, M_DRY, M_VAPOR = 8.3144598, 0.02897, 0.018015
CP_V, CP_L, LH0, T_TR, P_TR = 1859.0, 4181.0, 2500800.0, 273.16, 611.657
EPS = M_DRY / M_VAPOR
HEIGHT = 10.0


def _saturation_humidity(T, p, x):
    Rv, dcp = GAS / M_VAPOR, CP_V - CP_L
    e = x * P_TR * (T / T_TR) ** (dcp / Rv) * torch.exp((LH0 - dcp * T_TR) / Rv * (1 / T_TR - 1 / T))
    e = torch.minimum(e, 0.999 * p)
    return e / EPS / (p - (1 - 1 / EPS) * e)


def _cp(q):
    cpd = GAS / M_DRY * 3.5
    return cpd + (CP_V - cpd) * q


def _edson(z):
    """The momentum and scalar stability functions of Edson et al. (2013)."""
    n, s = z.clamp(max=0.0), z.clamp(min=0.0)

    def free(c):
        f = (1 - c * n) ** (1 / 3)
        return 1.5 * torch.log((1 + f + f * f) / 3) - 3 ** 0.5 * torch.atan((1 + 2 * f) / 3 ** 0.5) + math.pi / 3 ** 0.5

    x2 = torch.sqrt(1 - 15 * n)
    x = torch.sqrt(x2)
    m1 = 2 * torch.log((1 + x) / 2) + torch.log((1 + x2) / 2) - 2 * torch.atan(x) + math.pi / 2
    f = n * n / (1 + n * n)
    e = torch.exp(-(0.35 * s).clamp(max=50.0))
    d = 5 / 0.35
    m = torch.where(z < 0, (1 - f) * m1 + f * free(10.15), -0.7 * s - 0.75 * (s - d) * e - 0.75 * d)
    h = torch.where(z < 0, (1 - f) * 2 * torch.log((1 + x2) / 2) + f * free(34.15),
                    -(1 + 2 / 3 * s) ** 1.5 - 2 / 3 * (s - 14.28) * e - 8.525)
    return m, h


def _edson_iteration(c, us, ts, qs):
    b = GRAVITY / c["Tv"] * (ts * (1 + (EPS - 1) * c["qo"]) + (EPS - 1) * c["Tv"] * qs)
    gust = (1.2 * ((-us * b).clamp(min=0) * 512.0) ** (1 / 3)).clamp(min=0.01)
    U = torch.sqrt(c["dU2"] + gust * gust)
    charnock, factor = c["tuning"]
    lu = (charnock * us * us / GRAVITY + 0.11 * factor * 1.5e-5 / us).clamp(max=1.0)
    lq = (5.85e-5 * factor / (lu * us / 1.5e-5) ** 0.72).clamp(max=1.6e-4)
    h = (2 * lu).clamp(min=HEIGHT)
    iL = 0.4 * b / (us * us)
    mh, sh = _edson(h * iL)
    xu = 0.4 / (torch.log(h / lu) - mh + _edson(lu * iL)[0])
    xq = 0.4 / (torch.log(h / lq) - sh + _edson(lq * iL)[1])
    return xu * U, xq * c["dth"], xq * c["dq"]


def _neutral_drag(U):
    U = U.clamp(min=0.5)
    return torch.where(U < 33.0, (2.7 / U + 0.142 + U / 13.09 - 3.14807e-10 * U ** 6) / 1000, 2.34e-3)


def _large_yeager_iteration(c, us, ts, qs):
    dU = torch.sqrt(c["dU2"]).clamp(min=0.5)
    b = GRAVITY / c["Tv"] * (ts * (1 + (EPS - 1) * c["qo"]) + (EPS - 1) * c["Tv"] * qs)
    z = HEIGHT * 0.4 * b / (us * us)
    x2 = torch.sqrt(1 - 16 * z.clamp(max=0))
    x = torch.sqrt(x2)
    stable = -5 * z.clamp(max=10.0)
    pm = torch.where(z > 0, stable, 2 * torch.log((1 + x) / 2) + torch.log((1 + x2) / 2) - 2 * torch.atan(x) + math.pi / 2)
    ph = torch.where(z > 0, stable, 2 * torch.log((1 + x2) / 2))
    U10 = (dU / (1 + torch.sqrt(us * us / (dU * dU)) / 0.4 * (0 - pm))).clamp(min=0.5)
    s = torch.sqrt(_neutral_drag(U10))
    ch, cq = s / 1000 * torch.where(z > 0, 18.0, 32.7), s / 1000 * 34.6
    Cd = s * s / (1 + s / 0.4 * (0 - pm)) ** 2
    xh, ratio = s / 0.4 * (0 - ph), torch.sqrt(Cd) / s
    Ch, Cq = ch * ratio / (1 + ch * xh), cq * ratio / (1 + cq * xh)
    return torch.sqrt(Cd) * dU, Ch / torch.sqrt(Cd) * c["dth"], Cq / torch.sqrt(Cd) * c["dq"]


def _axis(x, n, x0, dx, periodic):
    f = (x - (x0 + 0.5 * dx)) / dx
    if n == 1:
        z = torch.zeros_like(f, dtype=torch.long)
        return z, z, torch.zeros_like(f)
    lo = torch.floor(f)
    w, lo = f - lo, lo.long()
    return (lo % n, (lo + 1) % n, w) if periodic else (lo.clamp(0, n - 1), (lo + 1).clamp(0, n - 1), w)


def _interp(g, field, time):
    t = min(max(time / SNAPSHOT_INTERVAL, 0.0), SNAPSHOTS - 1.0)
    k = min(int(t), SNAPSHOTS - 2)
    a = field[k] + (t - k) * (field[k + 1] - field[k])
    x0, x1, wx = _axis(g["lam"], g["Nxa"], g["lon"][0], g["dla"], g["periodic"])
    y0, y1, wy = _axis(g["phi"], g["Nya"], g["lat"][0], g["dpa"], False)
    wy = wy[:, None]
    a = a[y0] * (1 - wy) + a[y1] * wy
    return a[:, x0] * (1 - wx) + a[:, x1] * wx


def _update(g, case, T, S, time, dt, member=0):
    """Fluxes from the state, the freeze clamp (T changes in place), net fluxes and radiation."""
    ua, va, Ta, pa, qa, rain, snow = (_interp(g, g["atmos"][k], time) for k in ("u", "v", "T", "p", "q", "rain", "snow"))
    SW, LW = (_interp(g, g["rad"][k], time) for k in ("downwelling_shortwave", "downwelling_longwave"))
    wet = g["active"][-1]
    zero = torch.zeros_like(ua)
    uo, vo = 0.5 * (g["u"][-1][:, 1:] + g["u"][-1][:, :-1]), 0.5 * (g["v"][-1][1:] + g["v"][-1][:-1])
    du, dv = ua - torch.where(wet, uo, 0.0), va - torch.where(wet, vo, 0.0)
    To = T[-1] + KELVIN
    qo = _saturation_humidity(To, pa, 0.98)
    c = dict(qo=qo, Tv=To * (1 + (EPS - 1) * qo), dU2=du * du + dv * dv, dq=qa - qo,
             dth=Ta + GRAVITY * HEIGHT / _cp(qa) - To, tuning=_tuning(case, member))
    step = _large_yeager_iteration if case["fluxes"] == "large_yeager" else _edson_iteration
    us, ts, qs = (zero + 1e-4 for _ in range(3))
    going = wet.clone()
    for _ in range(20 if case["fluxes"] == "large_yeager" else 100):
        nu, nt, nq = step(c, us, ts, qs)
        drift = (nu - us).abs() + (nt - ts).abs() + (nq - qs).abs()
        us, ts, qs = (torch.where(going, a, b) for a, b in ((nu, us), (nt, ts), (nq, qs)))
        going = going & ~(drift < 1e-8)
        if not bool(going.any()):
            break
    us, ts, qs = (torch.where(wet, x, 0.0) for x in (us, ts, qs))
    dU = torch.sqrt(du * du + dv * dv)
    rho = pa / (GAS / M_DRY * (1 + (EPS - 1) * qa) * Ta)
    Lv = LH0 + (CP_V - CP_L) * (Ta - T_TR)
    Ts = torch.where(wet, T[-1], 0.0)
    fx = dict(latent_heat=-rho * Lv * us * qs, sensible_heat=-rho * _cp(qa) * us * ts, water_vapor=-rho * us * qs,
              x_momentum=torch.where(dU == 0, 0.0, -rho * us * us * du / dU),
              y_momentum=torch.where(dU == 0, 0.0, -rho * us * us * dv / dU), friction_velocity=us,
              temperature_scale=ts, water_vapor_scale=qs, interface_temperature=Ts)
    Tm = -0.054 * S
    frazil = (-(RHO * HEAT_CAPACITY * (Tm - T).clamp(min=0)) * g["dz"][:, None, None] / dt).sum(0)
    torch.maximum(T, Tm, out=T)
    x, y = fx["x_momentum"], fx["y_momentum"]
    west = torch.roll(x, 1, 1) if g["periodic"] else torch.cat([zero[:, :1], x[:, :-1]], 1)
    south = torch.cat([zero[:1], y[:-1]], 0)
    up = 5.670374419e-8 * 0.97 * (Ts + KELVIN) ** 4
    down, short = 0.97 * LW, 0.95 * SW
    Jw = (rain + snow - fx["water_vapor"]) / RHO
    radiative = (up - down - (0.0 if case["two_color"] else short)) / (RHO * HEAT_CAPACITY)
    net = dict(tau_x=(x + west) / 2 / RHO, tau_y=(y + south) / 2 / RHO, J_S=zero, J_w=Jw, J_H=T[-1] * Jw,
               J_T=(fx["sensible_heat"] + fx["latent_heat"]) / (RHO * HEAT_CAPACITY) + radiative)
    net = {k: torch.where(wet, v, 0.0) for k, v in net.items()}
    return dict(fluxes=fx, net=net, frazil=frazil, J0=short / (RHO * HEAT_CAPACITY),
                radiative=dict(upwelling_longwave=up, downwelling_longwave=down, downwelling_shortwave=short))


def _weno(c, a, vel, dim, wrap):
    """Upwind-biased values at the N + 1 faces of a dimension, of the order that the active cells around allow."""
    c, a, vel = (x.movedim(dim, -1) for x in (c, a, vel))
    if wrap:
        at = (torch.arange(-3, c.shape[-1] + 3, device=c.device) % c.shape[-1])
        c, a = c[..., at], a[..., at]
    else:
        c, a = torch.nn.functional.pad(c, (3, 3)), torch.nn.functional.pad(a, (3, 3))
    n = c.shape[-1] - 5
    A = [a[..., k:k + n] for k in range(6)]
    two = A[2] & A[3]
    four = two & A[1] & A[4]
    six = four & A[0] & A[5]
    left = vel >= 0
    q = [torch.where(left, c[..., k:k + n], c[..., 5 - k:5 - k + n]) for k in range(5)]
    b = [13 / 12 * (q[0] - 2 * q[1] + q[2]) ** 2 + (q[0] - 4 * q[1] + 3 * q[2]) ** 2 / 4,
         13 / 12 * (q[1] - 2 * q[2] + q[3]) ** 2 + (q[1] - q[3]) ** 2 / 4,
         13 / 12 * (q[2] - 2 * q[3] + q[4]) ** 2 + (3 * q[2] - 4 * q[3] + q[4]) ** 2 / 4]
    r = [(2 * q[0] - 7 * q[1] + 11 * q[2]) / 6, (-q[1] + 5 * q[2] + 2 * q[3]) / 6, (2 * q[2] + 5 * q[3] - q[4]) / 6]
    w = [d * (1 + ((b[0] - b[2]) / (x + 1e-8)) ** 2) for d, x in zip((0.1, 0.6, 0.3), b)]
    five = sum(x * y for x, y in zip(w, r)) / (w[0] + w[1] + w[2])
    b = [(q[2] - q[1]) ** 2, (q[3] - q[2]) ** 2]
    w = [d * (1 + ((b[0] - b[1]) / (x + 1e-8)) ** 2) for d, x in zip((1 / 3, 2 / 3), b)]
    three = (w[0] * (3 * q[2] - q[1]) / 2 + w[1] * (q[2] + q[3]) / 2) / (w[0] + w[1])
    value = torch.where(six, five, torch.where(four, three, q[2]))
    return torch.where(two, vel * value, 0.0).movedim(-1, dim)


def _tendencies(g, case, T, S, up):
    a, dz, Az = g["active"], g["dz"][:, None, None], g["Az"][:, None]
    V, out = dz * Az, []
    zf = g["zf"][:, None, None] - g["zf"][-1]
    for c, flux in ((T, up["net"]["J_T"]), (S, up["net"]["J_S"] + S[-1] * up["net"]["J_w"])):
        G = torch.zeros_like(c)
        if g["Nx"] > 1 or g["Ny"] > 1:
            Fx = g["dyx"][:, None] * dz * _weno(c, a, g["u"], 2, g["periodic"])
            Fy = g["dxy"][:, None] * dz * _weno(c, a, g["v"], 1, False)
            Fz = Az * _weno(c, a, g["w"], 0, False)
            G = -((Fx[:, :, 1:] - Fx[:, :, :-1]) + (Fy[:, 1:] - Fy[:, :-1]) + (Fz[1:] - Fz[:-1])) / V
        if c is T and case["two_color"]:
            J = up["J0"] * (0.58 * torch.exp(zf / 0.35) + 0.42 * torch.exp(zf / 23.0))
            below = torch.nn.functional.pad(a[:-1], (0, 0, 0, 0, 1, 0))
            G = G + (J[1:] - torch.where(below, J[:-1], 0.0)) / dz
        G[-1] -= flux * Az / V[-1]
        out.append(torch.where(a, G, 0.0))
    return out


def _exact_model(case, seed, member=0):
    g = _inputs(case, seed)
    T, S = g["T"].clone(), g["S"].clone()
    if case["kind"] == "diagnostics":
        _update(g, case, T, S, 0.0, math.inf)
        V = torch.where(g["active"], g["dz"][:, None, None] * g["Az"][:, None], 0.0)
        return dict(w=g["w"], heat=float((RHO * HEAT_CAPACITY * V * T).sum()), salt=float((V * S).sum()))
    up = _update(g, case, T, S, 0.0, math.inf, member)
    names = ("fluxes", "net", "radiative", "frazil")
    if case["kind"] == "phases":
        up = _update(g, case, T, S, 0.0, DT)
        GT, GS = _tendencies(g, case, T, S, up)
        return dict({k: up[k] for k in names}, G_T=GT, G_S=GS)
    T1, S1 = T, S
    for beta in ((1.0,) if case["stepper"] == "QuasiAdamsBashforth2" else (1 / 3, 1 / 2, 1.0)):
        GT, GS = _tendencies(g, case, T1, S1, up)
        T1, S1 = T + beta * DT * GT, S + beta * DT * GS
    up = _update(g, case, T1, S1, DT, DT, member)
    return dict({k: up[k] for k in names}, T=T1, S=S1)


def exact(case, seed):
    case = _filled(case)
    if case["kind"] == "ensemble":
        out = []
        for k, c in enumerate(_members(case)):
            e = _exact_model(dict(c, kind="step"), 97 * seed + k, k)
            n = e["net"]
            out.append([e["T"], e["S"]] + ([] if case["precision"] == "mixed" else [n["J_T"], n["J_w"], n["tau_x"]]))
        return out
    e = _exact_model(case, seed)
    if case["kind"] == "step" and case["precision"] == "mixed":
        return {k: e["fluxes"][k] if k in e["fluxes"] else e[k]
                for k in ("sensible_heat", "latent_heat", "x_momentum", "T", "S")}
    return e
