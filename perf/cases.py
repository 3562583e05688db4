"""Performance cases of the transport steps, through their public entry points.

A case is one call (or the few calls that always go together) of a program
that steps GITM on one GPU: ``VerticalSolver.advance``, ``prepare``,
``sources``, ``exchange`` + ``horizontal``, ``VerticalBatch`` and the
differentiable ``adjoint.window``.  The grids are the repository's own: one
default GITM block of 9 x 9 columns x 50 levels, the 5-degree grid (2,592
columns), 2.5 degrees (10,368), 1 degree (64,800 columns x 100 levels).

``listed`` gives the named cases, ``draw`` one more of the same ranges,
``prepare`` the inputs a program holds before the call (made on the GPU from
the seed alone), ``run`` one pass, ``work`` the bytes and operations that a
pass cannot do without, and ``exact`` the same results from plain torch in
64 bits, written from the reference's formulas and sharing no code with the
package.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gitm_amd import adjoint, synth, vertical

DEV = "cuda"
F64 = torch.float64
NSP, NION = 6, 10
KB, AMU, R_EARTH = 1.3807e-23, 1.6726e-27, 6372.0e3
MASS = (16.0 * AMU, 32.0 * AMU, 28.0 * AMU, 14.0 * AMU, 30.0 * AMU, 4.0 * AMU)
VIB = (5.0, 7.0, 7.0, 5.0, 7.0, 5.0)
BASE = (1e17, 1e18, 4e18, 1e13, 1e14, 1e14)  # O O2 N2 N NO He near 100 km
DT = 2.0
STATE = ("nds", "vvel", "vel", "temp", "rho")
RUN_LENGTH = 500  # steps of a model run; the next one starts from the analysis again
PREP_OUT = ("nden", "gamma", "mmm", "tempunit", "eddy", "cmax", "press", "cp")
MEMBER_ALTS = (50, 60, 70, 80, 90, 100, 110, 120)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one process's default GITM block, where a step is
        # one column's latency plus the call's own cost
        dict(name="block_ausm", kind="advance", solver="ausm", columns=81, alts=50,
             stretched=False, ions=False),
        # the 5-degree grid, GITM's everyday resolution
        dict(name="5deg_ausm", kind="advance", solver="ausm", columns=2592, alts=50,
             stretched=False, ions=False),
        # the 1-degree grid, the headline workload
        dict(name="1deg_ausm", kind="advance", solver="ausm", columns=64800, alts=100,
             stretched=True, ions=False),
        # the other solver at 2.5 degrees
        dict(name="2p5deg_rusanov", kind="advance", solver="rusanov", columns=10368, alts=100,
             stretched=True, ions=False),
        # ion advection, which GITM has on by default
        dict(name="2p5deg_ausm_ions", kind="advance", solver="ausm", columns=10368, alts=50,
             stretched=False, ions=True),
        # the step's inputs and time step from the state, every step
        dict(name="1deg_prepare", kind="prepare", columns=64800, alts=100, stretched=True),
        # conduction and viscosity, every step
        dict(name="1deg_sources", kind="sources", columns=64800, alts=100, stretched=True),
        # halo exchange and horizontal step of the 1-degree blocks
        dict(name="1deg_horizontal", kind="horizontal", blocks_lon=40, blocks_lat=20, alts=100,
             nlons=9, nlats=9, ions=False, topography=False),
        # terrain-following levels (one level after the other) with ions
        dict(name="5deg_horizontal_topo", kind="horizontal", blocks_lon=8, blocks_lat=4,
             alts=50, nlons=9, nlats=9, ions=True, topography=True),
        # a ragged ensemble: prep with a step per member, then one step of all
        dict(name="ensemble_10", kind="ensemble", members=10, columns=6480, first=0),
        # forward and backward through ten steps (sensitivities, 5 degrees)
        dict(name="5deg_window", kind="window", columns=2592, alts=50, steps=10),
        # the drop-in on host arrays: one process's 2 x 2 blocks
        dict(name="host_ausm", kind="host", solver="ausm", columns=324, alts=50,
             stretched=False, ions=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("advance", "advance", "advance", "prepare", "sources", "horizontal",
                       "ensemble", "window", "host"))
    # levels: GITM's range, from short test columns to the tall ones
    alts = _log_int(rng, 20, 180)
    if kind in ("advance", "host"):
        most = 324 if kind == "host" else min(40000, 40000 * 50 // alts)
        return dict(kind=kind, solver=rng.choice(("ausm", "ausm", "rusanov")),
                    columns=_log_int(rng, 9, most), alts=alts,
                    stretched=rng.random() < 0.5, ions=rng.random() < 0.35)
    if kind in ("prepare", "sources"):
        return dict(kind=kind, columns=_log_int(rng, 81, min(64800, 64800 * 100 // alts)),
                    alts=alts, stretched=rng.random() < 0.5)
    if kind == "horizontal":
        topo = rng.random() < 0.3
        return dict(kind=kind, blocks_lon=2 * rng.randint(1, 8 if topo else 14),
                    blocks_lat=rng.randint(1, 6 if topo else 14),
                    alts=_log_int(rng, 10, 50 if topo else 110),
                    nlons=rng.choice((9, 9, 9, 6, 12, 15)), nlats=rng.choice((9, 9, 9, 7, 12)),
                    ions=rng.random() < 0.4, topography=topo)
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(2, 10), columns=_log_int(rng, 81, 6480),
                    first=rng.randint(0, 7))
    return dict(kind=kind, columns=_log_int(rng, 81, 2592), alts=_log_int(rng, 20, 120),
                steps=rng.randint(2, 6))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=F64)


def _levels(alts, stretched):
    """Altitudes of levels -1..alts+2: uniform 100-600 km, or spacings that
    grow geometrically from 1.5 to 15 km."""
    k = np.arange(-1, alts + 3, dtype=np.float64)
    if not stretched:
        return 100.0e3 + (k - 0.5) * 500.0e3 / alts
    dz = 1.5e3 * (10.0 ** (1.0 / (alts - 2))) ** np.arange(alts + 3, dtype=np.float64)
    a = np.empty(alts + 4)
    a[2] = 100.0e3 + 0.5 * dz[0]
    a[3:] = a[2] + np.cumsum(dz[1:alts + 2])
    a[1], a[0] = a[2] - dz[0], a[2] - 2 * dz[0]
    return a


def _m(shape=(1, NSP, 1)):
    return torch.tensor(MASS, device=DEV, dtype=F64).view(shape)


def _prep_fields(nds, temp, rho, vvel):
    """calc_pressure, calc_rates' mean mass, the eddy coefficient and cMax on
    every level (calc_pressure.f90:17-86, calc_rates.Earth.f90:34-50,
    Earth.f90:376-411, calc_timestep.f90:113-118)."""
    n = nds.sum(1)
    vib2 = torch.tensor(VIB, device=nds.device, dtype=nds.dtype).view(1, NSP, 1) - 2.0
    gamma = (nds / vib2).sum(1) * 2.0 / n + 1.0
    cp = (vib2 * nds * (KB / _m())).sum(1) / (2.0 * n)
    mmm = (_m() * nds / (n + 1.0)[:, None]).sum(1)
    press = temp * rho
    eddy = torch.where(press > 0.01, torch.full_like(press, 50.0),
                       torch.where(press > 0.005, 50.0 * (press - 0.005) / (0.01 - 0.005),
                                   torch.zeros_like(press)))
    cs = torch.sqrt(gamma * temp)
    cmax = vvel.abs().amax(1) + cs
    return dict(nden=n, gamma=gamma, cp=cp, mmm=mmm, tempunit=mmm / KB, press=press, eddy=eddy,
                cmax=cmax), cs


def _columns(n, alts, stretched, ions, seed, tinf=1000.0):
    """A hydrostatic atmosphere under a Bates temperature profile with 5 %
    noise, winds of 50 m/s and species winds of 5 m/s."""
    g, L = _gen(seed), alts + 4
    alt = torch.tensor(_levels(alts, stretched), device=DEV, dtype=F64).expand(n, L).contiguous()
    nlat = max(1, int(math.sqrt(n / 2.0)))
    nlon = -(-n // nlat)
    c = torch.arange(n, device=DEV)
    lat = ((c // nlon).to(F64) + 0.5) * math.pi / nlat - 0.5 * math.pi
    lon = ((c % nlon).to(F64) + 0.5) * 2 * math.pi / nlon
    d = alt.clone()
    d[:, 1:-1] = 0.5 * (alt[:, 2:] - alt[:, :-2])
    d[:, 0], d[:, -1] = d[:, 1], d[:, -2]
    invr = 1.0 / (R_EARTH + alt)
    grav = -9.5 * (R_EARTH * invr) ** 2
    tk = (tinf - (tinf - 200.0) * torch.exp(-0.02e-3 * (alt - 100.0e3).clamp(min=0.0))) * \
        torch.exp(math.log(1.05) * _randn(g, n, L))
    # ln n_s from level 0 (just below 100 km) up and down
    step = torch.log(tk[:, :-1] / tk[:, 1:])
    h = 0.5 * (grav[:, 1:] + grav[:, :-1]) * (alt[:, 1:] - alt[:, :-1]) / \
        (KB * 0.5 * (tk[:, 1:] + tk[:, :-1]))
    inc = step[:, None] + _m() * h[:, None]
    ln = torch.zeros(n, NSP, L, device=DEV, dtype=F64)
    ln[:, :, 1:] = torch.cumsum(inc, 2)
    ln = ln - ln[:, :, 1:2] + torch.log(torch.tensor(BASE, device=DEV, dtype=F64)).view(1, NSP, 1)
    nds = torch.exp(ln)
    vvel = 5.0 * _randn(g, n, NSP, L)
    vel = torch.empty(n, 3, L, device=DEV, dtype=F64)
    vel[:, :2] = 50.0 * _randn(g, n, 2, L)
    rho = (_m() * nds).sum(1)
    vel[:, 2] = (_m() * nds * vvel).sum(1) / rho
    mmm = (_m() * nds / (nds.sum(1) + 1.0)[:, None]).sum(1)
    temp = tk / (mmm / KB)
    p, _ = _prep_fields(nds, temp, rho, vvel)
    out = dict(nds=nds, vvel=vvel, vel=vel, temp=temp, rho=rho, tempunit=p["tempunit"],
               mmm=p["mmm"], gamma=p["gamma"], cmax=p["cmax"], eddy=p["eddy"], alt=alt,
               grav=grav, invr=invr, dalt=d, coslat=torch.cos(lat))
    if ions:
        z = alt / 1e3
        i = torch.empty(n, NION, L, device=DEV, dtype=F64)
        i[:, 0] = 1e12 * torch.exp(1 - (z - 300) / 60 - torch.exp(-(z - 300) / 60)) * \
            torch.exp(0.05 * _randn(g, n, L)) + 1e3
        i[:, 1] = 1e11 * torch.exp(1 - (z - 120) / 20 - torch.exp(-(z - 120) / 20)) * \
            torch.exp(0.05 * _randn(g, n, L)) + 1e3
        for s in range(2, NION - 1):
            i[:, s] = 1e6 + 1e3 * s
        i[:, NION - 1] = i[:, :NION - 1].sum(1)
        out["ions"] = i
        out["ivel"] = 20.0 * _randn(g, n, 3, L)
        out["sza"] = torch.acos((torch.cos(lat) * torch.cos(lon - math.pi)).clamp(-1, 1))
        out["mlat"] = torch.rad2deg(lat)
    return {k: v.contiguous() for k, v in out.items()}


def _source_fields(c, seed):
    """Conductivity ~ T^0.75 and viscosity ~ T^0.69 within 5 %, a Gaussian
    heating at 150 km."""
    g = _gen(seed + 1000003)
    n, L = c["temp"].shape
    p, _ = _prep_fields(c["nds"], c["temp"], c["rho"], c["vvel"])
    tk = c["temp"] * c["tempunit"]
    visc = 1.3e-5 * (tk / 300.0) ** 0.69 * torch.exp(0.05 * _randn(g, n, L))
    q = 1.0e-5 * torch.exp(-((c["alt"] - 150.0e3) / 20.0e3) ** 2)
    return dict(cp=p["cp"], kappa_temp=3.6e-4 * tk ** 0.75 * torch.exp(0.05 * _randn(g, n, L)),
                visc_coef=visc,
                visc_coef_s=(visc[:, None] * c["nds"] / p["nden"][:, None]).contiguous(),
                raddist=R_EARTH + c["alt"], heating=q / (p["cp"] * c["tempunit"]))


def _blocks(case, seed):
    """A smooth global atmosphere on blocks with halo cells: waves in
    longitude and latitude whose phases and amplitudes come from the seed."""
    g = _gen(seed)
    nbl, nbt, nA, nlo, nla = (case[k] for k in ("blocks_lon", "blocks_lat", "alts", "nlons",
                                                "nlats"))
    nb, L, NLo, NLg = nbl * nbt, nA + 4, nlo + 4, nla + 4
    u = torch.rand(12, generator=g, device=DEV, dtype=F64)
    ph = (2 * math.pi * u[:6]).view(6, 1, 1, 1, 1)
    am = 0.5 + u[6:]
    dlon, dlat = 2 * math.pi / (nbl * nlo), math.pi / (nbt * nla)
    b = torch.arange(nb, device=DEV)
    ii = torch.arange(-1, nlo + 3, device=DEV)
    jj = torch.arange(-1, nla + 3, device=DEV)
    lon = (((b % nbl) * nlo)[:, None] + ii[None]).to(F64).sub(0.5).mul(dlon)
    lat = (((b // nbl) * nla)[:, None] + jj[None]).to(F64).sub(0.5).mul(dlat).sub(0.5 * math.pi)
    alt = 100.0e3 + (torch.arange(L, device=DEV, dtype=F64) - 1.5) * 5.0e3
    shp = (nb, L, NLg, NLo)
    X = lon[:, None, None, :].expand(shp)
    Y = lat[:, None, :, None].expand(shp)
    Z = alt[None, :, None, None].expand(shp)
    Rr = R_EARTH + Z
    cy, sx = torch.cos(Y), torch.sin(X + ph[0])
    T = (1000.0 - 800.0 * torch.exp(-(Z - 100.0e3) / 50.0e3)) * \
        (1.0 + 0.05 * am[0] * cy * sx + 0.02 * torch.sin(3 * Y + ph[1]))
    m = _m((1, NSP, 1, 1, 1))
    sp = torch.arange(NSP, device=DEV, dtype=F64).view(1, NSP, 1, 1, 1)
    X5, Y5, Z5 = X[:, None], Y[:, None], Z[:, None]
    nds = torch.tensor(BASE, device=DEV, dtype=F64).view(1, NSP, 1, 1, 1) * \
        torch.exp(-(Z5 - 100.0e3) * m * 9.5 / (KB * 600.0)) * \
        (1.0 + 0.1 * torch.sin(2 * X5 + sp + ph[2]) * torch.cos(Y5) +
         0.03 * torch.cos(Y5 * (sp + 1)))
    rho = (m * nds).sum(1)
    ntot = nds.sum(1)
    vel = torch.stack([80.0 * am[1] * cy * torch.sin(X + 2 * Y + ph[3]) + 20.0 * torch.sin(3 * X),
                       60.0 * am[2] * torch.sin(2 * Y) * torch.cos(X - ph[4]) +
                       10.0 * torch.cos(2 * X + Y),
                       3.0 * torch.sin(X + Y + ph[5]) * (Z / 400.0e3)], 1)
    vvel = vel[:, 2:3] + (1.0 + 0.3 * sp) * torch.cos(X5 * (sp % 3 + 1) + Y5 + ph[0])
    vib2 = torch.tensor(VIB, device=DEV, dtype=F64).view(1, NSP, 1, 1, 1) - 2.0
    temp = T / (rho / ntot / KB)
    gamma = 1.0 + 2.0 / ntot * (nds / vib2).sum(1)
    o = dict(rho=rho, temp=temp, vel=vel, vvel=vvel, nds=nds, gamma=gamma, itemp=temp.clone(),
             etemp=2.0 * temp)
    if case["ions"]:
        base = torch.tensor((2e11, 1e11, 5e10, 1e9, 1e10, 1e8, 1e8, 1e9, 1e8), device=DEV,
                            dtype=F64).view(1, 9, 1, 1, 1)
        q = torch.arange(9, device=DEV, dtype=F64).view(1, 9, 1, 1, 1)
        i9 = base * torch.exp(-((Z5 - 300e3) / 150e3) ** 2) * \
            (1.0 + 0.2 * torch.cos(X5 + 0.3 * q + ph[1]) * torch.cos(Y5)) + 1.0e3
        o["ions"] = torch.cat([i9, i9.sum(1, keepdim=True)], 1)
        o["ivel"] = torch.stack([150.0 * sx * cy, 100.0 * torch.cos(2 * X) * torch.sin(Y),
                                 10.0 * torch.sin(Y + ph[2])], 1)
        o["ivel_par"] = torch.stack([40.0 * torch.cos(X + ph[3]) * torch.sin(2 * Y),
                                     60.0 * torch.sin(Y) * torch.cos(X),
                                     30.0 * torch.sin(Y + ph[4]) * (Z / 400.0e3)], 1)
        for key, ang, cnt in (("grad_lon", lon, nlo), ("grad_lat", lat, nla)):
            dm = ang[:, 2:cnt + 2] - ang[:, 1:cnt + 1]
            dp = ang[:, 3:cnt + 3] - ang[:, 2:cnt + 2]
            r2 = (dm / dp) ** 2
            inv = 1.0 / (r2 * dp + dm)
            o[key] = torch.stack([-inv, inv * (1 - r2), inv * r2], 1)
    # cell sizes and distances between cell centres; on this uniform grid the
    # radius does not change along a row
    fl = torch.cos(lat).abs().clamp(min=0.01)[:, None, :, None]
    o["dlat_fb"] = (dlat * Rr).contiguous()
    o["dlon_fb"] = (dlon * Rr * fl).contiguous()
    o["inv_dlat_gb"] = o["inv_dlat_fb"] = 1.0 / o["dlat_fb"]
    o["inv_dlon_gb"] = o["inv_dlon_fb"] = 1.0 / o["dlon_fb"]
    o["inv_dlat_fb"], o["inv_dlon_fb"] = o["inv_dlat_fb"].clone(), o["inv_dlon_fb"].clone()
    o["raddist"], o["invr"] = Rr, 1.0 / Rr
    o["latitude"], o["cos_lat"] = lat, torch.cos(lat)
    o["tan_lat"] = torch.tan(lat).abs().clamp(max=100.0) * torch.sign(lat)
    if case["topography"]:
        fade = torch.exp(-(Z - 100.0e3) / 200.0e3)
        A = Z + (3000.0 * (1 + torch.sin(2 * X + ph[5]) * cy) + 800.0 * torch.cos(3 * Y)) * fade
        da = A.clone()
        da[:, 1:-1] = 0.5 * (A[:, 2:] - A[:, :-2])
        da[:, 0], da[:, -1] = da[:, 1], da[:, -2]
        o["dalt"] = da
        o["dalt_dlon"] = 6000.0 * torch.cos(2 * X + ph[5]) * cy * fade / \
            (Rr * cy.abs().clamp(min=0.01))
        o["dalt_dlat"] = (-3000.0 * torch.sin(2 * X + ph[5]) * torch.sin(Y) -
                          2400.0 * torch.sin(3 * Y)) * fade / Rr
    cs = torch.sqrt(gamma * temp)
    inner = (slice(None), slice(1, nA + 3), slice(1, nla + 3), slice(1, nlo + 3))
    o["cmax"] = torch.stack([(vel[:, 0].abs() + cs)[inner], (vel[:, 1].abs() + cs)[inner],
                             (vvel.abs().amax(1) + cs)[inner]], 1)
    # the CFL step of calc_timestep_horizontal at 0.25
    c = o["cmax"][:, :, 1:-1, 1:-1, 1:-1]
    own = (slice(None), slice(2, -2), slice(2, -2), slice(2, -2))
    dt = 0.25 / float((c[:, 0] * o["inv_dlon_gb"][own] + c[:, 1] * o["inv_dlat_gb"][own]).max())
    return {k: v.contiguous() for k, v in o.items()}, dt


def _members(case, seed):
    return [_columns(case["columns"], MEMBER_ALTS[(case["first"] + i) % 8], False, False,
                     seed * 64 + i, tinf=700.0 + 70.0 * ((3 * i) % 11))
            for i in range(case["members"])]


def _seeds(case, seed):
    """Adjoints of the window's outputs: a loss of order one per field."""
    g = _gen(seed + 2000003)
    n, L = case["columns"], case["alts"] + 4
    c = _columns(n, case["alts"], False, False, seed)
    scale = dict(nds=1.0 / c["nds"], vvel=0.1 * torch.ones_like(c["vvel"]),
                 vel=0.02 * torch.ones_like(c["vel"]), temp=1.0 / c["temp"], rho=1.0 / c["rho"])
    return [_randn(g, *c[k].shape) * scale[k] for k in STATE]


def _heat(c):
    return 1.0e-5 * torch.exp(-((c["alt"] - 150.0e3) / 20.0e3) ** 2)


# ---------------------------------------------------------------------------
# what a program holds, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    s = _prepare(case, seed)
    # the fields that a pass steps in place, and the analysis they start from
    held = {"ensemble": s.get("members"), "horizontal": [s.get("grid")]}.get(
        case["kind"], [s.get("cols")])
    s["stepped"] = [(d, k) for d in held if d is not None and case["kind"] != "prepare"
                    for k in STATE + ("ions",) if k in d]
    copy = np.copy if case["kind"] == "host" else torch.clone
    s["analysis"] = [copy(d[k]) for d, k in s["stepped"]]
    s["passes"] = 0
    return s


def _prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "ensemble":
        s["solver"] = vertical.VerticalSolver()
        s["members"] = [dict(c, logns=torch.zeros_like(c["nds"]), nden=torch.zeros_like(c["temp"]))
                        for c in _members(case, seed)]
        s["batch"] = vertical.VerticalBatch(s["solver"], s["members"])
        s["params"] = synth.StepParams(dt=DT)
        s["prep"] = synth.PrepParams(fixed_dt=DT)
        return s
    if kind == "horizontal":
        s["solver"] = vertical.VerticalSolver()
        s["grid"], s["dt"] = _blocks(case, seed)
        return s
    c = _columns(case["columns"], case["alts"], case.get("stretched", False),
                 case.get("ions", False), seed)
    s["solver"] = vertical.VerticalSolver()
    s["params"] = synth.StepParams(dt=DT, use_ion_advection=bool(case.get("ions")))
    if kind in ("advance", "host"):
        c["logns"], c["nden"] = torch.zeros_like(c["nds"]), torch.zeros_like(c["temp"])
        s["cols"] = {k: v.cpu().numpy() for k, v in c.items()} if kind == "host" else c
    elif kind == "prepare":
        for k in PREP_OUT:
            c[k] = torch.zeros_like(c["temp"])
        s["cols"], s["prep"] = c, synth.PrepParams()
    elif kind == "sources":
        src = _source_fields(c, seed)
        for k, like in (("conduction", "temp"), ("viscosity", "vel"), ("vert_viscosity", "vvel")):
            src[k] = torch.zeros_like(c[like])
        s["cols"], s["src"] = c, src
    else:  # window
        s["state"] = {k: c[k].requires_grad_(True) for k in STATE}
        s["heat"] = _heat(c).requires_grad_(True)
        s["fixed"] = {k: c[k] for k in adjoint.GEOMETRY}
        s["seeds"] = _seeds(case, seed)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if s["passes"] == RUN_LENGTH:
        s["passes"] = 0
        for (d, k), a in zip(s["stepped"], s["analysis"]):
            d[k][...] = a
    s["passes"] += 1
    if kind in ("advance", "host"):
        step = s["solver"].advance if kind == "advance" else s["solver"].advance_host
        step(s["cols"], s["params"], case["solver"])
        return {k: s["cols"][k] for k in STATE + ("logns", "nden") +
                (("ions",) if case["ions"] else ())}
    if kind == "prepare":
        dt = s["solver"].prepare(s["cols"], s["prep"])
        return dict({k: s["cols"][k] for k in PREP_OUT}, dt=dt)
    if kind == "sources":
        s["solver"].sources(s["cols"], s["src"], DT)
        return dict({k: s["cols"][k] for k in ("temp", "vel", "vvel")},
                    **{k: s["src"][k] for k in ("conduction", "viscosity", "vert_viscosity")})
    if kind == "horizontal":
        g = s["grid"]
        s["solver"].exchange(g, case["blocks_lon"], use_ion_advection=case["ions"])
        s["solver"].horizontal(g, s["dt"], use_ion_advection=case["ions"],
                               use_improved_ion_advection=case["ions"],
                               use_topography=case["topography"])
        return {k: g[k] for k in STATE + ("itemp", "etemp") +
                (("ions", "ivel_par") if case["ions"] else ())}
    if kind == "ensemble":
        dt = s["batch"].prepare(s["prep"])
        s["batch"].advance(s["params"], "ausm", dt=dt)
        return [dt] + [{k: m[k] for k in STATE} for m in s["members"]]
    out = adjoint.window(s["state"], s["heat"], s["solver"], s["fixed"], s["params"],
                         case["steps"])
    grads = torch.autograd.grad([out[k] for k in STATE],
                                [s["state"][k] for k in STATE] + [s["heat"]], s["seeds"])
    return dict({k: out[k].detach() for k in STATE},
                **{"g_" + k: v for k, v in zip(STATE + ("heat",), grads)})


def work(case):
    """Bytes: each input read once, each output written once.  Operations:
    those of the column and cell formulas, a division, root or
    transcendental as one (AUSM counted over the column code, 10.9e3 per level
    and step; the others by hand)."""
    kind = case["kind"]
    if kind == "ensemble":
        lev = sum(case["columns"] * (MEMBER_ALTS[(case["first"] + i) % 8] + 4)
                  for i in range(case["members"]))
        return {"bytes": lev * 8.0 * (17 + 1 + 4 + 24 + 7 + 5), "flops": lev * 1.1e4}
    if kind == "horizontal":
        nb = case["blocks_lon"] * case["blocks_lat"]
        own = nb * case["nlons"] * case["nlats"] * case["alts"]
        full = nb * (case["nlons"] + 4) * (case["nlats"] + 4) * case["alts"]
        nv = 17 + (2 if case["ions"] else 0)
        carried = 19 + (13 if case["ions"] else 0)
        return {"bytes": 8.0 * (carried * (own + 2 * (full - own)) + (nv + 11) * full + nv * own),
                "flops": own * 4.0 * nv * 120}
    lev = case["columns"] * (case["alts"] + 4.0)
    if kind in ("advance", "host"):
        ions = 9 + 1 + 10 if case["ions"] else 0
        return {"bytes": lev * 8.0 * (26 + 24 + ions),
                "flops": lev * (1.1e4 if case["solver"] == "ausm" else 4.5e3)}
    if kind == "prepare":
        return {"bytes": lev * 8.0 * (15 + 8), "flops": lev * 60.0}
    if kind == "sources":
        return {"bytes": lev * 8.0 * (32 + 20), "flops": lev * 9 * 60.0}
    # a window: each step forward, recomputed and reversed (about as many
    # operations again as the forward); the state, heat, geometry and
    # gradients once
    return {"bytes": lev * 8.0 * (18 + 4 + 17 + 17 + 18), "flops": lev * case["steps"] * 3.0e4}


# ---------------------------------------------------------------------------
# the same results from plain torch in 64 bits
# ---------------------------------------------------------------------------
BETA = 2.0
OMEGA = 2.0 * 3.141592653589793 / (24.0 * 3600.0)
PHOTO = (3, 4)  # N(4S) and NO: photochemical at the bottom
F1, F2 = 0.6250000, 0.0416667
D0 = ((0.0, 0.969, 0.969, 0.969, 0.715, 3.440), (0.969, 0.0, 0.715, 0.969, 0.715, 3.208),
      (0.969, 0.715, 0.0, 0.969, 0.527, 2.939), (0.969, 0.969, 0.969, 0.0, 0.969, 2.939),
      (0.715, 0.715, 0.527, 0.969, 0.0, 2.939), (3.440, 3.208, 2.939, 2.939, 2.939, 0.0))
DEXP = ((0.0, 0.774, 0.774, 0.774, 0.750, 0.749), (0.774, 0.0, 0.750, 0.774, 0.750, 0.710),
        (0.774, 0.750, 0.0, 0.774, 0.810, 0.718), (0.774, 0.774, 0.774, 0.0, 0.774, 0.718),
        (0.750, 0.750, 0.810, 0.774, 0.0, 0.718), (0.749, 0.710, 0.718, 0.718, 0.718, 0.0))
THERMAL_DIFFUSION = (0.0, 0.0, 0.0, 0.0, 0.0, -0.38)


def _mc(up, dn):
    """Limiter_mc (ModLimiter.f90:16-36)."""
    mid = (up + dn) * 0.5
    pos = torch.minimum(torch.minimum(BETA * up, BETA * dn), mid)
    neg = torch.maximum(torch.maximum(BETA * up, BETA * dn), mid)
    zero = torch.zeros_like(mid)
    return torch.where((up > 0) & (dn > 0), pos, torch.where((up < 0) & (dn < 0), neg, zero))


def _one_sided(h1, h2, h3, h4):
    """Weights of the one-sided five-point slope (set_vertical_bcs.Earth.f90
    :228-248)."""
    H2, H3, H4 = h1 + h2, h1 + h2 + h3, h1 + h2 + h3 + h4
    return (-(H2 * H3 * H4 + h1 * H3 * H4 + h1 * H2 * H4 + h1 * H2 * H3) / (h1 * H2 * H3 * H4),
            (H2 * H3 * H4) / (h1 * h2 * (h2 + h3) * (h2 + h3 + h4)),
            -(h1 * H3 * H4) / (H2 * h2 * h3 * (h3 + h4)),
            (h1 * H2 * H4) / (H3 * (h3 + h2) * h3 * h4),
            -(h1 * H2 * H3) / (H4 * (h2 + h3 + h4) * (h3 + h4) * h4))


def _wsum(w, v):
    return sum(a * b for a, b in zip(w, v))


class _Column:
    """Per-level constants of one step's columns ([column, level], levels
    -1..nAlts+2 at 0..L-1; cells 2..L-3)."""

    def __init__(self, c):
        alt, self.dC, self.invr, self.gam = c["alt"], c["dalt"], c["invr"], c["gamma"]
        cent = (c["coslat"] * OMEGA) ** 2
        self.cent, self.cor = cent[:, None], (2 * c["coslat"] * OMEGA)[:, None]
        self.eg = c["grav"] + self.cent / self.invr
        self.grav, self.eddy, self.mmm, self.gm1 = c["grav"], c["eddy"], c["mmm"], c["gamma"] - 1
        d = alt[:, 1:] - alt[:, :-1]
        self.dF = torch.cat([d[:, :1], d], 1)
        self.iF = 1.0 / self.dF
        cm = c["cmax"]
        self.cmf = torch.cat([cm[:, :1], 0.5 * torch.maximum(cm[:, :-1], cm[:, 1:])], 1)
        self.mgh = torch.cat([self.eg[:, :1], 0.5 * (self.eg[:, 1:] + self.eg[:, :-1])], 1)
        t = 1.0 + torch.tanh((alt - 160.0e3) / 15.0e3)
        inside = torch.zeros_like(alt)
        inside[:, 2:-2] = 1.0

        def blend(lo, hi):
            a, b = math.log(lo), math.log(hi)
            return torch.exp(a + 0.5 * (b - a) * t) * inside
        self.kp, self.ku = blend(1.0e-19, 1.0e-09), blend(0.25, 0.50)
        rd = 1.0 / self.invr
        r = 0.5 * (rd[:, 1:] + rd[:, :-1])
        self.am, self.ap = r[:, 1:-2] ** 2, r[:, 2:-1] ** 2
        self.vol = (r[:, 2:-1] ** 3 - r[:, 1:-2] ** 3) / 3.0
        self.hf = 0.35 * torch.exp(-(alt - alt[:, 1:2]) / 45.0e3)
        g = c["gamma"]
        sl = _mc((g[:, 2:] - g[:, 1:-1]) * self.iF[:, 2:], (g[:, 1:-1] - g[:, :-2]) * self.iF[:, 1:-1])
        # faces k|k+1, k = 0..nAlts (left cell at index 1..L-3)
        self.gL = g[:, 1:-2] + 0.5 * sl[:, :-1] * self.dF[:, 1:-2]
        self.gR = g[:, 2:-1] - 0.5 * sl[:, 1:] * self.dF[:, 2:-1]
        h1, h2, h3, h4 = (self.dF[:, 1:-3], self.dF[:, 2:-2], self.dF[:, 3:-1], self.dF[:, 4:])
        m2, m3, m4 = h2 + h1, h3 + h2 + h1, h4 + h3 + h2 + h1
        self.w5 = (h2 * h3 * (h3 + h4) / (h1 * m2 * m3 * m4),
                   -m2 * h3 * (h3 + h4) / (h1 * h2 * (h2 + h3) * (h2 + h3 + h4)),
                   (h2 * h3 * (h3 + h4) + m2 * h3 * (h3 + h4) - m2 * h2 * (h3 + h4) -
                    m2 * h2 * h3) / (m2 * h2 * h3 * (h3 + h4)),
                   m2 * h2 * (h4 + h3) / (m3 * (h2 + h3) * h3 * h4),
                   -m2 * h2 * h3 / (m4 * (h2 + h3 + h4) * (h3 + h4) * h4))
        f = self.dF
        self.ca = [w[:, None] for w in _one_sided(f[:, 3], f[:, 4], f[:, 5], f[:, 6])]
        self.cb = [w[:, None] for w in _one_sided(f[:, 2], f[:, 3], f[:, 4], f[:, 5])]
        self.ct = [[-w[:, None] for w in _one_sided(f[:, -3 + t], f[:, -4 + t], f[:, -5 + t],
                                                    f[:, -6 + t])] for t in (0, 1)]
        if "sza" in c:
            self.ivu = c["ivel"][:, 2, 2:-2]
            ml = c["mlat"]
            self.plasma = (c["sza"] > math.pi / 2) & (((ml > 30) & (ml < 70)) |
                                                      ((ml > -60) & (ml < -30)))

    def slope_and_flux(self, v):
        """4th-order limited gradient and Rusanov dissipation of [.., field,
        level] on cells (vertical_solver_ausm.f90:1007-1090)."""
        def e(a):
            return a[:, None]
        iF, dF = self.iF, self.dF
        up4 = e(iF[:, 3:-1]) * 2.0 * (F1 * (v[..., 3:-1] - v[..., 2:-2]) -
                                      F2 * (v[..., 4:] - v[..., 1:-3]))
        dn4 = e(iF[:, 2:-2]) * 2.0 * (F1 * (v[..., 2:-2] - v[..., 1:-3]) -
                                      F2 * (v[..., 3:-1] - v[..., :-4]))
        s = _mc(up4, dn4)
        lo = _mc((v[..., 2:3] - v[..., 1:2]) * e(iF[:, 2:3]), (v[..., 1:2] - v[..., 0:1]) * e(iF[:, 1:2]))
        hi = _mc((v[..., -1:] - v[..., -2:-1]) * e(iF[:, -1:]),
                 (v[..., -2:-1] - v[..., -3:-2]) * e(iF[:, -2:-1]))
        s = torch.cat([lo, s, hi], -1)  # levels 0..nAlts+1
        vv = v[..., 1:-1]
        right = vv - 0.5 * s * e(dF[:, 1:-1])
        left = vv + 0.5 * s * e(dF[:, 2:])
        L0, R0, L1, R1 = left[..., :-2], right[..., 1:-1], left[..., 1:-1], right[..., 2:]
        dC = e(self.dC[:, 2:-2])
        cm0, cm1 = e(self.cmf[:, 2:-2]), e(self.cmf[:, 3:-1])
        return 0.5 * (L1 + R1 - L0 - R0) / dC, (cm1 * (R1 - L1) - cm0 * (R0 - L0)) / dC

    def faces(self, v):
        """Left and right states of faces 0|1 .. nAlts|nAlts+1
        (calc_kt_facevalues, :2073-2117)."""
        iF, dF = self.iF[:, None], self.dF[:, None]
        s = _mc((v[..., 2:] - v[..., 1:-1]) * iF[..., 2:], (v[..., 1:-1] - v[..., :-2]) * iF[..., 1:-1])
        return (v[..., 1:-2] + 0.5 * s[..., :-1] * dF[..., 1:-2],
                v[..., 2:-1] - 0.5 * s[..., 1:] * dF[..., 2:-1])

    def log_gradient(self, v):
        return _wsum((w[:, None] for w in self.w5),
                     (v[..., :-4], v[..., 1:-3], v[..., 2:-2], v[..., 3:-1], v[..., 4:]))


def _bcs(K, U):
    """set_vertical_bcs (no MSIS, no tides) on the state dict U: LR, T, VE, VN,
    VU [column, level], LN, W [column, species, level], ION [column, 9, level]."""
    LN, W, T, m = U["LN"], U["W"], U["T"], _m()
    ca, cb = K.ca, K.cb
    d1, d0, dm1 = K.dF[:, 2:3], K.dF[:, 1:2], K.dF[:, 0:1]
    photo = torch.zeros(1, NSP, device=T.device, dtype=torch.bool)
    photo[0, list(PHOTO)] = True
    no = torch.zeros_like(photo)
    no[0, 4] = True
    oxygen = torch.zeros_like(photo)
    oxygen[0, 0] = True
    l = [LN[..., q] for q in range(7)]
    d = _wsum(ca, l[2:7])
    p0 = torch.where(d <= 0, l[2], l[2] - d1 * d)
    p0 = torch.where(no & (p0 < l[2] - 0.333), l[2] - 0.333, p0)
    d = _wsum(cb, [p0] + l[2:6])
    pm = torch.where(d <= 0, p0, p0 - d0 * d)
    pm = torch.where(no & (pm < p0 - 0.333), p0 - 0.333, pm)
    ish = -K.mgh[:, 1:2] * (0.5 * (K.mmm[:, 1:2] + K.mmm[:, 0:1])) / (T[:, 1:2] * KB)
    hm = torch.where(oxygen, l[1], l[1] + ish * dm1)
    n0, nm = torch.where(photo, p0, l[1]), torch.where(photo, pm, hm)
    w = [W[..., q] for q in range(7)]
    w0 = w[2] - d1 * _wsum(ca, w[2:7])
    wm = w0 - d0 * _wsum(cb, [w0] + w[2:6])
    flip = photo & (w[2] > 0)
    w0r, wmr = torch.where(flip, -w[2], w0), torch.where(flip, -w[2], wm)
    mm = m[..., 0]

    def ghost(ln, wbulk):
        ns = torch.exp(ln)
        sr = (mm * ns).sum(1, keepdim=True)
        return torch.log(sr), (ns * mm * wbulk).sum(1, keepdim=True) / sr
    lr0, vu0 = ghost(n0, w0)
    lrm, vum = ghost(nm, wm)
    tn = T[:, -3:-2]
    wn, wn1 = W[..., -3], W[..., -4]
    out = photo & (wn < 0)
    wt1, wt2 = torch.where(out, -wn, wn), torch.where(out, -wn1, wn)
    i1 = -K.mgh[:, -2:-1] * mm / (tn * KB)
    i2 = -K.mgh[:, -1:] * mm / (tn * KB)
    l1 = LN[..., -3] - i1 * K.dF[:, -2:-1]
    l2 = l1 - i2 * K.dF[:, -1:]
    z = torch.zeros_like(tn)
    vt = U["VU"][:, -3:-2].abs()

    def top(lnv):
        return torch.log((mm * torch.exp(lnv)).sum(1, keepdim=True))

    def cat(a, b, mid, y, x):
        return torch.cat([a, b, mid[..., 2:-2], y, x], -1)
    V = dict(LN=cat(nm[..., None], n0[..., None], LN, l1[..., None], l2[..., None]),
             W=cat(wmr[..., None], w0r[..., None], W, wt1[..., None], wt2[..., None]),
             LR=cat(lrm, lr0, U["LR"], top(l1), top(l2)), T=cat(T[:, 1:2], T[:, 1:2], T, tn, tn),
             VE=cat(z, z, U["VE"], U["VE"][:, -3:-2], U["VE"][:, -3:-2]),
             VN=cat(z, z, U["VN"], U["VN"][:, -3:-2], U["VN"][:, -3:-2]),
             VU=cat(vum, vu0, U["VU"], vt, vt))
    if "ION" in U:
        i = U["ION"].clone()
        i[..., 0] = i[..., 1] = i[..., 2]
        tec = (K.dF[:, 2:-2] * i[:, 0, 2:-2]).sum(1) / 1e16
        keep = (K.plasma & (tec < 2.0))[:, None]
        for t in (0, 1):
            jk = i.shape[-1] - 2 + t
            ln = [torch.log(i[..., jk - q]) for q in range(6)]
            dn = _wsum(K.ct[t], ln[1:])
            dn = torch.minimum(dn, -0.001 * ln[0] / K.dF[:, -3:-2])
            i[..., jk] = torch.where(keep, i[..., jk], torch.exp(ln[1] + dn * K.dF[:, jk:jk + 1]))
        V["ION"] = i
    return V


def _friction(dt, w, nt, ns, glc, eddy, T):
    """calc_neutral_friction.f90:47-106 on [column, species, cell]."""
    a, x = [], [w[:, i] for i in range(NSP)]
    for i in range(NSP):
        row = []
        for q in range(NSP):
            dij = 1.0e-4 * (1.0e17 * D0[i][q] * T ** DEXP[i][q]) / (nt * 1.0e-6) if q != i else None
            row.append(dt * KB * T / MASS[i] * ns[:, q] / nt / dij if q != i else None)
        total = sum(c for c in row if c is not None)
        a.append([1.0 + total if c is None else -c for c in row])
    # dominant by rows, so elimination in the natural order is stable
    for p in range(NSP):
        for i in range(p + 1, NSP):
            f = a[i][p] / a[p][p]
            for q in range(p + 1, NSP):
                a[i][q] = a[i][q] - f * a[p][q]
            x[i] = x[i] - f * x[p]
    for i in range(NSP - 1, -1, -1):
        for q in range(i + 1, NSP):
            x[i] = x[i] - a[i][q] * x[q]
        x[i] = x[i] / a[i][i]
    return torch.stack(x, 1) - eddy[:, None] * glc


def _cells(a):
    return a[..., 2:-2]


def _ausm_stage(K, U, dt):
    """advance_vertical_1stage_ausm (vertical_solver_ausm.f90:436-999): the new
    values on cells."""
    m = _m()
    T, VE, VN, VU, W = U["T"], U["VE"], U["VN"], U["VU"], U["W"]
    NS = torch.exp(U["LN"])
    rhos, rho, nt = m * NS, torch.exp(U["LR"]), NS.sum(1)
    te = nt * KB * T / K.gm1 + 0.5 * rho * (VU ** 2 + VN ** 2 + VE ** 2)
    glc = K.log_gradient(torch.log(rhos / rho[:, None]))
    grad, diff = K.slope_and_flux(torch.stack([T, VE, VN], 1))
    # hydrostatic densities from level 0
    tm = 0.5 * (T[:, 1:] + T[:, :-1])
    fac = (T[:, 1:-1] / T[:, 2:])[:, None] * torch.exp(
        K.dF[:, None, 2:] * m * K.mgh[:, None, 2:] / (KB * tm[:, None, 1:]))
    ns0 = NS[..., 1:2]
    ishb = -0.5 * (K.mmm[:, 0:1] + K.mmm[:, 1:2]) * K.mgh[:, 1:2] / (KB * tm[:, :1])
    below = ns0 * (T[:, 1:2] / T[:, 0:1] * torch.exp(K.dF[:, :1] * ishb))[:, None]
    hns = torch.cat([below, ns0, ns0 * torch.cumprod(fac, -1)], -1)
    hrho = m * hns
    sub = (rhos - hrho).abs() / rhos <= 1.0
    HL, HR = (torch.exp(v) for v in K.faces(torch.log(hns * KB * T[:, None])))
    VL, VR = K.faces(W)
    RL, RR = (torch.exp(v) for v in K.faces(torch.log(rhos)))
    PL, PR = (torch.exp(v) for v in K.faces(torch.log(NS * T[:, None] * KB)))
    hv = K.faces(torch.stack([VE, VN], 1))
    VEL, VNL, VER, VNR = hv[0][:, 0], hv[0][:, 1], hv[1][:, 0], hv[1][:, 1]
    bRL, bRR, bPL, bPR = RL.sum(1), RR.sum(1), PL.sum(1), PR.sum(1)
    VUL, VUR = (RL * VL).sum(1) / bRL, (RR * VR).sum(1) / bRR
    k2L, k2R = VUL ** 2 + VEL ** 2 + VNL ** 2, VUR ** 2 + VER ** 2 + VNR ** 2
    gL, gR = K.gL, K.gR
    EL, ER = bPL / (gL - 1) + 0.5 * bRL * k2L, bPR / (gR - 1) + 0.5 * bRR * k2R
    cL = torch.sqrt(2 * (gL - 1) / (gL + 1) * (0.5 * k2L + gL / (gL - 1) * bPL / bRL))
    cR = torch.sqrt(2 * (gR - 1) / (gR + 1) * (0.5 * k2R + gR / (gR - 1) * bPR / bRR))
    CS = torch.minimum(cL * cL / torch.maximum(cL, VUL),
                       cR * cR / torch.maximum(cR, -VUR))[:, None]
    ML, MR = VL / CS, VR / CS
    M2 = 0.5 * (ML * ML + MR * MR)
    MZ = torch.sqrt(M2.clamp(min=1.0e-19).clamp(max=1.0))
    FA = MZ * (2.0 - MZ)
    mp = torch.where(ML.abs() >= 1, 0.5 * (ML + ML.abs()),
                     0.25 * (ML + 1) ** 2 * (1 + 0.5 * (ML - 1) ** 2))
    mn = torch.where(MR.abs() >= 1, 0.5 * (MR - MR.abs()),
                     -0.25 * (MR - 1) ** 2 * (1 + 0.5 * (MR + 1) ** 2))
    f1 = (1.0 - M2).clamp(min=0.0)
    mps, mhps, mrs = 0.5 * (PL + PR), 0.5 * (HL + HR), 0.5 * (RL + RR)
    rvd = RR * VR - RL * VL

    def side(cell):
        """The flux of faces k|k+1 as the cell at index ``cell`` sees it."""
        sh = sub[..., cell]
        dp = torch.where(sh, (PR - HR) - (PL - HL), PR - PL)
        mpv = K.kp[:, None, cell] * f1 * dp / (mrs * CS * (FA * CS + K.dC[:, None, cell] / dt))
        nv = CS * (mp + mn - mpv)
        npr = torch.where(sh, mps - mhps, mps) - 0.5 * K.ku[:, None, cell] * CS * rvd
        fr = torch.where(nv >= 0, RL * nv, RR * nv)
        fm = torch.where(nv >= 0, RL * VL * nv, RR * VR * nv)
        bnv = ((RL + RR) * nv).sum(1) / (bRL + bRR)
        pos = bnv >= 0
        ef = torch.where(pos, (EL + bPL) * bnv, (ER + bPR) * bnv)
        fe = torch.where(pos, bRL * VEL * bnv, bRR * VER * bnv)
        fn = torch.where(pos, bRL * VNL * bnv, bRR * VNR * bnv)
        return fr, fm, npr, ef, fe, fn
    plus = [a[..., 1:] for a in side(slice(1, -2))]   # upper faces of the cells
    minus = [a[..., :-1] for a in side(slice(2, -1))]  # lower faces
    ap, am, vol = K.ap, K.am, K.vol

    def div(q, e=False):
        if e:
            return (ap * plus[q] - am * minus[q]) / vol
        return (ap[:, None] * plus[q] - am[:, None] * minus[q]) / vol[:, None]
    dC = _cells(K.dC)[:, None]
    rsf, msf = div(0), div(1) + (plus[2] - minus[2]) / dC
    ef, mfe, mfn = div(3, True), div(4, True), div(5, True)
    rs, rh, W0, eg = _cells(rhos), _cells(rho), _cells(W), _cells(K.eg)
    nrs = rs - dt * rsf
    nns = nrs / m
    nrho, nnt = nrs.sum(1), nns.sum(1)
    nm = rs * W0 - dt * msf + dt * torch.where(_cells(sub), rs - _cells(hrho), rs) * eg[:, None]
    ve, vn = _cells(VE), _cells(VN)
    tdc = torch.tensor(THERMAL_DIFFUSION, device=T.device, dtype=F64).view(1, NSP, 1)
    w = nm / nrs + (dt * (vn ** 2 + ve ** 2) * _cells(K.invr) + dt * K.cor * ve)[:, None] - \
        dt * tdc * KB * grad[:, None, 0] / m
    nve = (rh * ve - dt * mfe) / nrho + _cells(K.hf) * dt * diff[:, 1]
    nvn = (rh * vn - dt * mfn) / nrho + _cells(K.hf) * dt * diff[:, 2]
    nte = _cells(te) - dt * ef + dt * rh * _cells(VU) * eg
    w = _friction(dt, w, nnt, nns, glc, _cells(K.eddy), _cells(T)).clamp(-1000.0, 1000.0)
    nvu = (w * nrs).sum(1) / nrho
    np_ = (nte - 0.5 * nrho * (nvu ** 2 + nvn ** 2 + nve ** 2)) * _cells(K.gm1)
    N = dict(LN=torch.log(nns), LR=torch.log(nrho), W=w, VE=nve, VN=nvn, VU=nvu,
             T=np_ / (KB * nnt))
    return _ion_stage(K, U, N, dt)


def _ion_stage(K, U, N, dt):
    if "ION" in U:
        g, d = K.slope_and_flux(U["ION"][:, :2])
        i = _cells(U["ION"])
        N["ION"] = torch.cat([i[:, :2] - dt * K.ivu[:, None] * g + dt * d, i[:, 2:]], 1)
    return N


def _rusanov_stage(K, U, dt):
    """advance_vertical_1stage (vertical_solver_rusanov.f90:387-686)."""
    m = _m()
    NS = torch.exp(U["LN"])
    rho = torch.exp(U["LR"])
    bulk = torch.stack([U["T"], U["VE"], U["VN"], U["VU"]], 1)
    ga, da = K.slope_and_flux(bulk)
    gl, dl = K.slope_and_flux(U["LN"])
    gw, dw = K.slope_and_flux(U["W"])
    glc = K.log_gradient(torch.log(m * NS / rho[:, None]))
    T, ve, vn, vu = (_cells(U[k]) for k in ("T", "VE", "VN", "VU"))
    ir, W = _cells(K.invr), _cells(U["W"])
    divv = ga[:, 3] + 2 * vu * ir
    nln = _cells(U["LN"]) - dt * (gw + 2 * W * ir[:, None] + W * gl) + dt * dl
    tdc = torch.tensor(THERMAL_DIFFUSION, device=T.device, dtype=F64).view(1, NSP, 1)
    w = W - dt * (W * gw - ((vn ** 2 + ve ** 2) * ir)[:, None] + T[:, None] * gl * KB / m +
                  ga[:, None, 0] * KB / m - _cells(K.grav)[:, None]) + dt * dw - W / 1.0e9
    w = w + (dt * (K.cent / ir + K.cor * ve))[:, None] - dt * tdc * KB * ga[:, None, 0] / m
    ns, rh = _cells(NS), _cells(rho)
    w = _friction(dt, w, ns.sum(1), ns, glc, _cells(K.eddy), T).clamp(-1000.0, 1000.0)
    N = dict(LN=nln, W=w, VU=(w * m * ns).sum(1) / rh, VE=ve - dt * vu * ga[:, 1] + dt * da[:, 1],
             VN=vn - dt * vu * ga[:, 2] + dt * da[:, 2],
             T=T - dt * (vu * ga[:, 0] + _cells(K.gm1) * T * divv) + dt * da[:, 0],
             LR=torch.log((m * torch.exp(nln)).sum(1)))
    return _ion_stage(K, U, N, dt)


def _inside(U, new):
    """The ghost levels of U with the cells ``new``."""
    return {k: torch.cat([U[k][..., :2], new[k], U[k][..., -2:]], -1) for k in U}


def _step(c, dt, solver="ausm", ions=False):
    """One vertical step of the columns c (advance_vertical.f90:84-219)."""
    K = _Column(c)
    U = dict(LN=torch.log(c["nds"]), W=c["vvel"], LR=torch.log(c["rho"]),
             T=c["temp"] * c["tempunit"], VE=c["vel"][:, 0], VN=c["vel"][:, 1],
             VU=c["vel"][:, 2])
    if ions:
        U["ION"] = c["ions"][:, :9]
    U = _bcs(K, U)
    Y = {k: _cells(v) for k, v in U.items()}
    y_ion = U.get("ION")
    S, acc = U, None
    for n in range(4):
        old = {k: _cells(v) for k, v in S.items()}
        if solver == "ausm":
            new = _ausm_stage(K, S, (0.5 * dt, 0.5 * dt, dt, 0.5 * dt)[n])
            d = {k: new[k] - old[k] for k in new}
            nxt = {k: Y[k] + d[k] for k in d}
            if n == 0:
                acc = {k: nxt[k] - Y[k] for k in d}
            elif n < 3:
                acc = {k: acc[k] + (2.0 if n == 1 else 1.0) * nxt[k] for k in d}
            else:
                nxt = {k: (acc[k] + d[k]) / 3.0 for k in d}
        else:
            new = _rusanov_stage(K, S, dt)
            d = {k: new[k] - old[k] for k in new}
            acc = d if n == 0 else {k: acc[k] + (2.0 if n < 3 else 1.0) * d[k] for k in d}
            nxt = {k: Y[k] + ((0.5, 0.5, 1.0, None)[n] * d[k] if n < 3 else acc[k] / 6.0)
                   for k in d}
        S = _inside(S, nxt)
        if ions:  # the boundary reads the ghost ions of the step's first state
            S["ION"] = torch.cat([y_ion[..., :2], nxt["ION"], y_ion[..., -2:]], -1)
        S = _bcs(K, S)
    out = dict(nds=torch.exp(S["LN"]), vvel=S["W"], vel=torch.stack([S["VE"], S["VN"], S["VU"]], 1),
               temp=S["T"] / c["tempunit"], rho=torch.exp(S["LR"]), logns=S["LN"])
    out["nden"] = out["nds"].sum(1)
    if ions:
        i = S["ION"].clone()
        i[..., 2:-2] = i[..., 2:-2].clamp(min=1.0)
        out["ions"] = torch.cat([i, i.sum(1, keepdim=True)], 1)
    return out


def _exact_sources(c, f):
    """calc_conduction.f90:19-244 and calc_viscosity.f90:4-189: two half steps
    and a full one of each implicit diffusion solve, then 2 H - F."""
    m = _m()
    rd2 = f["raddist"] ** 2
    rho, eddy, T, tu = c["rho"], c["eddy"], c["temp"], c["tempunit"]
    n, L = T.shape
    wind = f["visc_coef"] + rho * eddy
    diff = torch.cat([(f["kappa_temp"] * rd2)[:, None], (wind * rd2)[:, None].expand(n, 2, L),
                      ((4.0 / 3.0) * f["visc_coef_s"] + m * c["nds"] * eddy[:, None]) *
                      rd2[:, None]], 1)
    mass = torch.cat([(rho * f["cp"] * rd2)[:, None], (rho * rd2)[:, None].expand(n, 2, L),
                      m * c["nds"] * rd2[:, None]], 1)
    q0 = torch.cat([T[:, None], c["vel"][:, :2], c["vvel"]], 1)
    unit = torch.cat([tu[:, None], torch.ones(n, 8, L, device=T.device, dtype=F64)], 1)
    alt = c["alt"]
    du, dl = (alt[:, 2:-1] - alt[:, 1:-2])[:, None], (alt[:, 1:-2] - alt[:, :-3])[:, None]
    r = du / dl  # levels 0..nAlts
    du12, du22 = (du * (1 + r)) ** 2, 0.5 * (dl * du + du * du)
    rt = ((alt[:, -1:] - alt[:, -2:-1]) / (alt[:, -2:-1] - alt[:, -3:-2]))[:, None]
    dut, dlt = (alt[:, -1:] - alt[:, -2:-1])[:, None], (alt[:, -2:-1] - alt[:, -3:-2])[:, None]
    d0 = diff[..., 2:-2]
    r, du12, du22 = r[..., 1:], du12[..., 1:], du22[..., 1:]  # levels 1..nAlts
    dd = diff[..., 3:-1] - r * r * diff[..., 1:-3] - (1 - r * r) * d0
    lo, up = d0 / du22 * r - dd / du12 * r * r, d0 / du22 + dd / du12
    mid = -d0 / du22 * (1 + r) - dd / du12 * (1 - r * r)

    def solve(q, dt):
        told = q * unit
        mm = dt / mass
        b = -1.0 / mm[..., 2:-2] + mid
        d = -told[..., 2:-2] / mm[..., 2:-2]
        at = rt * (1 + rt) * diff[..., -2:-1] * mm[..., -2:-1] / (0.5 * (dlt * dut + dut * dut))
        a = torch.cat([lo, at], -1)
        b = torch.cat([b, -(1.0 + at)], -1)
        d = torch.cat([d, -told[..., -2:-1]], -1)
        cc = torch.cat([up, torch.zeros_like(at)], -1)
        cps, dps = [torch.zeros_like(d[..., 0])], [told[..., 1]]
        for i in range(d.shape[-1]):
            den = b[..., i] - cps[-1] * a[..., i]
            dps.append((d[..., i] - dps[-1] * a[..., i]) / den)
            cps.append(cc[..., i] / den)
        t = [dps[-1]]
        for i in range(len(dps) - 2, -1, -1):
            t.append(dps[i] - cps[i] * t[-1])
        new = torch.stack(t[::-1], -1)
        res = torch.zeros_like(q)
        res[..., 1:-1] = new - told[..., 1:-1]
        return res
    r1 = solve(q0, DT / 2)
    s1 = q0 + r1 / unit
    h = s1 + solve(s1, DT / 2) / unit
    rc = solve(q0, DT)
    inc = (2.0 * h - (q0 + rc / unit)) - q0
    inc[..., 0] = 0.0
    inc[..., -1] = 0.0
    rc[..., 0] = 0.0
    rc[..., -1] = 0.0
    heat = torch.zeros_like(T)
    heat[:, 2:-2] = DT * f["heating"][:, 2:-2]
    vup = rc[:, 8]
    vel = c["vel"].clone()
    vel[:, :2] += inc[:, 1:3]
    vel[:, 2] += vup
    return dict(temp=T + heat + inc[:, 0], vel=vel, vvel=c["vvel"] + inc[:, 3:],
                conduction=inc[:, 0], viscosity=torch.cat([inc[:, 1:3], vup[:, None]], 1),
                vert_viscosity=inc[:, 3:])


def _fill_halo(case, g):
    """exchange_messages_sphere.f90:4-95 for the blocks of one device: halo
    cells of levels 1..nAlts from the global grid (past a pole the mirrored
    row half way round), then the horizontal winds past a pole turned."""
    nbl, nbt, nA, nlo, nla = (case[k] for k in ("blocks_lon", "blocks_lat", "alts", "nlons",
                                                "nlats"))
    NLAT, NLON = nbt * nla, nbl * nlo
    names = ["rho", "temp", "itemp", "etemp", "vel", "vvel", "nds"] + \
        (["ions", "ivel_par"] if case["ions"] else [])
    rows = torch.arange(-2, NLAT + 2, device=DEV)
    turn = (rows < 0) | (rows >= NLAT)
    src = torch.where(rows < 0, -1 - rows, torch.where(rows >= NLAT, 2 * NLAT - 1 - rows, rows))
    for k in names:
        v = g[k]
        v5 = v if v.dim() == 5 else v[:, None]
        own = v5[:, :, 2:-2, 2:-2, 2:-2]
        nc = own.shape[1]
        G = own.reshape(nbt, nbl, nc, nA, nla, nlo).permute(2, 3, 0, 4, 1, 5).reshape(
            nc, nA, NLAT, NLON)
        G = G[:, :, src]
        G = torch.where(turn[None, None, :, None], torch.roll(G, -(NLON // 2), 3), G)
        G = torch.cat([G[..., -2:], G, G[..., :2]], -1)
        new = G.unfold(2, nla + 4, nla).unfold(3, nlo + 4, nlo)  # nc nA nbt nbl NLg NLo
        new = new.permute(2, 3, 0, 1, 4, 5).reshape(nbl * nbt, nc, nA, nla + 4, nlo + 4)
        v5 = v5.clone()
        v5[:, :, 2:-2] = new
        if k in ("vel", "ivel_par"):
            v5[:nbl, :2, :, :2] *= -1.0
            v5[-nbl:, :2, :, -2:] *= -1.0
        g[k] = v5 if v.dim() == 5 else v5[:, 0]
    if "ivel_par" in g and not case["ions"]:
        raise ValueError("ion velocity without ions")
    return g


def _exact_horizontal(case, g, dt):
    """advance_horizontal.f90:58-924 after the exchange."""
    g = _fill_halo(case, dict(g))
    ions, topo, nA = case["ions"], case["topography"], case["alts"]
    nv = 17 + (2 if ions else 0)
    parts = [g["rho"][:, None], g["temp"][:, None], g["vel"], g["nds"], g["vvel"]] + \
        ([g["ions"][:, :2]] if ions else [])
    Q = torch.cat(parts, 1)
    own = slice(2, -2)

    def k_of(a, k):
        return a[:, k]
    lat_i = dict(tan=g["tan_lat"][:, own], cos=g["cos_lat"][:, own],
                 sin=torch.sin(g["latitude"][:, own]))

    def level(ks):
        """RK4 of the levels ks (a slice of the level axis)."""
        def one(a):
            return a[:, ks]
        ifo, ifa = one(g["inv_dlon_fb"])[:, None], one(g["inv_dlat_fb"])[:, None]
        dfo, dfa = one(g["dlon_fb"])[:, None], one(g["dlat_fb"])[:, None]
        gbo = one(g["inv_dlon_gb"])[:, None, :, own, own]
        gba = one(g["inv_dlat_gb"])[:, None, :, own, own]
        kc = slice(ks.start - 1, ks.stop - 1)
        cmo = g["cmax"][:, 0, kc, 1:-1][:, None]
        cma = g["cmax"][:, 1, kc][..., 1:-1][:, None].transpose(-1, -2)
        ir = one(g["invr"])[..., own, own]
        rdist = one(g["raddist"])[..., own, own]
        gam = one(g["gamma"])[..., own, own]
        tl, co, si = (lat_i[n][:, None, :, None] for n in ("tan", "cos", "sin"))
        q0 = Q[:, :, ks]
        if topo:
            dz = (Q[:, :, ks.start + 1:ks.stop + 1] - Q[:, :, ks.start - 1:ks.stop - 1])[
                ..., own, own] * (0.5 / one(g["dalt"])[..., own, own])[:, None]
            dzo = dz * one(g["dalt_dlon"])[..., own, own][:, None]
            dza = dz * one(g["dalt_dlat"])[..., own, own][:, None]
        if ions:
            ive, ivn = one(g["ivel"][:, 0])[..., own, own], one(g["ivel"][:, 1])[..., own, own]

        def line(v, f, dfb, gb, cm):
            """Along the last axis: v on cells -1..n+2, f and dfb on faces."""
            d = v[..., 1:] - v[..., :-1]           # faces 0..n+2
            s4 = f[..., 2:-1] * 2 * (F1 * d[..., 1:-1] - F2 * (v[..., 3:] - v[..., :-3]))
            fd = torch.cat([d[..., :1] * f[..., 1:2], s4, d[..., -1:] * f[..., -1:]], -1)
            sl = _mc(fd[..., 1:], fd[..., :-1])    # cells 0..n+1
            w = v[..., 1:-1]
            l = w[..., :-1] + 0.5 * sl[..., :-1] * dfb[..., 2:-1]
            r = w[..., 1:] - 0.5 * sl[..., 1:] * dfb[..., 2:-1]
            fl = 0.5 * torch.maximum(cm[..., :-1], cm[..., 1:]) * (r - l)
            return (0.5 * (l[..., 1:] + r[..., 1:] - l[..., :-1] - r[..., :-1]) * gb,
                    (fl[..., 1:] - fl[..., :-1]) * gb)

        def rate(q):
            go, do = line(q[..., own, :], ifo[..., own, :], dfo[..., own, :], gbo, cmo)
            qt = q[..., own].transpose(-1, -2)
            ga, da = line(qt, ifa[..., own].transpose(-1, -2), dfa[..., own].transpose(-1, -2),
                          gba.transpose(-1, -2), cma)
            ga, da = ga.transpose(-1, -2), da.transpose(-1, -2)
            if topo:
                go, ga = go - dzo, ga - dza
            c = q[..., own, own]
            rho, t, ve, vn, vu = (c[:, i] for i in range(5))
            div = ga[:, 3] + go[:, 2] - tl * vn * ir
            K = torch.empty_like(c)
            K[:, 0] = -(rho * div + ga[:, 0] * vn + go[:, 0] * ve)
            K[:, 1] = -((gam - 1) * t * div + ga[:, 1] * vn + go[:, 1] * ve)
            K[:, 2] = -(vn * ga[:, 2] + ve * go[:, 2] + ve * (vu - tl * vn) * ir + go[:, 1] +
                        go[:, 0] * t / rho) + 2 * OMEGA * (si * vn - co * vu)
            K[:, 3] = -(vn * ga[:, 3] + ve * go[:, 3] + (vn * vu + tl * ve * ve) * ir + ga[:, 1] +
                        ga[:, 0] * t / rho) - (OMEGA * OMEGA * co * si * rdist +
                                               2 * OMEGA * si * ve)
            K[:, 4] = -(vn * ga[:, 4] + ve * go[:, 4])
            K[:, 5:11] = -(c[:, 5:11] * div[:, None] + ga[:, 5:11] * vn[:, None] +
                           go[:, 5:11] * ve[:, None])
            K[:, 11:17] = -(ga[:, 11:17] * vn[:, None] + go[:, 11:17] * ve[:, None])
            if ions:
                K[:, 17:] = -(ga[:, 17:] * ivn[:, None] + go[:, 17:] * ive[:, None])
            return dt * (K + do + da)
        q, acc = q0.clone(), 0.0
        base = q0[..., own, own].clone()
        for n in range(4):
            k = rate(q)
            acc = acc + (1.0, 2.0, 2.0, 1.0)[n] * k
            q[..., own, own] = base + (0.5 * k if n < 2 else k if n == 2 else acc / 6.0)
        Q[:, :, ks][..., own, own] = q[..., own, own]
    if topo:
        for k in range(2, nA + 2):
            level(slice(k, k + 1))
    else:
        for k in range(2, nA + 2, 10):
            level(slice(k, min(k + 10, nA + 2)))
    out = dict(rho=Q[:, 0], temp=Q[:, 1], vel=Q[:, 2:5], nds=Q[:, 5:11], vvel=Q[:, 11:17],
               itemp=g["itemp"], etemp=g["etemp"])
    if ions:
        i = g["ions"].clone()
        inner = (slice(None), slice(None), slice(2, -2), own, own)
        adv = Q[:, 17:][inner].clamp(min=1.0e2)
        # UseImprovedIonAdvection: the divergence of the field-aligned velocity
        v = g["ivel_par"]
        ir = g["invr"][:, 2:-2, own, own]
        cl = lat_i["cos"][:, None, :, None]
        glo, gla = (g[k][:, :, None] for k in ("grad_lon", "grad_lat"))
        ve, vn, vu = v[:, 0, 2:-2], v[:, 1, 2:-2], v[:, 2]
        east = (glo[:, 0, :, None] * ve[..., own, 1:-3] + glo[:, 1, :, None] * ve[..., own, own] +
                glo[:, 2, :, None] * ve[..., own, 3:-1]) * ir / cl.clamp(min=0.17)
        gl = gla[..., None]
        north = (gl[:, 0] * vn[..., 1:-3, own] + gl[:, 1] * vn[..., own, own] +
                 gl[:, 2] * vn[..., 3:-1, own]) * ir
        rd = g["raddist"][..., own, own]
        dp, dm = rd[:, 3:-1] - rd[:, 2:-2], rd[:, 2:-2] - rd[:, 1:-3]
        q = dm / dp
        vo = vu[..., own, own]
        radial = (q * q * vo[:, 3:-1] - vo[:, 1:-3] - (q * q - 1) * vo[:, 2:-2]) / (dm * (1 + q))
        tl = lat_i["tan"][:, None, :, None].clamp(-5.0, 5.0)
        div = (east + north - tl * vn[..., own, own] * ir + radial + 2 * vo[:, 2:-2] * ir) * cl
        i[:, :2][inner] = adv / (1 + dt * div)[:, None]
        i[:, 9] = i[:, :9].sum(1)
        out["ions"], out["ivel_par"] = i, g["ivel_par"]
    return out


def _exact_window(case, seed):
    c0 = _columns(case["columns"], case["alts"], False, False, seed)
    geo = {k: c0[k] for k in ("alt", "grav", "invr", "dalt", "coslat")}
    heat = _heat(c0)

    def one(state, heat):
        p, _ = _prep_fields(state["nds"], state["temp"], state["rho"], state["vvel"])
        o = _step(dict(state, **geo, **{k: p[k] for k in ("tempunit", "mmm", "gamma", "cmax",
                                                         "eddy")}), DT)
        t = o["temp"].clone()
        t[:, 2:-2] = t[:, 2:-2] + DT * heat[:, 2:-2] / (p["cp"] * p["tempunit"])[:, 2:-2]
        return dict({k: o[k] for k in STATE}, temp=t)
    state = {k: c0[k] for k in STATE}
    kept = []
    with torch.no_grad():
        for _ in range(case["steps"]):
            kept.append(state)
            state = one(state, heat)
    lam = _seeds(case, seed)
    g_heat = torch.zeros_like(heat)
    for s in reversed(kept):
        s = {k: v.detach().clone().requires_grad_(True) for k, v in s.items()}
        h = heat.detach().clone().requires_grad_(True)
        o = one(s, h)
        g = torch.autograd.grad([o[k] for k in STATE], [s[k] for k in STATE] + [h], lam)
        lam = list(g[:5])
        g_heat = g_heat + g[5]
    return dict(state, **{"g_" + k: v for k, v in zip(STATE, lam)}, g_heat=g_heat)


def _prep_exact(c):
    """The prep's outputs as the entry point leaves them (cMax on levels
    0..nAlts+1, zero elsewhere) and the time step (0.75 CFL, at most 2 s)."""
    p, _ = _prep_fields(c["nds"], c["temp"], c["rho"], c["vvel"])
    cm = p["cmax"].clone()
    cm[:, 0] = cm[:, -1] = 0.0
    rate = (cm / c["dalt"])[:, 2:-2].max()
    return dict(p, cmax=cm), torch.minimum(0.75 / rate, torch.tensor(DT, device=DEV, dtype=F64))


def exact(case, seed):
    kind = case["kind"]
    if kind == "horizontal":
        g, dt = _blocks(case, seed)
        return _exact_horizontal(case, g, dt)
    if kind == "window":
        return _exact_window(case, seed)
    if kind == "ensemble":
        outs, dts = [], []
        for c in _members(case, seed):
            p, dt = _prep_exact(c)
            o = _step(dict(c, **{k: p[k] for k in ("gamma", "mmm", "tempunit", "eddy", "cmax")}),
                      dt)
            outs.append({k: o[k] for k in STATE})
            dts.append(dt)
        return [torch.stack(dts)] + outs
    c = _columns(case["columns"], case["alts"], case["stretched"], case.get("ions", False), seed)
    if kind == "prepare":
        p, dt = _prep_exact(c)
        return dict({k: p[k] for k in PREP_OUT}, dt=dt.view(1))
    if kind == "sources":
        return _exact_sources(c, _source_fields(c, seed))
    # large grids in slices of columns, so that the intermediates fit
    n, most = case["columns"], max(1, 1_200_000 // (case["alts"] + 4))
    parts = []
    for i in range(0, n, most):
        sub = {k: v[i:i + most] for k, v in c.items()}
        parts.append(_step(sub, DT, case["solver"], case["ions"]))
    names = STATE + ("logns", "nden") + (("ions",) if case["ions"] else ())
    return {k: torch.cat([p[k] for p in parts]) for k in names}
