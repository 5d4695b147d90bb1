"""Workloads of the flow solver: what a program that uses it has it do.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` builds what the program holds before the call, ``run`` is one pass
through the public entry points, ``work`` the bytes and operations of a pass
and ``exact`` its results in 64 bits where plain numpy gives them in seconds.

The geometry of a case (grid, buildings, terrain) is fixed by its values; the
seed gives the weather on it: wind speed, direction, stability and, where a
case needs them, perturbations, gradients or particle positions.  That is the
use the solver is built for: one city, many weather situations.

The kinds:

* ``plain``: one situation, ``ITER`` SIMPLE iterations (what the solver runs
  between two looks at its residuals), then the fields of the situation;
* ``batch``: several directions of one city in lock step, then each
  situation's flow-field file (the int16 payload GRAL stores per situation);
* ``terrain``: one k-eps situation over hills with vegetation;
* ``situation``: a situation from nothing to its file: set-up on the GPU,
  handle, prologue, 100 iterations with the stop test, epilogue, payload;
* ``diagnostic``: the mass-conservation pass over the full column height that
  follows every prognostic solve;
* ``window``: a window of pressure-correction steps and its VJP;
* ``momentum``: one momentum sweep of each component and its VJP;
* ``particles``: the particle model's wind at many positions.
"""
import ctypes
import dataclasses
import math

import numpy as np

from gral_amd import domain, pf

ITER = 20                 # iterations of a pass
ITER_MAX = 1000000        # never reached: a state can run any number of passes
F32 = np.float32


def listed():
    return [
        # the smallest domain of use: one house, 24 x 27 cells; launches and the serial path count
        {"name": "house_plain", "kind": "plain", "nii": 24, "njj": 27, "layers": 16, "city": 0, "model": 1, "width": 8},
        # one building on flat ground, 100 x 100 cells, 200 m square: the configuration of a first test run
        {"name": "building_plain", "kind": "plain", "nii": 100, "njj": 100, "layers": 30, "city": 0, "model": 1,
         "width": 8},
        # a city block of 400 x 400 cells, one wind direction at a time
        {"name": "city_plain", "kind": "plain", "nii": 400, "njj": 400, "layers": 40, "city": 20260001, "model": 1,
         "width": 8},
        # the same block under its 8 wind directions as one batch: the production run, and the largest case
        {"name": "city_batch", "kind": "batch", "nii": 400, "njj": 400, "layers": 40, "city": 20260001, "model": 1,
         "width": 8, "situations": 8},
        # k-eps closure, four directions of a smaller, odd-sized block
        {"name": "keps_batch", "kind": "batch", "nii": 259, "njj": 243, "layers": 40, "city": 20260001, "model": 2,
         "width": 8, "situations": 4},
        # hills, buildings and vegetation, k-eps, stretched levels
        {"name": "terrain_plain", "kind": "terrain", "n": 301, "layers": 30},
        # towers up to 130 m under 50 layers: columns of more than 128 levels
        {"name": "towers_plain", "kind": "plain", "nii": 181, "njj": 167, "layers": 50, "city": 20260011, "model": 1,
         "width": 8, "hmax": 130.0},
        # a situation from its buildings and weather to its file, as a run over a weather list does it
        {"name": "situation_whole", "kind": "situation", "n": 160, "layers": 40, "city": 20260001},
        # the mass-conservation pass after the prognostic solve, full height (222 levels)
        {"name": "city_diagnostic", "kind": "diagnostic", "nii": 400, "njj": 400, "layers": 40, "city": 20260001,
         "level": 2},
        # sensitivities: 10 pressure-correction steps and their VJP on a 256 x 256 block
        {"name": "window_vjp", "kind": "window", "nii": 256, "njj": 256, "layers": 32, "city": 20264000, "steps": 10},
        # the U, V and W momentum sweeps and their VJPs on the same block
        {"name": "momentum_vjp", "kind": "momentum", "nii": 256, "njj": 256, "layers": 32, "city": 20264000},
        # the particle model's wind for a release of a million particles
        {"name": "particles", "kind": "particles", "nii": 200, "njj": 200, "layers": 40, "city": 20260001,
         "count": 1000000, "topo": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Two sides of a domain: the first over the whole range, the second up to a third longer or shorter."""
    a = _log_int(rng, lo, hi)
    return a, max(lo, min(hi, int(round(a * rng.uniform(0.75, 1.33)))))


def draw(rng):
    """A case of the listed kinds; sizes over their whole range, odd ones among them."""
    kind = rng.choice(["plain", "plain", "plain", "batch", "batch", "terrain", "towers", "situation", "diagnostic",
                       "window", "momentum", "particles"])
    city = rng.randrange(1, 1 << 30)
    if kind == "plain":
        a, b = _sides(rng, 24, 400)
        width = rng.choice([8, 8, 16])
        return {"kind": "plain", "nii": a, "njj": b, "layers": rng.randint(max(16, width), 50), "model": rng.choice([1, 1, 2, 0]),
                "city": 0 if a < 60 else city, "width": width}
    if kind == "batch":
        a, b = _sides(rng, 60, 260)
        return {"kind": "batch", "nii": a, "njj": b, "layers": rng.randint(30, 50), "city": city,
                "model": rng.choice([1, 1, 2]), "width": 8, "situations": rng.randint(2, 8)}
    if kind == "terrain":
        return {"kind": "terrain", "n": _log_int(rng, 100, 300), "layers": rng.randint(20, 32)}
    if kind == "towers":
        a, b = _sides(rng, 80, 180)
        return {"kind": "plain", "nii": a, "njj": b, "layers": rng.randint(44, 56), "city": city,
                "model": rng.choice([1, 1, 2]), "width": 8, "hmax": round(rng.uniform(115.0, 150.0), 1)}
    if kind == "situation":
        return {"kind": "situation", "n": _log_int(rng, 60, 160), "layers": rng.randint(30, 50), "city": city}
    if kind == "diagnostic":
        a, b = _sides(rng, 50, 400)
        return {"kind": "diagnostic", "nii": a, "njj": b, "layers": rng.randint(30, 50), "city": city,
                "level": rng.choice([1, 2])}
    if kind == "window":
        a, b = _sides(rng, 60, 256)
        return {"kind": "window", "nii": a, "njj": b, "layers": rng.randint(16, 40), "city": city,
                "steps": rng.randint(4, 12)}
    if kind == "momentum":
        a, b = _sides(rng, 60, 256)
        return {"kind": "momentum", "nii": a, "njj": b, "layers": rng.randint(16, 40), "city": city}
    a, b = _sides(rng, 60, 200)
    return {"kind": "particles", "nii": a, "njj": b, "layers": rng.randint(30, 50), "city": city,
            "count": _log_int(rng, 1000, 1000000), "topo": rng.choice([0, 1])}


# ---- inputs ----------------------------------------------------------------

def _weather(seed):
    r = np.random.default_rng(seed)
    return r, float(r.uniform(1.0, 6.0)), float(r.uniform(0.0, 360.0))


def _buildings(c):
    """city 0: one 20 x 20 x 15 m building (smaller in a small domain) in the middle; otherwise cuboids at 30 %
    plan area, footprints 8-40 m, heights from 6 m up to hmax."""
    nii, njj = c["nii"], c["njj"]
    if c["city"] == 0:
        w = min(10, min(nii, njj) // 4)
        i0, j0 = (nii - w) // 2 + 1, (njj - w) // 2 + 1
        return [domain.Building(i0, i0 + w - 1, j0, j0 + w - 1, 1.5 * w)]
    return domain.city_buildings(nii, njj, 2.0, c["city"], hmax=c.get("hmax", 40.0))


def _case(c, speed, direction):
    """The situation of a flat case: log profile of the given wind at 10 m over the case's buildings."""
    z0 = 0.2 if c["city"] == 0 else 0.5
    s = domain.build_case(c["kind"], c["nii"], c["njj"], _buildings(c), dx=2.0, vertcellsff=c["layers"], speed10=speed,
                          direction=direction, z0=z0, turbulence_model=c.get("model", 1), iterations=ITER_MAX)
    s.simd_width = c.get("width", 8)
    return s


def _turned(base, speed10, speed, direction):
    """The same buildings under another wind: the profile of base (blowing along +x, speed10) turned and scaled."""
    u, v = domain.wind_components(speed / speed10, direction)
    free = base.uk                                   # profile in the free cells, 0 in the blocked ones and their west faces
    prof = free.max(axis=(0, 1))
    n = base.nii, base.njj
    s = dataclasses.replace(base)
    blocked = np.zeros((n[0] + 2, n[1] + 2, base.nkk + 2), bool)
    blocked[:, :, 1:base.nkk + 1] = np.arange(1, base.nkk + 1)[None, None, :] <= base.kkart[:, :, None]
    blocked[[0, -1], :, :] = False
    blocked[:, [0, -1], :] = False
    s.uk = np.ascontiguousarray(free * F32(u))
    s.vk = np.zeros_like(free)
    s.vk[1:n[0] + 1, 1:n[1] + 1, :] = (prof * F32(v))[None, None, :]
    s.vk[blocked] = 0
    south = blocked[1:n[0] + 1, 1:n[1], :]
    s.vk[1:n[0] + 1, 2:n[1] + 1, :][south] = 0
    s.vk[1:n[0] + 1, n[1] + 1, :] = s.vk[1:n[0] + 1, n[1], :]
    return s


def _terrain(c, speed, direction, stability):
    s = domain.config5(direction=direction, speed=speed, stability=stability, n=c["n"], iterations=ITER_MAX,
                       vertcellsff=c["layers"])
    return s


def _solver(case):
    s = pf.PrognosticFlowfield(case)
    s.prepare()
    return s


def _fields(shape, names):
    """Host arrays the program downloads into, touched once."""
    return {n: np.zeros(shape, F32) + F32(0) for n in names}


FIELDS = ("uk", "vk", "wk", "uks", "vks", "wks", "dpm", "dpmnew", "turb", "tdiss")
FP = ctypes.POINTER(ctypes.c_float)


def _download(s, out):
    """gral_pf_download_fields into the caller's arrays (a field not asked for is NULL)."""
    args = [out[n].ctypes.data_as(FP) if n in out else None for n in FIELDS]
    rc = s.lib.gral_pf_download_fields(s.h, *args)
    if rc != 0:
        raise RuntimeError(s.lib.gral_pf_last_error(s.h).decode())
    return out


def _perturbed(base, r):
    """base's wind with 5 % of seeded noise in its free cells (a field in the middle of a solve)."""
    for a in (base.uk, base.vk):
        a *= (1 + F32(0.05) * r.standard_normal(a.shape, dtype=F32))
    return base


def _city_situations(c, seed):
    r, speed, direction = _weather(seed)
    base = _case(c, 3.0, 270.0)
    return [_turned(base, 3.0, float(r.uniform(1.0, 6.0)), direction + 45.0 * q) for q in range(c["situations"])]


def _particles(c, case, r):
    n = c["count"]
    ci = r.integers(1, case.nii + 1, n).astype(np.int32)
    cj = r.integers(1, case.njj + 1, n).astype(np.int32)
    x = 600000 + (ci - 1 + r.uniform(0, 1, n)) * case.dxk
    y = 5200000 + (cj - 1 + r.uniform(0, 1, n)) * case.dyk
    ahmin = 100.0 if c["topo"] else 0.0
    z = (r.uniform(0.0, float(case.hokart[case.nkk]), n) + ahmin).astype(F32)
    return {"topo": c["topo"], "ahmin": ahmin, "ci": ci, "cj": cj, "ahint": np.zeros(n, F32), "x": x, "y": y, "z": z}


def _particle_inputs(c, seed):
    r, speed, direction = _weather(seed)
    case = _perturbed(_case(c, speed, direction), r)
    case.wk[1:-1, 1:-1, 1:-1] = F32(0.1) * r.standard_normal(case.wk[1:-1, 1:-1, 1:-1].shape, dtype=F32)
    return case, _particles(c, case, r)


def prepare(case, seed):
    c, kind = case, case["kind"]
    r, speed, direction = _weather(seed)
    if kind == "plain":
        s = _solver(_case(c, speed, direction))
        names = FIELDS if c["nii"] * c["njj"] <= 20000 else ("uk", "vk", "wk", "dpmnew")
        names = tuple(n for n in names if c["model"] != 1 or n not in ("turb", "tdiss"))
        return {"kind": kind, "s": s, "out": _fields(s.case.uk.shape, names)}
    if kind == "terrain":
        s = _solver(_terrain(c, speed, direction, 1 + seed % 7))
        return {"kind": kind, "s": s, "out": _fields(s.case.uk.shape, ("uk", "vk", "wk", "dpmnew", "turb", "tdiss"))}
    if kind == "batch":
        ss = [_solver(x) for x in _city_situations(c, seed)]
        kinds = (2, 3) if c["model"] == 2 else (2,)
        return {"kind": kind, "batch": pf.Batch(ss), "files": [(s, k, np.zeros(s.gff_size(k), np.uint8)) for s in ss for k in kinds]}
    if kind == "situation":
        cut = np.zeros((c["n"] + 2, c["n"] + 2), F32)
        for b in domain.city_buildings(c["n"], c["n"], 2.0, c["city"]):
            sl = (slice(b.i0, b.i1 + 1), slice(b.j0, b.j1 + 1))
            cut[sl] = np.maximum(cut[sl], F32(b.height))
        return {"kind": kind, "cut": cut, "c": dict(c), "met": (speed, direction, 1 + seed % 7)}
    if kind == "diagnostic":
        s = _solver(_perturbed(_case(c, speed, direction), r))
        return {"kind": kind, "s": s, "level": c["level"], "out": _fields(s.case.uk.shape, ("uk", "vk", "wk", "dpm"))}
    if kind in ("window", "momentum"):
        s = _solver(_case(c, speed, direction))
        s.iterate(3)                                 # sensitivities are taken at a developed state
        shape = s.case.uk.shape
        d = [r.standard_normal(shape, dtype=F32) for _ in range(3)]
        return {"kind": kind, "s": s, "d": d, "steps": c.get("steps"), "out": _fields(shape, ("uk", "vk", "wk"))}
    fc, p = _particle_inputs(c, seed)
    return {"kind": "particles", "s": _solver(fc), "p": p}


def run(state):
    kind = state["kind"]
    if kind in ("plain", "terrain"):
        st = state["s"].iterate(ITER)
        return [_download(state["s"], state["out"]), st["iterations_run"]]
    if kind == "batch":
        state["batch"].iterate(ITER)
        for s, k, buf in state["files"]:
            s.gff_payload_into(k, buf)
        return [buf[32:].view(np.int16) for _, _, buf in state["files"]]
    if kind == "situation":
        c, (speed, direction, stab) = state["c"], state["met"]
        s = pf.PrognosticFlowfield(domain.flat_case("situation", c["n"], c["n"], state["cut"], vertcellsff=c["layers"],
                                                    speed=speed, direction=direction, stability=stab, iterations=100))
        with s:
            st = s.solve()
            f = np.zeros(s.gff_size(2), np.uint8)
            s.gff_payload_into(2, f, direction, speed, stab)
        return {"file": f[32:].view(np.int16), "delta": st["delta_finish"], "mass_div": st["mass_div"], "mass_flux": st["mass_flux"]}
    if kind == "diagnostic":
        state["s"].diagnostic(state["level"])
        return _download(state["s"], state["out"])
    if kind == "window":
        s = state["s"]
        s.forward_ckpt(state["steps"])
        g = s.vjp(*state["d"])
        out = _download(s, state["out"])             # the window's result
        s.restore_ckpt()
        return [out, list(g)]
    if kind == "momentum":
        s, g = state["s"], []
        for comp in range(3):
            s.momentum_sweep(comp)
            g.append(s.momentum_vjp(state["d"][comp]))
        return [_download(s, state["out"]), g]
    p = state["p"]
    ux, uy, uz, k = state["s"].wind_at_particles(p["topo"], 600000, 5200000, p["ahmin"], p["ci"], p["cj"], p["ahint"],
                                                 p["x"], p["y"], p["z"])
    return {"ux": ux, "uy": uy, "uz": uz, "k": k}


# ---- the least a pass can do -----------------------------------------------

def work(case):
    """Bytes and operations of a pass.  A SIMPLE iteration is a fixed sequence of passes over the fields, each in its
    own sweep order, so no array can be kept from one to the next: divergence reads 3 and writes 2 of them, the
    pressure sweep reads 3 and writes 2, the correction 4 and 3, the averages 3 and 3, each momentum sweep 7 and 1,
    and the k-eps sweep 5 and 2 (4 bytes a cell and array).  Operations: about 2.9 per byte."""
    c, kind = case, case["kind"]
    if kind == "situation":
        cells = _case({**c, "nii": c["n"], "njj": c["n"]}, 3.0, 270.0).active_cells()
        b = 188.0 * 100 * cells
        return {"bytes": b, "flops": 2.9 * b}
    if kind == "terrain":                            # all columns lie in the sub-domains: 30 layers under the top
        b = 212.0 * ITER * c["n"] * c["n"] * c["layers"]
        return {"bytes": b, "flops": 2.9 * b}
    base = _case(c, 3.0, 270.0)
    cells, full = base.active_cells(), base.nii * base.njj * base.nkk
    if kind in ("plain", "batch"):
        b = {0: 188.0, 1: 188.0, 2: 212.0}[c["model"]] * ITER * cells * c.get("situations", 1)
    elif kind == "diagnostic":                       # divergence 3 + 1, pressure 2 + 1, correction 4 + 3, per iteration
        b = 56.0 * full * (10 if c["level"] == 2 else 5)
    elif kind == "window":                           # 17 arrays a step forward, the same transposed
        b = 2 * 68.0 * cells * c["steps"]
    elif kind == "momentum":                         # three sweeps; the VJP reads the same 7 arrays and 2 more
        b = 3 * (32.0 + 44.0) * cells
    else:
        return {"bytes": 72.0 * c["count"], "flops": 20.0 * c["count"]}
    return {"bytes": b, "flops": 2.9 * b}


# ---- 64 bits ---------------------------------------------------------------

def exact(case, seed):
    """The particle wind in 64 bits.  The solves have no value here: sweeps whose columns depend on one another, level
    by level, take plain numpy far more than 20 s for 20 iterations, and the files hold whole numbers."""
    if case["kind"] != "particles":
        return None
    fc, p = _particle_inputs(case, seed)
    u, v, w = (a.astype(np.float64) for a in (fc.uk, fc.vk, fc.wk))
    nii, njj, nkk = fc.nii, fc.njj, fc.nkk
    # what the solver's set-up does to the field: east and north ghost faces, no wind inside the buildings
    u[nii + 1, 1:njj + 1, 1:nkk] = u[nii, 1:njj + 1, 1:nkk]
    v[1:nii + 1, njj + 1, 1:nkk] = v[1:nii + 1, njj, 1:nkk]
    kk = fc.kkart.astype(int)
    top = np.minimum(kk, np.minimum(nkk - 1, kk + fc.vertcellsff))
    lev = np.arange(nkk + 2)
    inside = (fc.advdom[:, :, None] == 1) & (lev >= 1) & (lev <= top[:, :, None])
    inside[[0, -1]] = False
    inside[:, [0, -1]] = False
    for a in (u, v, w):
        a[inside] = 0
    hok, dzk = fc.hokart.astype(np.float64), fc.dzk.astype(np.float64)
    i, j = p["ci"], p["cj"]
    h = p["z"].astype(np.float64) - p["ahmin"]
    k = np.clip(np.searchsorted(hok[:nkk + 1], h), 1, nkk)
    ux = u[i, j, k] + (u[i + 1, j, k] - u[i, j, k]) / fc.dxk * (p["x"] - (600000 + (i - 1) * fc.dxk))
    uy = v[i, j, k] + (v[i, j + 1, k] - v[i, j, k]) / fc.dyk * (p["y"] - (5200000 + (j - 1) * fc.dyk))
    uz = w[i, j, k] + (w[i, j, k + 1] - w[i, j, k]) / dzk[k] * (h - hok[k - 1])
    return {"ux": ux, "uy": uy, "uz": uz, "k": None}
