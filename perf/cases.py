"""The work that users of this package have it do, as timed cases.

Four kinds, each through the public entry points:

  sweep     one directional sweep on device buffers (hp_ppmsolver_noalloc)
  evolve    a box's state goes in, some steps run on the device, the new state
            comes out; static or comoving, with or without gravity and
            particles (hp_upload_device, Box.speed / evolve / evolve_cosmo,
            hp_download_device)
  ensemble  independent boxes from host arrays advanced together (Batch)
  serve     a burst of seeded shock-tube requests through the request loop

listed() names the cases, draw() makes further ones of the same ranges,
prepare() builds inputs and handles from a seed, run() is one pass, work()
the bytes and operations a pass cannot do without, and exact() the same
outputs computed in 64 bits with torch alone.
"""
import ctypes
import math

import numpy as np
import torch

import hydropad_amd as hp
from hydropad_amd import batch, ic

FIELDS = ("p", "rho", "vx", "vy", "vz")
NB = 3
PRECISION = {"fp64": 0, "mixed": 1, "fp64_exact": 2}
COUR = 0.8
A_START = 1.0 / 51.0
GAMMA = 5.0 / 3.0
GAMMA_NAMELIST = 1.66666667          # the reference namelist's value, not 5/3
SIZES = (32, 48, 64, 96, 128, 192)   # the ensemble workload's box sizes
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _case(name, kind, nx, ny, nz, precision="fp64", flow="tube", gamma=GAMMA, axis=0, steps=1, **more):
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "precision": precision, "flow": flow, "gamma": gamma,
         "axis": axis, "steps": steps, "cosmo": False, "gravity": False, "particles": 0, "boxes": 0, "direction": 0}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one x sweep of the smallest ensemble box
        _case("sweep_x_32", "sweep", 32, 32, 32, direction=1),
        # the reference-order form, whose results a port is checked against, on a ragged turbulent box
        _case("sweep_y_exact_odd", "sweep", 117, 83, 61, "fp64_exact", "field", direction=2),
        # a mixed z sweep with gravity, ragged, on the cell-to-cell noise of the tests
        _case("sweep_z_mixed_gravity", "sweep", 150, 97, 131, "mixed", "noise", direction=3, gravity=True),
        # the 64^3 shock tube, 100 steps
        _case("tube_64_100steps", "evolve", 64, 64, 64, steps=100),
        # the 512^3 shock tube of the benchmark
        _case("tube_512", "evolve", 512, 512, 512, steps=3),
        # one GPU's share of that tube over eight (512 x 512 x 64), mixed
        _case("tube_slab_mixed", "evolve", 512, 512, 64, "mixed", steps=12),
        # the comoving 256^3 box
        _case("cosmo_256", "evolve", 256, 256, 256, flow="field", steps=4, cosmo=True),
        # a comoving box of ragged sides in the mixed form
        _case("cosmo_mixed_odd", "evolve", 93, 110, 101, "mixed", "field", steps=12, cosmo=True),
        # a turbulent box with the reference namelist's gamma
        _case("namelist_gamma_128", "evolve", 128, 128, 128, flow="field", gamma=GAMMA_NAMELIST, steps=8),
        # hydro with a static potential and particles, host particles in and out
        _case("nbody_96", "evolve", 96, 96, 96, flow="field", steps=10, gravity=True, particles=200000),
        # an ensemble of comoving boxes, host arrays in and out
        _case("ensemble_8", "ensemble", 32, 64, 0, flow="field", steps=40, cosmo=True, boxes=8),
        # a burst of requests, final states returned
        _case("serve_10", "serve", 32, 96, 0, steps=40, boxes=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("sweep", "sweep", "evolve", "evolve", "evolve", "ensemble", "serve"))
    prec = rng.choice(("fp64", "fp64", "mixed"))
    if kind in ("ensemble", "serve"):
        lo = rng.choice(SIZES[:3])
        hi = min(96, lo + rng.randrange(17, 49))
        return _case("", kind, lo, hi, 0, prec, "field" if kind == "ensemble" else "tube", steps=rng.randrange(15, 41),
                     boxes=rng.choice((4, 5, 6, 8, 9, 10)), cosmo=kind == "ensemble" and rng.random() < 0.7)
    if kind == "sweep" and rng.random() < 0.2:
        prec = "fp64_exact"
    n = _log_int(rng, 24, 96 if prec == "fp64_exact" else 320 if kind == "sweep" else 256)
    nx, ny, nz = (max(16, int(n * rng.uniform(0.6, 1.4)) + rng.randrange(0, 2)) for _ in range(3))
    flow = rng.choice(("tube", "field", "field", "noise") if kind == "sweep" else ("tube", "field"))
    gamma = rng.choice((GAMMA, GAMMA, GAMMA, GAMMA_NAMELIST, 1.4))
    if kind == "sweep":
        return _case("", kind, nx, ny, nz, prec, flow, gamma, rng.randrange(3),
                     direction=rng.randrange(1, 4), gravity=rng.random() < 0.25)
    cosmo = rng.random() < 0.4
    steps = max(2, min(60, int(4e7 / (nx * ny * nz))))
    return _case("", kind, nx, ny, nz, prec, "field" if cosmo else flow, GAMMA if cosmo else gamma, rng.randrange(3),
                 steps, cosmo=cosmo, gravity=not cosmo and rng.random() < 0.25)


# ---- inputs -------------------------------------------------------------------
# Tensors are (nz, ny, nx) contiguous: the memory of the Fortran (nx, ny, nz)
# arrays.  The interior is made first, then padded with its periodic images.

def _pad(a):
    for d in range(3):
        n = a.shape[d]
        a = torch.cat((a.narrow(d, n - NB, NB), a, a.narrow(d, 0, NB)), d)
    return a.contiguous()


def _tube(shape, axis, gamma, seed):
    """A developed periodic shock tube along axis 0..2 (x, y, z): the exact
    solutions of its two discontinuities, at the split and at the wrap, with
    ripples of a per cent or two where the gas moves (a computed tube's
    plateaus are not constant to the last bit) and undisturbed gas at rest."""
    r = np.random.default_rng(seed)
    left = (1.0 + 0.2 * (r.random() - 0.5), 1.0 + 0.2 * (r.random() - 0.5))
    right = (0.125 + 0.02 * r.random(), 0.1 + 0.02 * r.random())
    x0, t = 0.45 + 0.1 * r.random(), 0.04 + 0.05 * r.random()
    n = shape[axis]
    x = (np.arange(n) + 0.5) / n
    rho, u, p = ic.sod_exact(x, t, gamma, left, right, x0)
    for s, near in ((x, x < 0.5 * x0), (x - 1.0, x > 0.5 * (1.0 + x0))):
        mr, mu, mp = ic.sod_exact(-s, t, gamma, left, right, 0.0)    # the mirrored tube at the wrap
        rho, u, p = np.where(near, mr, rho), np.where(near, -mu, u), np.where(near, mp, p)
    moves, ph = u != 0.0, 2.0 * math.pi * (r.random(3)[:, None] + np.array([[3.0], [5.0], [4.0]]) * x)
    p, rho, u = (a * (1.0 + moves * e * np.sin(s)) for a, e, s in zip((p, rho, u), (0.01, 0.02, 0.015), ph))
    prof = {"p": p, "rho": rho, ("vx", "vy", "vz")[axis]: u}
    view = [1, 1, 1]
    view[2 - axis] = n
    full = tuple(reversed(shape))
    out = {k: torch.zeros(full, dtype=torch.float64, device=DEV) for k in FIELDS}
    for k, v in prof.items():
        out[k] = torch.from_numpy(np.array(v)).to(DEV).reshape(view).expand(full).contiguous()
    return out


def _field(shape, gamma, seed, cosmo):
    """A Gaussian random density field with growing-mode velocities at uniform
    temperature: P(k) ~ k^-2, Mach 50 and the Zel'dovich amplitude for a
    comoving box; the turbulent k^-11/3, Mach 0.8 and unit sound speed for a
    static one."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    full = tuple(reversed(shape))
    big = max(shape)
    white = torch.fft.rfftn(torch.randn(full, generator=g, dtype=torch.float64, device=DEV))
    kz, ky = (2.0 * math.pi * big * torch.fft.fftfreq(n, device=DEV, dtype=torch.float64) for n in full[:2])
    kx = 2.0 * math.pi * big * torch.fft.rfftfreq(full[2], device=DEV, dtype=torch.float64)
    k = (kx[None, None, :], ky[None, :, None], kz[:, None, None])
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    k2[0, 0, 0] = 1.0
    white = white * k2 ** (-0.5 if cosmo else -11.0 / 12.0)
    white[0, 0, 0] = 0.0
    delta = torch.fft.irfftn(white, s=full)
    rms = 0.05 if cosmo else 0.15
    white = white * (rms / delta.std())
    rho = (1.0 + delta * (rms / delta.std())).clamp_min(0.2)
    vel = [torch.fft.irfftn(1j * q * white / k2, s=full) for q in k]
    vrms = torch.sqrt(sum((v * v).mean() for v in vel) / 3.0)
    if cosmo:
        vel = [ic.eds_adot(A_START) * v for v in vel]
        cs = ic.eds_adot(A_START) * vrms / 50.0
    else:
        vel = [(0.8 / vrms) * v for v in vel]
        cs = 1.0
    return dict(zip(FIELDS, (rho * (cs * cs / gamma), rho, *vel)))


def _noise(shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    full = tuple(reversed(shape))
    a = [torch.rand(full, generator=g, dtype=torch.float64, device=DEV) for _ in FIELDS]
    return dict(zip(FIELDS, (1.0 + 0.3 * a[0], 1.0 + 0.3 * a[1], *(0.3 * (v - 0.5) for v in a[2:]))))


def _interior(case, seed, shape=None):
    shape = shape or (case["nx"], case["ny"], case["nz"])
    if case["flow"] == "tube":
        return _tube(shape, case["axis"], case["gamma"], seed)
    if case["flow"] == "noise":
        return _noise(shape, seed)
    return _field(shape, case["gamma"], seed, case["cosmo"])


def _gforce(case):
    """(3, nx, ny, nz) Fortran-ordered host array of the static Gaussian potential."""
    return ic.gaussian_gforce(tuple(case[k] + 2 * NB for k in ("nx", "ny", "nz"))) if case["gravity"] else None


def _boxes(case):
    """Sides of the boxes of an ensemble or of the requests of a burst: from nx to ny, in no order."""
    n = case["boxes"]
    return [case["nx"] + (case["ny"] - case["nx"]) * (7 * i % n) // max(1, n - 1) for i in range(n)]


def _requests(case, seed):
    r = np.random.default_rng(seed + 78)
    return [{"n": n, "nsteps": int(case["steps"] + r.integers(-5, 6)), "seed": int(r.integers(1 << 30)),
             "precision": case["precision"], "arrival_s": 0.0} for n in _boxes(case)]


def _schedule():
    ca, tstop = ic.eds_schedule(A_START, 1.0 / 11.0, 200)
    return hp.cosmo_init(A_START, COUR, ca, tstop)


def _vmax(f, gamma):
    speed = torch.maximum(torch.maximum(f["vx"].abs(), f["vy"].abs()), f["vz"].abs())
    return float((speed + torch.sqrt(gamma * f["p"] / f["rho"])).max())


# ---- one pass -------------------------------------------------------------------

def prepare(case, seed):
    s = {"case": case}
    if case["kind"] == "serve":
        s["requests"] = _requests(case, seed)
        return s
    if case["kind"] == "ensemble":
        s["states"] = []
        for i, n in enumerate(_boxes(case)):
            f = _interior(case, seed * 64 + i, (n, n, n))
            s["states"].append({k: _pad(v).cpu().numpy().T for k, v in f.items()})
        return s
    shape = tuple(case[k] + 2 * NB for k in ("nx", "ny", "nz"))
    inner = _interior(case, seed)
    s["in"] = [_pad(inner[k]) for k in FIELDS]
    s["out"] = [torch.zeros_like(a) for a in s["in"]]
    g = _gforce(case)
    if case["kind"] == "sweep":
        s["gforce"] = torch.from_numpy(g.T.copy()).to(DEV) if g is not None else None   # (nz, ny, nx, 3)
        s["params"] = hp.params_init(case["gamma"], max(shape) - 2 * NB)
        hp.timedet(s["params"], _vmax(inner, case["gamma"]), COUR)
        return s
    box = s["box"] = hp.Box(shape, case["precision"], case["gamma"])
    if g is not None:
        box.upload_gforce(g)
        s["gforce"] = torch.from_numpy(g.T.copy()).to(DEV)
    if case["cosmo"]:
        s["schedule"] = _schedule()
    if case["particles"]:
        s["particles"] = ic.particles(shape, case["particles"], seed)
    return s


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def run(s):
    case = s["case"]
    if case["kind"] == "serve":
        results, _, fields = batch.serve(s["requests"], hbm_budget=64 << 30, max_boxes=64,
                                         keep_fields=range(len(s["requests"])))
        return {"t": np.array([r["t"] for r in results]), "steps": np.array([r["steps"] for r in results]),
                "state": [[fields[i][k] for k in FIELDS] for i in range(len(results))]}
    if case["kind"] == "ensemble":
        with batch.Batch(max_boxes=case["boxes"], hbm_budget=64 << 30) as b:
            ids = [b.add(f, nsteps=case["steps"], precision=case["precision"], gamma=case["gamma"], cour=COUR,
                         cosmo=_schedule() if case["cosmo"] else None) for f in s["states"]]
            b.use_graph(True)
            b.step(case["steps"])
            out = [b.download(i) for i in ids]
        return [[f[k] for k in FIELDS] for f in out]
    if case["kind"] == "sweep":
        L = hp.hydro._capi.lib()
        stream = torch.cuda.current_stream().cuda_stream
        hp.hydro.check("hp_ppmsolver_noalloc", L.hp_ppmsolver_noalloc(
            ctypes.byref(s["params"]), *map(_p, s["in"]), *map(_p, s["out"]), _p(s["gforce"]),
            *(case[k] + 2 * NB for k in ("nx", "ny", "nz")), NB, case["direction"], PRECISION[case["precision"]], 0,
            None, ctypes.c_void_p(stream)))
        return s["out"]
    box = s["box"]
    hp.hydro.check("hp_upload_device", box.L.hp_upload_device(box._h, *map(_p, s["in"]), _p(s.get("gforce"))))
    if case["particles"]:
        box.particles_upload(*s["particles"], 0.01)
    if case["cosmo"]:
        sched = box.evolve_cosmo(1, case["steps"], s["schedule"].copy())
        times = [sched.t, sched.dt, sched.at]
    else:
        dt, t = box.timedet(box.speed(), COUR)
        times = list(box.evolve(1, case["steps"], COUR, t, dt))
    hp.hydro.check("hp_download_device", box.L.hp_download_device(box._h, *map(_p, s["out"])))
    return {"state": s["out"], "times": times, "particles": box.particles_download() if case["particles"] else ()}


def work(case):
    """Per cell and sweep: five doubles read and five written, and about 600
    operations (parabolas, two traced faces, one Riemann problem, update)."""
    if case["kind"] in ("ensemble", "serve"):
        mean = 0.5 * (case["nx"] + case["ny"])
        updates = case["boxes"] * mean ** 3 * case["steps"] * 3
    else:
        updates = case["nx"] * case["ny"] * case["nz"] * case["steps"] * (1 if case["kind"] == "sweep" else 3)
    byts = updates * (80.0 + (8.0 if case["gravity"] else 0.0))
    return {"bytes": byts + case["particles"] * case["steps"] * 96.0, "flops": updates * 600.0}


# ---- the same outputs from torch in 64 bits ----------------------------------------
# The reference's algorithm on interior arrays (nz, ny, nx); a sweep pads
# three periodic cells along its axis.  FP32 literals as the reference has them.
_F = np.float32
_SIXTH, _THIRD, _C01, _C05, _TINY, _TERR = (float(_F(v)) for v in (0.16666667, 0.33333333, 0.01, 0.05, 1e-15, 1e-3))
_K23, _KM13 = float(_F(2.0) / _F(3.0)), float(_F(-1.0) / _F(3.0))


def _scalars(gamma, ngrid):
    dx = float(_F(1.0) / _F(ngrid))
    return {"g": gamma, "m": (gamma - 1.0) / (2.0 * gamma), "gf": (gamma + 1.0) / (2.0 * gamma),
            "g1": (gamma + 1.0) / (gamma - 1.0), "dx": dx, "dt": 0.0, "dtat": 0.0, "at": 1.0, "dat": 0.0}


def _slope(a, b, c):
    dl, dr, da = b - a, c - b, 0.5 * (c - a)
    mn = torch.minimum(da.abs(), 2.0 * torch.minimum(dl.abs(), dr.abs()))
    return torch.where(dl * dr > 0, torch.copysign(mn, da), torch.zeros_like(da))


def _limit(a, l, r, flat):
    d, a6 = r - l, 6.0 * (a - 0.5 * (l + r))
    level = (r - a) * (a - l) <= 0
    over, under = ~level & (d * a6 > d * d), ~level & (d * a6 < -d * d)
    l, r = torch.where(over, 3 * a - 2 * r, torch.where(level, a, l)), torch.where(under, 3 * a - 2 * l, torch.where(level, a, r))
    l, r = flat * a + (1 - flat) * l, flat * a + (1 - flat) * r
    return l, r, r - l, 6.0 * (a - 0.5 * (l + r))


def _trace(q, a, cs, S, right):
    """Traced state of the cells' right (or left) faces."""
    rat = 1.0 / S["at"]
    u = a[2]
    sg = 1.0 if right else -1.0

    def avg(v, x):
        l, r, d, a6 = q[v]
        w = (1.0 - 2.0 * x * _THIRD) * a6
        return r - 0.5 * x * (d - w) if right else l + 0.5 * x * (d + w)

    x = [sg * S["dt"] * s * rat / S["dx"] for s in (u - cs, u, u + cs)]
    xt = x[2 if right else 0].clamp_min(0.0)
    pt, rt, ut, vt, wt = (avg(v, xt) for v in range(5))
    pt, rt = torch.where(pt < 0, _TINY, pt), torch.where(rt < 0, _TINY, rt)
    ct = torch.sqrt(S["g"] * pt * rt)

    def beta(k, sign):
        pc, uc = avg(0, x[k]), avg(2, x[k])
        gc = avg(5, x[k]) if len(q) > 5 else 0.0
        s = (ut - uc) + sign * (pt - pc) / ct + sign * S["dt"] * (2.0 * S["dat"] * pc / (ct * S["at"]))
        s = s + S["dt"] * (-gc + S["dat"] * uc) * rat
        return torch.where(sg * (u + sign * cs) > 0, -sign * s / (2.0 * ct), 0.0)

    bm, bp = beta(0, -1.0), beta(2, 1.0)
    mid = sg * u > 0
    pc = avg(0, x[1])
    b0 = (pt - pc) / (ct * ct) + 1.0 / rt - 1.0 / avg(1, x[1]) + 2.0 * S["dat"] * pc / (S["at"] * ct * ct) * S["dt"]
    b0 = torch.where(mid, b0, 0.0)
    fp, fr = pt + ct * ct * (bp + bm), 1.0 / (1.0 / rt - bm - b0 - bp)
    return (torch.where(fp <= 0, pt, fp), torch.where(fr <= 0, rt, fr), ut + ct * (bp - bm),
            torch.where(mid, avg(3, x[1]), vt), torch.where(mid, avg(4, x[1]), wt))


def _newton(L, R, S, p):
    """van Leer's iteration from p to the reference's tolerance."""
    cl, cr = torch.sqrt(S["g"] * L[0] * L[1]), torch.sqrt(S["g"] * R[0] * R[1])
    done, v = torch.zeros_like(p, dtype=torch.bool), torch.zeros_like(p)

    def side(p, ps, c):
        x = p / ps
        xm = x ** S["m"]
        a = torch.where((x >= 1) | (xm == 1), c * torch.sqrt(S["gf"] * x + S["m"]), S["m"] * c * (1 - x) / (1 - xm))
        return a, torch.where(x >= 1, (a * a + c * c) / (2 * a ** 3), x ** -S["gf"] / c)

    for _ in range(100):
        a, da = side(p, L[0], cl)
        b, db = side(p, R[0], cr)
        new = p + ((L[2] - (p - L[0]) / a) - (R[2] + (p - R[0]) / b)) / (da + db)
        new = torch.where(new <= 0, p / 1000.0, new)
        v = torch.where(done, v, (L[0] - R[0] + a * L[2] + b * R[2]) / (a + b))
        new = torch.where(done, p, new)
        done = done | ((p - new).abs() / p <= _TERR)
        p = new
        if bool(done.all()):
            break
    return p, v


def _riemann(L, R, S):
    g, m = S["g"], S["m"]
    (pl, rl, ul), (pr, rr, ur) = L[:3], R[:3]
    cl, cr = torch.sqrt(g * pl / rl), torch.sqrt(g * pr / rr)
    low = pl <= pr
    p1, p2, r1 = torch.minimum(pl, pr), torch.maximum(pl, pr), torch.where(low, rl, rr)
    c2, dv = torch.where(low, cr, cl), ul - ur
    two = dv >= (p2 - p1) / torch.sqrt(0.5 * r1 * ((g - 1) * p1 + (g + 1) * p2))
    one = ~two & (dv >= -(2 * c2 / (g - 1)) * (1 - (p1 / p2) ** m))
    rare = ~two & ~one & (dv > -2 * (cl + cr) / (g - 1))
    guess = 0.5 * (pl + pr) + 0.5 * torch.sqrt(g * (pl + pr) * (rl + rr) * 0.25) * (ul + ur)
    other = torch.where(two, p2, ((cl + cr + dv * (g - 1) * 0.5) / (cl / pl ** m + cr / pr ** m)).clamp_min(0) ** (1 / m))
    zeta = (cr / cl) * (pl / pr) ** m
    vl, vr = ul + 2 * cl / (g - 1), ur - 2 * cr / (g - 1)
    newt = (two | one).nonzero(as_tuple=True)
    pm = pl * ((g - 1) * (vl - vr) / (2 * cl * (1 + zeta))).clamp_min(0) ** (1 / m)
    um = (vl * zeta + vr) / (1 + zeta)
    if newt[0].numel():
        pm[newt], um[newt] = _newton([a[newt] for a in L], [a[newt] for a in R], S,
                                     torch.where(guess > 0, guess, other)[newt])
    vac = ~(two | one | rare)
    pm, um = torch.where(vac, 0.0, pm), torch.where(vac, 0.0, um)

    # each side's star density and outermost and innermost wave speeds, seen from the left (sign -1) or right
    def side(p, r, u, c, sign, shock):
        x = pm / p
        rs = r * (S["g1"] * x + 1) / (S["g1"] + x)
        vs = torch.where(rs == r, 0.0, (rs * um - r * u) / torch.where(rs == r, 1.0, rs - r))
        rc = torch.where(vac, 0.0, r * x.clamp_min(0) ** (1 / g))
        tail = torch.where(vac, u - 2 * c / (g - 1), um + sign * torch.sqrt(g * pm / torch.where(rc > 0, rc, 1.0)))
        return torch.where(shock, rs, rc), torch.where(shock, vs, u + sign * c), torch.where(shock, vs, tail)

    lshock, rshock = two | (one & (pl < pr)), two | (one & (pl >= pr))
    rml, hl, tl = side(pl, rl, ul, cl, -1.0, lshock)
    rmr, hr, tr = side(pr, rr, ur, cr, 1.0, rshock)
    right_out = torch.where(rshock, hr < 0, hr <= 0)
    left_out = torch.where(lshock, (hl > 0) & ~(two & (um <= 0)), hl >= 0)
    fan_r, fan_l = ~rshock & (tr <= 0) & (hr > 0), ~lshock & (tl > 0) & (hl <= 0)
    wr, wl = tr / torch.where(tr == hr, 1.0, tr - hr), tl / torch.where(tl == hl, 1.0, tl - hl)
    star = torch.where(um <= 0, rmr, rml)
    out = []
    for mid, a, b, ma, mb in ((pm, pl, pr, pm, pm), (star, rl, rr, rml, rmr), (um, ul, ur, um, um)):
        v = torch.where(fan_l, ma + wl * (a - ma), mid)
        v = torch.where(fan_r, mb + wr * (b - mb), v)
        v = torch.where(left_out, a, v)
        out.append(torch.where(right_out & ~(lshock & ~rshock & left_out), b, v))
    dadt = 1.0 - 0.5 * S["dat"] * S["dt"] / S["at"]
    up = out[2] >= 0
    return out + [dadt * torch.where(up, L[k], R[k]) for k in (3, 4)]


def _update(a, F1, F2, S, g):
    p, r, u, v, w = a[:5]
    lam, ga = S["dtat"] / S["dx"], S["g"]
    m1, m2 = F1[1] * F1[2], F2[1] * F2[2]
    rn = r + lam * (m1 - m2)
    un = (u * r + lam * ((m1 * F1[2] + F1[0]) - (m2 * F2[2] + F2[0])) + S["dtat"] * (r + rn) * g * 0.5) / rn
    vn, wn = ((r * b + lam * (f1 * m1 - f2 * m2)) / rn for b, f1, f2 in ((v, F1[3], F2[3]), (w, F1[4], F2[4])))
    e1, e2 = ((ga * F[0] / (ga - 1) + 0.5 * F[1] * (F[2] ** 2 + F[3] ** 2 + F[4] ** 2)) * F[2] for F in (F1, F2))
    ei = p / (ga - 1)
    en = ei + 0.5 * r * (u * u + v * v + w * w) + lam * (e1 - e2) + S["dtat"] * (r * u + rn * un) * g * 0.5
    ein = ei + lam * 0.5 * (F1[0] + F2[0]) * (F1[2] - F2[2]) + lam * (F1[0] * F1[2] - F2[0] * F2[2]) / (ga - 1)
    ein = torch.where(ein < 0, ei, ein)
    ex = en - 0.5 * rn * (un * un + vn * vn + wn * wn)
    ein = torch.where(ex / en >= 0.1, ex, ein)
    pn = (ga - 1) * torch.where(ex / en >= 1e-3, ex, ein)
    return torch.where(ein <= 0, p, pn), torch.where(rn <= 0, r, rn), un, vn, wn


def _pencils(a, S):
    """One sweep of pencils along the last axis; a: (p, rho, u, v, w[, g])."""
    n = a[0].shape[-1]
    wrap = torch.arange(-NB, n + NB, device=a[0].device) % n
    a = [v[..., wrap] for v in a]

    def at(v, k, width):                 # cells k .. k+width-1
        return v[..., k:k + width]

    sl = [_slope(v[..., :-2], v[..., 1:-1], v[..., 2:]) for v in a]                       # cells 1 ..
    iv = [at(v, 1, n + 3) + 0.5 * (at(v, 2, n + 3) - at(v, 1, n + 3)) + (at(d, 0, n + 3) - at(d, 1, n + 3)) * _SIXTH
          for v, d in zip(a, sl)]                                                          # left of cells 2 ..
    steep = None
    for v in a[:5]:
        x, y = v[..., :-1], v[..., 1:]
        lo = torch.minimum(x, y)
        s = (x * y != 0) & ((y - x).abs() >= 0.25 * lo.abs())
        steep = s if steep is None else steep | s
    w = n + 2                                                                              # cells 2 .. n+3
    flat = 0.15 * (at(steep, 0, w) | at(steep, 1, w) | at(steep, 2, w) | at(steep, 3, w)).double()
    q = []
    for k, (v, f) in enumerate(zip(a, iv)):
        l, r = f[..., :-1], f[..., 1:]
        if k == 1:
            b = [at(v, j, w) for j in range(5)]
            p0, p2 = at(a[0], 1, w), at(a[0], 3, w)
            sw = 0.5 * S["g"] * (b[3] - b[1]).abs() / torch.minimum(b[1], b[3]) >= (p2 - p0).abs() / torch.minimum(p0, p2)
            d0, d1 = (b[2] - 2 * b[1] + b[0]), (b[4] - 2 * b[3] + b[2])
            on = sw & (-d0 * d1 > 0) & ((b[3] - b[1]).abs() - _C01 * torch.minimum(b[1].abs(), b[3].abs()) > 0)
            e = -_SIXTH * (d1 - d0) / torch.where(b[3] == b[1], 1.0, b[3] - b[1])
            eta = torch.where(on, (20.0 * (e - _C05)).clamp(0.0, 1.0), 0.0)
            l = (1 - eta) * l + eta * (b[1] + 0.5 * at(sl[1], 0, w))
            r = (1 - eta) * r + eta * (b[3] - 0.5 * at(sl[1], 2, w))
        q.append(_limit(at(v, 2, w), l, r, flat))
    c = [at(v, 2, w) for v in a]
    cs = torch.sqrt(S["g"] * c[0] / c[1])
    R, L = _trace(q, c, cs, S, True), _trace(q, c, cs, S, False)
    F = _riemann([v[..., :-1] for v in R], [v[..., 1:] for v in L], S)
    mid = [at(v, NB, n) for v in a]
    return _update(mid, [f[..., :-1] for f in F], [f[..., 1:] for f in F], S, mid[5] if len(a) > 5 else 0.0)


def _sweep(f, direction, S, gforce):
    dim = 3 - direction
    u = ("vx", "vy", "vz")[direction - 1]
    order = ("p", "rho", u) + {1: ("vy", "vz"), 2: ("vx", "vz"), 3: ("vy", "vx")}[direction]
    a = [f[k].transpose(dim, 2) for k in order]
    if gforce is not None:
        a.append(-gforce[..., direction - 1].transpose(dim, 2))
    rows = max(1, 3000000 // (a[0].shape[1] * a[0].shape[2]))
    parts = [_pencils([v[i:i + rows] for v in a], S) for i in range(0, a[0].shape[0], rows)]
    return {k: torch.cat([p[j] for p in parts]).transpose(dim, 2).contiguous() for j, k in enumerate(order)}


_ORDER = ((1, 2, 3), (3, 2, 1), (2, 3, 1), (1, 3, 2), (3, 1, 2), (2, 1, 3))


class _Eds:
    """The Einstein-de Sitter step schedule."""

    def __init__(self):
        self.ca, self.tstop = ic.eds_schedule(A_START, 1.0 / 11.0, 200)
        told = A_START ** 1.5
        self.n, self.dt = 0, float(_F(0.01)) * told
        self.t = told + self.dt
        self._at(told)

    def _at(self, told):
        half = told + 0.5 * self.dt
        self.at, self.dat = told ** _K23, _K23 * told ** _KM13
        ath = half ** _K23
        self.dtat, self.afact = self.dt / ath, self.dt * (_K23 * half ** _KM13 / ath)

    def next(self, vmax, dx):
        self.n += 1
        told, at = self.t, self.t ** _K23
        rdt = 5.0 / (6.0 * self.dt) if self.n > 1 else 0.0
        dt = min(1.0 / max(rdt, vmax / (COUR * dx * at)), ((1.0 + self.ca) * at) ** 1.5 - told)
        dt = 0.1 if dt >= 10.0 else dt
        self.t = min(told + dt, self.tstop)
        self.dt = self.t - told if told + dt > self.tstop else dt
        self._at(told)


def _kick(x, v, g, ngrid, dtat):
    cell = x * torch.tensor([float(n) for n in ngrid], dtype=x.dtype, device=x.device)
    lead = (cell + 0.5).long()
    d = cell - (lead.double() - 0.5)
    i = lead + NB - 1
    force = torch.zeros_like(v)
    for c in range(8):
        o = [(c >> k) & 1 for k in range(3)]
        w = 1.0
        for k in range(3):
            w = w * (d[:, k] if o[k] else 1.0 - d[:, k])
        force += w[:, None] * g[i[:, 2] + o[2], i[:, 1] + o[1], i[:, 0] + o[0]]
    return v + 0.5 * dtat * force


def _evolve(f, ngrid, gamma, steps, sched, gforce, particles):
    S = _scalars(gamma, max(ngrid))
    inner = gforce[NB:-NB, NB:-NB, NB:-NB] if gforce is not None else None
    x = v = None
    vpart = 0.0
    if particles is not None:
        x, v = (torch.from_numpy(a).to(DEV) for a in particles)
        vpart = float(v.abs().max())
        size = torch.tensor(ic.boxsize(ngrid), dtype=x.dtype, device=x.device)
    t = 0.0
    if sched is None:
        t = S["dt"] = S["dtat"] = COUR * S["dx"] / max(_vmax(f, gamma), vpart)
    for step in range(1, steps + 1):
        if sched is not None:
            S.update(dt=sched.dt, dtat=sched.dtat, at=sched.at, dat=sched.dat)
            old = f
        for d in _ORDER[0 if step == 1 else step % 6]:
            f = _sweep(f, d, S, inner)
        if sched is not None:
            af, p = sched.afact, f["p"]
            f = {k: (2.0 * f[k] - af * old[k]) / (2.0 + af) if k in ("vx", "vy", "vz") else f[k] for k in FIELDS}
            pn = (p - af * old["p"]) / (1.0 + af)
            f["p"] = torch.where(pn <= 0, torch.where(p > 0, p, old["p"]), pn)
        if x is not None:
            v = _kick(x, v, gforce, ngrid, 0.01)
            x = x + S["dtat"] * v
            x = torch.where(x < 0, x + size, x)
            x = torch.where(x >= size, x - size, x)
            v = _kick(x, v, gforce, ngrid, 0.01)
            vpart = float(v.abs().max())
        vmax = max(_vmax(f, gamma), vpart)
        if sched is None:
            S["dt"] = S["dtat"] = COUR * S["dx"] / vmax
            t = t + S["dt"]
        else:
            sched.next(vmax, S["dx"])
    times = [t, S["dt"]] if sched is None else [sched.t, sched.dt, sched.at]
    return f, times, () if x is None else (x, v)


def _planar(f, axis):
    """One pencil of a planar tube along `axis`: the others are the same."""
    keep = [slice(0, 1)] * 3
    keep[2 - axis] = slice(None)
    return {k: a[tuple(keep)] for k, a in f.items()}


def _spread(f, shape):
    """A planar tube's pencil back over the whole box."""
    return {k: a.expand(shape) for k, a in f.items()}


def _served(request):
    """Initial tube of a request, one pencil: its seed's axis, split and orientation."""
    h, mask = request["seed"] + 0x9E3779B97F4A7C15, (1 << 64) - 1
    h &= mask
    h = ((h ^ (h >> 30)) * 0xBF58476D1CE4E5B9) & mask
    h = ((h ^ (h >> 27)) * 0x94D049BB133111EB) & mask
    h ^= h >> 31
    axis, x0, flip, n = h % 3, 0.25 + 0.5 * ((h >> 8) & 0xFFFF) / 65536.0, (h >> 40) & 1, request["n"]
    left = ((np.arange(n) + 0.5) / n < x0) != bool(flip)
    view = [1, 1, 1]
    view[2 - axis] = n
    f = {k: torch.zeros(view, dtype=torch.float64, device=DEV) for k in FIELDS}
    for k, (hi, lo) in (("p", (1.0, 0.1)), ("rho", (1.0, 0.125))):
        f[k] = torch.from_numpy(np.where(left, hi, lo)).to(DEV).reshape(view)
    return f


def exact(case, seed):
    gamma = case["gamma"]
    if case["kind"] == "serve":
        out = {"t": [], "steps": None, "state": []}
        for r in _requests(case, seed):
            n = r["n"]
            f, times, _ = _evolve(_served(r), (n, n, n), gamma, r["nsteps"], None, None, None)
            out["t"].append(times[0])
            f = _spread(f, (n, n, n))
            out["state"].append([_pad(f[k]).cpu().numpy().T for k in FIELDS])
        out["t"] = np.array(out["t"])
        return out
    if case["kind"] == "ensemble":
        out = []
        for i, n in enumerate(_boxes(case)):
            f, _, _ = _evolve(_interior(case, seed * 64 + i, (n, n, n)), (n, n, n), gamma, case["steps"],
                              _Eds() if case["cosmo"] else None, None, None)
            out.append([_pad(f[k]).cpu().numpy().T for k in FIELDS])
        return out
    ngrid = (case["nx"], case["ny"], case["nz"])
    full = tuple(reversed(ngrid))
    f = _interior(case, seed)
    g = _gforce(case)
    g = torch.from_numpy(g.T.copy()).to(DEV) if g is not None else None
    if case["kind"] == "sweep":
        S = _scalars(gamma, max(ngrid))
        S["dt"] = S["dtat"] = COUR * S["dx"] / _vmax(f, gamma)
        f = _sweep(f, case["direction"], S, g[NB:-NB, NB:-NB, NB:-NB] if g is not None else None)
        out = [_pad(f[k]) for k in FIELDS]
        for a in out:                     # a sweep fills face ghosts, not edges and corners
            edge = [torch.zeros(n + 2 * NB, dtype=torch.bool, device=a.device) for n in full]
            for e in edge:
                e[:NB] = True
                e[-NB:] = True
            a[edge[0][:, None, None].int() + edge[1][None, :, None].int() + edge[2][None, None, :].int() > 1] = 0.0
        return out
    if case["flow"] == "tube" and g is None:
        f = _planar(f, case["axis"])
    x = ic.particles(ngrid, case["particles"], seed) if case["particles"] else None
    f, times, x = _evolve(f, ngrid, gamma, case["steps"], _Eds() if case["cosmo"] else None, g, x)
    f = _spread(f, full)
    return {"state": [_pad(f[k]) for k in FIELDS], "times": times, "particles": x}
