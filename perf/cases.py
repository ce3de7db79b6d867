"""What the framework's speed is measured on: the hot-path pass, the timestep loop and batches of
boxes, through their public entry points, over the sizes, kernels and arithmetic forms in use.

A case is a dict of plain values; ``kind`` says which entry points it takes:

* ``noalloc``: ``hydro_pass_noalloc`` on device buffers (callers that may not allocate: serving
  loops, code under capture), at most 16,384 particles;
* ``pass``: ``density`` -> ``hydro_gradient_calc`` -> ``hydro_force`` on a resident box whose radii
  the last step converged, every particle or a share of them active, and the results read out;
* ``cold``: the same from ``gz_load`` on, with initial radii that the density rounds iterate;
* ``wide``: ``pass`` on a clustered (lognormal) field with the search over many levels;
* ``job``: a whole short simulation of a point explosion: load, ``run_begin``, ``run_steps``, results;
* ``batch``: an ensemble of boxes of uneven size through one ``Batch``: add, begin, steps, results,
  remove (host data in and out, as a server's requests are).

``gz_load`` and ``gz_store`` copy whichever way their pointers say, so a torch program hands over
device tensors; the batch interface takes host arrays.  The FP32-mixed form's results are kept in
single precision, as snapshots are.
"""
import ctypes
import itertools
import math

import numpy as np
import torch

from gizmo_amd.batch import Batch
from gizmo_amd.hydro import FIELD_WIDTH, GZ_FP32_MIXED, GZ_FP64, Fields, GizmoHipError, Hydro, hydro_pass_noalloc, lib

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
GAMMA = 5.0 / 3.0
VOLNORM = 4.188790204786  # 4 pi / 3 as the reference writes it

# what a program reads back after a pass, and after a run
PASS_OUT = ("h", "rho", "press", "grad_rho", "grad_p", "grad_v", "accel", "dtu", "maxsig")
JOB_OUT = ("pos", "vel", "u", "h", "rho")

# timestep-loop parameters of the point explosion and of an ensemble's boxes
SEDOV_INTEG = dict(courant_fac=0.05, err_tol_int_accuracy=0.002, max_size_timestep=0.01, min_size_timestep=0.0,
                   time_begin=0.0, time_max=1.0, min_egy_spec=0.0, domain_build_active_fraction=0.5)
BATCH_INTEG = dict(courant_fac=0.2, err_tol_int_accuracy=0.02, max_size_timestep=0.01, min_size_timestep=0.0,
                   time_begin=0.0, time_max=100.0, min_egy_spec=0.0)


def listed():
    return [
        # the smallest calls: a few thousand particles, latency and launches
        dict(name="noalloc_16_fp64", kind="noalloc", side=16, kernel=3, mixed=False, mach=0.1),
        # near the static scratch's limit, the serving form (Wendland C2, 64 neighbours, FP32-mixed)
        dict(name="noalloc_25_mixed", kind="noalloc", side=25, kernel=6, mixed=True, mach=1.0),
        # the reference's small test box (cubic spline, 32 neighbours) from its initial conditions
        dict(name="cold_32_fp64", kind="cold", side=32, kernel=3, mixed=False, mach=0.1),
        # an ordinary box with the first-derivative volume correction
        dict(name="pass_64_fp64_fd", kind="pass", side=64, kernel=6, mixed=False, mach=0.5, active=1.0, fd=True),
        # a step of the adaptive timeline that has an eighth of an odd-sized box active
        dict(name="pass_101_fp64_eighth", kind="pass", side=101, kernel=6, mixed=False, mach=0.3, active=0.125, fd=False),
        # the 2M-particle box, every particle active, in both arithmetic forms
        dict(name="pass_128_fp64", kind="pass", side=128, kernel=6, mixed=False, mach=0.3, active=1.0, fd=False),
        dict(name="pass_128_mixed", kind="pass", side=128, kernel=6, mixed=True, mach=0.3, active=1.0, fd=False),
        # clustered fields, radii over two orders of magnitude
        dict(name="wide_1m_fp64", kind="wide", n=1048576, grid=128, mixed=False),
        dict(name="wide_4m_mixed", kind="wide", n=4194304, grid=256, mixed=True),
        # whole jobs on the adaptive timeline: few active rows per step
        dict(name="job_128_fp64_200", kind="job", side=128, steps=200, mixed=False),
        dict(name="job_47_mixed_60", kind="job", side=47, steps=60, mixed=True),
        # an ensemble of boxes of uneven size, stepped together
        dict(name="batch_12_mixed", kind="batch", boxes=12, side_lo=16, side_hi=64, steps=20, mixed=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["noalloc", "pass", "pass", "cold", "wide", "job", "batch"])
    mixed = rng.random() < 0.5
    if kind == "noalloc":
        return dict(kind=kind, side=rng.randint(10, 25), kernel=rng.choice([3, 6]), mixed=mixed, mach=round(rng.uniform(0.1, 1.0), 3))
    if kind == "pass":
        return dict(kind=kind, side=_log_int(rng, 20, 128), kernel=rng.choice([3, 6]), mixed=mixed, mach=round(rng.uniform(0.1, 0.5), 3),
                    active=rng.choice([1.0, 1.0, 0.25, 0.03]), fd=rng.random() < 0.25)
    if kind == "cold":
        return dict(kind=kind, side=_log_int(rng, 20, 110), kernel=rng.choice([3, 6]), mixed=mixed, mach=round(rng.uniform(0.1, 1.0), 3))
    if kind == "wide":
        return dict(kind=kind, n=_log_int(rng, 60000, 3000000), grid=rng.choice([64, 128, 128]), mixed=mixed)
    if kind == "job":
        return dict(kind=kind, side=_log_int(rng, 24, 120), steps=rng.randint(30, 200), mixed=mixed)
    return dict(kind=kind, boxes=rng.randint(2, 12), side_lo=16, side_hi=rng.randint(24, 60), steps=rng.randint(5, 20), mixed=mixed)


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _neighbours_of(kernel):
    return 32.0 if kernel == 3 else 64.0


def _params(kernel, gamma=GAMMA):
    ngb = _neighbours_of(kernel)
    return dict(box=1.0, kernel=kernel, gamma=gamma, des_num_ngb=ngb, max_num_ngb_dev=max(ngb / 640.0, 0.05),
                min_kernel_radius=0.0, max_kernel_radius=0.25, time=0.0, time_begin=0.0)


def _h_guess(n, ngb):
    return (ngb / (VOLNORM * n)) ** (1.0 / 3.0)


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _lattice(side, seed, kernel, mach, pressure=1.0):
    """A periodic unit box: side^3 equal masses on a cubic lattice, each coordinate jittered by up
    to a tenth of a spacing, uniform density 1 and pressure, Gaussian velocities of `mach` sound
    speeds per component."""
    g = _generator(seed)
    n, dx = side ** 3, 1.0 / side
    c = (torch.arange(side, dtype=F64, device=DEV) + 0.5) * dx
    pos = torch.stack(torch.meshgrid(c, c, c, indexing="ij"), dim=-1).reshape(n, 3)
    pos = (pos + (torch.rand(n, 3, dtype=F64, device=DEV, generator=g) - 0.5) * (0.2 * dx)) % 1.0
    vel = torch.randn(n, 3, dtype=F64, device=DEV, generator=g) * (mach * math.sqrt(GAMMA * pressure))
    one = torch.ones(n, dtype=F64, device=DEV)
    return dict(pos=pos, vel=vel, mass=one / n, u=one * (pressure / (GAMMA - 1.0)), h=one * _h_guess(n, _neighbours_of(kernel)))


def _sedov(side, seed):
    """The point explosion: the cold lattice at rest, energy 1 in the 64 particles nearest the
    centre, weighted by the Wendland kernel."""
    f = _lattice(side, seed, 6, 0.0, pressure=1e-6)
    r = (f["pos"] - 0.5).square().sum(1).sqrt()
    near = torch.topk(r, 65, largest=False, sorted=True)
    q = near.values[:64] / near.values[64]
    w = (1 - q) ** 4 * (1 + 4 * q)
    f["u"][near.indices[:64]] += (w / w.sum()) / f["mass"][near.indices[:64]]
    return f


def _lognormal(n, grid, seed):
    """n particles drawn from a lognormal density field (sigma of ln rho 2, P(k) ~ k^-3), nearly
    isothermal (gamma 1.001, P = rho), solenoidal velocities at rms Mach 2."""
    g = _generator(seed)
    k1 = torch.fft.fftfreq(grid, d=1.0 / grid, device=DEV, dtype=F64) * (2 * math.pi)
    kz = torch.fft.rfftfreq(grid, d=1.0 / grid, device=DEV, dtype=F64) * (2 * math.pi)
    k = torch.meshgrid(k1, k1, kz, indexing="ij")
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    amp = torch.where(k2 > 0, k2.clamp_min(1e-30) ** -0.75, torch.zeros_like(k2))

    def white():
        return torch.complex(torch.randn(k2.shape, dtype=F64, device=DEV, generator=g),
                             torch.randn(k2.shape, dtype=F64, device=DEV, generator=g)) * amp

    delta = torch.fft.irfftn(white(), s=(grid,) * 3)
    delta = delta - delta.mean()
    rho = torch.exp(delta * (2.0 / delta.std())).reshape(-1)
    # the draw made over a fixed 2^-40 partition of the cumulated mass (sums of integers: the same on every run)
    w = (rho / rho.sum() * 2.0 ** 40).round().to(torch.int64).clamp_min(1)
    cum = torch.cumsum(w, 0)
    pick = torch.randint(0, 1 << 62, (n,), device=DEV, generator=g) % cum[-1]
    cell = torch.searchsorted(cum, pick, right=True)
    ijk = torch.stack((cell // (grid * grid), (cell // grid) % grid, cell % grid), 1).to(F64)
    pos = ((ijk + torch.rand(n, 3, dtype=F64, device=DEV, generator=g)) / grid) % 1.0
    vk = [white() for _ in range(3)]
    kd = (k[0] * vk[0] + k[1] * vk[1] + k[2] * vk[2]) / k2.clamp_min(1e-30)
    vel = torch.stack([torch.fft.irfftn(v - kc * kd, s=(grid,) * 3).reshape(-1)[cell] for v, kc in zip(vk, k)], 1)
    vel = vel * (2.0 * math.sqrt(1.001) / vel.square().sum(1).mean().sqrt())
    one = torch.ones(n, dtype=F64, device=DEV)
    h = (64.0 / (VOLNORM * n * rho[cell] / rho.mean())) ** (1.0 / 3.0)
    return dict(pos=pos, vel=vel, mass=one / n, u=one / 0.001, h=h.clamp_max(0.2))


def _offsets(reach):
    """The lattice offsets, in ascending order, whose particles can lie within `reach` spacings (of
    jittered lattices: up to 0.2 sqrt(3) nearer than their sites)."""
    m = int(math.ceil(reach + 0.35))
    return [o for o in itertools.product(range(-m, m + 1), repeat=3) if math.sqrt(o[0] ** 2 + o[1] ** 2 + o[2] ** 2) - 0.3465 < reach]


def _shift(x, side, o):
    """The values of the particles at lattice offset o from each (x: n or n x c, lattice order)."""
    return torch.roll(x.reshape(side, side, side, -1), (-o[0], -o[1], -o[2]), (0, 1, 2)).reshape(x.shape)


def _separation(pos, side, o):
    d = pos - _shift(pos, side, o)
    return d - torch.round(d)


def _kernel(kernel, r, h):
    """W(r, h) and dW/dr, zero beyond h."""
    u = r / h
    q = (1 - u).clamp_min(0)
    if kernel == 3:
        norm = 8.0 / math.pi
        w = torch.where(u < 0.5, 1 + 6 * (u - 1) * u * u, 2 * q ** 3)
        dw = torch.where(u < 0.5, u * (18 * u - 12), -6 * q * q)
    else:
        norm = 21.0 / (2.0 * math.pi)
        w = q ** 4 * (1 + 4 * u)
        dw = -20 * u * q ** 3
    return w * norm / h ** 3, dw * norm / h ** 4


def _reach(side, kernel):
    return 1.12 * _h_guess(side ** 3, _neighbours_of(kernel)) * side


def _converged_radii(pos, side, kernel):
    """The radii a converged density pass leaves: the kernel-weighted neighbour number at its
    target (Newton's method from the mean-density guess)."""
    ngb, n = _neighbours_of(kernel), side ** 3
    r = torch.stack([_separation(pos, side, o).square().sum(1).sqrt() for o in _offsets(_reach(side, kernel))])
    h = torch.full((n,), _h_guess(n, ngb), dtype=F64, device=DEV)
    for _ in range(7):
        num, slope = torch.zeros_like(h), torch.zeros_like(h)
        for rk in r:
            w, dw = _kernel(kernel, rk, h)
            num += w
            slope -= 3 * w / h + dw * rk / h
        h = h - (VOLNORM * h ** 3 * num - ngb) / (VOLNORM * (3 * h * h * num + h ** 3 * slope))
    return h


def _sides(case, seed):
    """The boxes of an ensemble: lattice sides log-uniform over the case's range, rms Mach 0.1-5."""
    rng = np.random.Generator(np.random.Philox(1004))  # the mix of sizes is the case's, not the seed's
    sides = [int(round(math.exp(rng.uniform(math.log(case["side_lo"]), math.log(case["side_hi"]))))) for _ in range(case["boxes"])]
    return [(s, float(rng.uniform(0.1, 5.0)), seed * 1009 + k) for k, s in enumerate(sides)]


# ------------------------------------------------------------------------------------------
# prepare and run
# ------------------------------------------------------------------------------------------
def _fields(tensors):
    """gz_fields of device tensors."""
    f = Fields()
    for k, t in tensors.items():
        setattr(f, k, ctypes.cast(ctypes.c_void_p(t.data_ptr()), type(getattr(f, k))))
    return f


def _outputs(names, n):
    return {k: torch.zeros((n, FIELD_WIDTH[k]) if FIELD_WIDTH[k] > 1 else n, dtype=F64, device=DEV) for k in names}


def _check(hydro, rc):
    if rc:
        raise GizmoHipError(rc, lib().gz_last_error(hydro.ctx).decode())


def _load(s):
    _check(s["hydro"], lib().gz_load(s["hydro"].ctx, s["n"], ctypes.byref(s["fin"])))


def _results(s):
    _check(s["hydro"], lib().gz_store(s["hydro"].ctx, ctypes.byref(s["fout"])))
    return _kept(s)


def _kept(s):
    return {k: t.float() for k, t in s["out"].items()} if s["mixed"] else s["out"]


def _inputs(case, seed):
    kind = case["kind"]
    if kind == "wide":
        return _lognormal(case["n"], case["grid"], seed)
    if kind == "job":
        return _sedov(case["side"], seed)
    f = _lattice(case["side"], seed, case["kernel"], case["mach"])
    if kind != "cold":
        f["h"] = _converged_radii(f["pos"], case["side"], case["kernel"])
    return f


def prepare(case, seed):
    kind, mixed = case["kind"], case["mixed"]
    precision = GZ_FP32_MIXED if mixed else GZ_FP64
    if kind == "batch":
        boxes = []
        for side, mach, box_seed in _sides(case, seed):
            f = _lattice(side, box_seed, 6, mach / math.sqrt(3.0))
            boxes.append({k: v.cpu().numpy() for k, v in f.items()})
        batch = Batch(_params(6), sum(len(b["mass"]) for b in boxes), len(boxes), precision)
        return dict(kind=kind, mixed=mixed, batch=batch, boxes=boxes, steps=case["steps"], params=_params(6))
    fin = _inputs(case, seed)
    n = len(fin["mass"])
    params = _params(6, 1.001) if kind == "wide" else _params(6 if kind == "job" else case["kernel"])
    out = _outputs(JOB_OUT if kind == "job" else PASS_OUT, n)
    s = dict(kind=kind, mixed=mixed, n=n, params=params, precision=precision, inputs=fin, out=out, steps=case.get("steps", 0))
    if kind == "noalloc":
        s["dev_in"] = {k: t.data_ptr() for k, t in fin.items()}
        s["dev_out"] = {k: t.data_ptr() for k, t in out.items()}
        return s
    s["hydro"] = hydro = Hydro(params, n, precision)
    s["fin"], s["fout"] = _fields(fin), _fields(out)
    if kind == "wide":
        hydro.set_option("wide_search", 1)
    if case.get("fd"):
        hydro.set_option("fd_correction", 1)
    torch.cuda.synchronize()
    if kind in ("pass", "wide"):
        _load(s)
    if case.get("active", 1.0) < 1.0:
        hydro.hydro_pass()  # the inactive particles' state, as their own last steps left it
        rng = np.random.Generator(np.random.Philox(seed))
        hydro.set_active(rng.random(n) < case["active"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "noalloc":
        hydro_pass_noalloc(s["params"], s["n"], s["dev_in"], s["dev_out"], s["precision"], torch.cuda.current_stream().cuda_stream)
        return _kept(s)
    if kind == "batch":
        b = s["batch"]
        ids = [b.add(f, s["params"], BATCH_INTEG) for f in s["boxes"]]
        b.begin()
        for _ in range(s["steps"]):
            b.step()
        out = [b.store(i, ["pos", "vel", "u", "rho"]) for i in ids]
        for i in ids:
            b.remove(i)
        return [{k: v.astype(np.float32) for k, v in o.items()} for o in out] if s["mixed"] else out
    hydro = s["hydro"]
    if kind in ("cold", "job"):
        _load(s)
    if kind == "job":
        hydro.run_begin(SEDOV_INTEG)
        active, woken = hydro.run_steps(s["steps"])
        hydro.drift_all()
        return dict(_results(s), n_active=np.array(active), n_woken=np.array(woken))
    hydro.density()
    hydro.hydro_gradient_calc()
    hydro.hydro_force()
    return _results(s)


# pair arithmetic of the three stages (operations per pair of the published formulas, divisions
# and square roots counted once)
_DENSITY, _GRADIENTS, _FORCE = 60.0, 60.0, 320.0


def work(case):
    kind = case["kind"]
    if kind == "batch":
        rows = sum(side ** 3 for side, _, _ in _sides(case, 0))
        n, ngb, passes, values = rows, 64.0, 1.0 + 0.5 * case["steps"], 9 + 8
    elif kind == "job":
        # the start's two density passes and one pass, then steps over a few hundred rows
        n, ngb, values = case["side"] ** 3, 64.0, 9 + 9
        passes = 1.2 + 300.0 * case["steps"] / n
    else:
        n = case["n"] if kind == "wide" else case["side"] ** 3
        ngb, values = (64.0 if kind == "wide" else _neighbours_of(case["kernel"])), 9 + sum(FIELD_WIDTH[k] for k in PASS_OUT)
        passes = case.get("active", 1.0)
    size = 8.0
    return {"bytes": n * values * size, "flops": n * passes * ngb * (_DENSITY + _GRADIENTS + _FORCE)}


# ------------------------------------------------------------------------------------------
# the pass in plain 64-bit torch, for lattices with converged radii (each particle's partners are
# its lattice neighbours: one vector operation over all particles per lattice offset)
# ------------------------------------------------------------------------------------------
def _inverse3(t):
    """Inverse of the symmetric matrices [xx, yy, zz, xy, yz, xz] (n x 6), and their condition number."""
    m = torch.stack((t[:, 0], t[:, 3], t[:, 5], t[:, 3], t[:, 1], t[:, 4], t[:, 5], t[:, 4], t[:, 2]), 1).reshape(-1, 3, 3)
    inv = torch.linalg.inv(m)
    cn = (m.square().sum((1, 2)) * inv.square().sum((1, 2))).sqrt() / 3
    return inv, cn.clamp_min(1.0)


def _limit(grad, cmax, cmin, h, tol, alim, positive=None, dmax=None):
    size = grad.square().sum(1).sqrt()
    hi, lo = torch.maximum(cmax.abs(), cmin.abs()), torch.minimum(cmax.abs(), cmin.abs())
    fc = torch.minimum(lo + tol * hi, hi)
    fac = fc / (alim * h * size)
    if positive is not None:
        floor = torch.minimum(positive, torch.minimum(0.5 * (positive + cmin), positive - fc).clamp_min(0))
        fac = torch.minimum(fac, (positive - floor) / dmax / size)
    return torch.where(((size > 0) & (fac < 1))[:, None], grad * fac[:, None], grad)


def _face_values(qi, gi, qj, gj, di, dj):
    """The two sides' values at the face, limited between the particles' values."""
    r, l = qi + (gi * di).sum(1), qj + (gj * dj).sum(1)
    top, low, mid = torch.maximum(qi, qj), torch.minimum(qi, qj), 0.5 * (qi + qj)
    half, med = 0.5 * (top - low), 0.375 * (top - low)
    te, le = top + half, low - half
    te = torch.where((top < 0) & (te > 0), top * top / (top - half), te)
    le = torch.where((low > 0) & (le < 0), low * low / (low + half), le)
    mt, ml = torch.minimum(mid + med, te), torch.maximum(mid - med, le)
    up = qi < qj
    r2 = torch.where(up, torch.minimum(torch.maximum(r, le), mt), torch.maximum(torch.minimum(r, te), ml))
    l2 = torch.where(up, torch.maximum(torch.minimum(l, te), ml), torch.minimum(torch.maximum(l, le), mt))
    same = qi == qj
    return torch.where(same, qi, l2), torch.where(same, qi, r2)


def _exact_star(rl, pl, vl, cl, rr, pr, vr, cr):
    """Pressure and speed of the contact of the exact Riemann solution (Newton's method)."""
    g1, g2, g4, g5, g6 = (GAMMA - 1) / (2 * GAMMA), (GAMMA + 1) / (2 * GAMMA), 2 / (GAMMA - 1), 2 / (GAMMA + 1), (GAMMA - 1) / (GAMMA + 1)
    p = torch.maximum(0.5 * (pl + pr) - 0.125 * (vr - vl) * (pl + pr) * (cl + cr), 1e-6 * (pl + pr))
    vacuum = g4 * (cl + cr) < vr - vl

    def wave(p, rho, pk, c):
        s = torch.sqrt(g5 / rho / (p + g6 * pk))
        shock = p > pk
        ratio = p / pk
        f = torch.where(shock, (p - pk) * s, g4 * c * (ratio ** g1 - 1))
        df = torch.where(shock, s * (1 - 0.5 * (p - pk) / (g6 * pk + p)), ratio ** -g2 / (rho * c))
        return f, df

    for _ in range(60):
        (fl, dl), (fr, dr) = wave(p, rl, pl, cl), wave(p, rr, pr, cr)
        p = torch.maximum(p - (fl + fr + vr - vl) / (dl + dr), 0.1 * p)
    fl, fr = wave(p, rl, pl, cl)[0], wave(p, rr, pr, cr)[0]
    s = 0.5 * (vl + vr) + 0.5 * (fr - fl)
    sl, sr = vl + g4 * cl, vr - g4 * cr
    sv = torch.where(sl >= 0, sl, torch.where(sr <= 0, sr, torch.zeros_like(sl)))
    return torch.where(vacuum, torch.zeros_like(p), p), torch.where(vacuum, sv, s)


def _riemann(rl, pl, ul, rr, pr, ur, n, limit):
    """Star pressure and speed and the fluxes (momentum along n, energy) between two states (u:
    velocities n x 3): the first of HLLC, Roe-averaged and primitive-variable estimates within the
    pressure limit, else the exact star state (whose fluxes stay the last estimate's)."""
    tiny = 1e-56
    vl, vr = (ul * n).sum(1), (ur * n).sum(1)
    cl, cr = (GAMMA * pl / rl).sqrt(), (GAMMA * pr / rr).sqrt()
    cmax = torch.maximum(cl, cr)
    wl, wr = rl * (torch.minimum(vl, vr) - cmax - vl), rr * (torch.maximum(vl, vr) + cmax - vr)
    s = ((pr - pl) + wl * vl - wr * vr) / (wl - wr)
    p = (pl * wr - pr * wl + wl * wr * (vr - vl)) / (wr - wl)
    s, p = torch.where(p <= tiny, torch.zeros_like(s), s), p.clamp_min(tiny)
    bad = ~(p <= limit)
    hl, hr = GAMMA / (GAMMA - 1) * pl / rl + 0.5 * ul.square().sum(1), GAMMA / (GAMMA - 1) * pr / rr + 0.5 * ur.square().sum(1)
    al, ar = rl.sqrt(), rr.sqrt()
    uroe = (al[:, None] * ul + ar[:, None] * ur) / (al + ar)[:, None]
    vroe, hroe = (uroe * n).sum(1), (al * hl + ar * hr) / (al + ar)
    croe = ((GAMMA - 1) * (hroe - 0.5 * uroe.square().sum(1))).clamp_min(1e-30).sqrt()
    sl, sr = torch.minimum(vl - cl, vroe - croe), torch.maximum(vr + cr, vroe + croe)
    wl, wr = -rl * (sl - vl), rr * (sr - vr)
    s2 = ((wr * vr + wl * vl) + (pl - pr)) / (wr + wl)
    p2 = rl * (vl - sl) * (vl - s2) + pl
    s2, p2 = torch.where(p2 <= tiny, torch.zeros_like(s2), s2), p2.clamp_min(tiny)
    s, p = torch.where(bad, s2, s), torch.where(bad, p2, p)
    bad = bad & ~(p2 <= limit)
    p3 = 0.5 * ((pl + pr) + (vl - vr) * 0.25 * (rl + rr) * (cl + cr))
    s3 = 0.5 * (vr + vl) + 2 * (pl - pr) / ((rl + rr) * (cl + cr))
    sp = torch.maximum(torch.maximum((vl - cl).abs(), (vr - cr).abs()), torch.maximum((vl + cl).abs(), (vr + cr).abs()))
    s3 = torch.maximum(torch.minimum(s3, sp), -sp)
    s3, p3 = torch.where(p3 <= tiny, torch.zeros_like(s3), s3), p3.clamp_min(tiny)
    s, p = torch.where(bad, s3, s), torch.where(bad, p3, p)
    vacuum = vr - vl > cmax
    s, p = torch.where(vacuum, torch.zeros_like(s), s), torch.where(vacuum, torch.full_like(p, tiny), p)
    fm, fe = p.clone(), p * s
    at = torch.nonzero(~(p <= limit)).reshape(-1)
    if len(at):
        p[at], s[at] = _exact_star(rl[at], pl[at], vl[at], cl[at], rr[at], pr[at], vr[at], cr[at])
    return p, s, fm, fe


def _force_of_pairs(kernel, I, J, dp, r):
    """Fluxes (momentum n x 3, energy) of each pair on particle i and its signal speed."""
    (wi, dwi), (wj, dwj) = _kernel(kernel, r, I["h"]), _kernel(kernel, r, J["h"])
    dv = I["vel"] - J["vel"]
    vdr = (dp * dv).sum(1) / r
    signal = I["cs"] + J["cs"] - vdr.clamp_max(0) + (I["cs"] - J["cs"]).abs()
    vi, vj = I["mass"] / I["rho"], J["mass"] / J["rho"]
    leak = 0.5 * (I["fce"] + J["fce"])
    far = (vi - vj).abs() / torch.minimum(vi, vj) / 3 > 1.25
    mean = vi * vj * (wi + wj) / (vi * wi + vj * wj)
    ti, tj = torch.where(far, mean, vi), torch.where(far, mean, vj)
    area = (wi * ti)[:, None] * (I["inv"] @ dp[:, :, None])[:, :, 0] + (wj * tj)[:, None] * (J["inv"] @ dp[:, :, None])[:, :, 0]
    back = (area * dp).sum(1) < 0
    simple = -(ti * vi * dwi + tj * vj * dwj) / r
    area = torch.where(back[:, None], dp * simple[:, None], area)
    size = area.square().sum(1).sqrt()
    n = area / size[:, None]
    half = 0.5 * dp
    vf = 0.5 * (I["vel"] + J["vel"])
    fvi, fvj = (I["vel"] * n).sum(1), (J["vel"] * n).sum(1)
    adv = 0.5 * (fvi + fvj)
    va2 = torch.maximum(vdr.clamp_max(0).square(), (fvi - fvj).clamp_max(0).square())
    first = (leak > 1)[:, None]

    def both(a, b, ga, gb):
        l, rr = _face_values(a, ga, b, gb, -half, half)
        return torch.where(first[:, 0], b, l), torch.where(first[:, 0], a, rr)

    rl, rr = both(I["rho"], J["rho"], I["grad_rho"], J["grad_rho"])
    pl, pr = both(I["press"], J["press"], I["grad_p"], J["grad_p"])
    ui, uj = I["vel"] - vf, J["vel"] - vf
    comp = [both(ui[:, c], uj[:, c], I["grad_v"][:, 3 * c:3 * c + 3], J["grad_v"][:, 3 * c:3 * c + 3]) for c in range(3)]
    ul, ur = torch.stack([c[0] for c in comp], 1), torch.stack([c[1] for c in comp], 1)
    limit = 1.1 * torch.maximum(I["press"] + I["rho"] * va2, J["press"] + J["rho"] * va2)
    limit = torch.where(first[:, 0], torch.maximum(limit, torch.maximum(torch.maximum(I["press"], J["press"]),
                                                                        2 * torch.maximum(I["rho"], J["rho"]) * va2)), limit)
    p, s, fm, fe = _riemann(rl, pl, ul, rr, pr, ur, n, limit)
    for scale, zero in ((1.4, 0.0), (2.0, 1.0)):  # first-order states, then at rest
        at = torch.nonzero((p < 0) | torch.isnan(p) | ((p > 1.4 * limit) if not zero else torch.zeros_like(p, dtype=torch.bool))).reshape(-1)
        if len(at):
            k = 1.0 - zero
            got = _riemann(J["rho"][at], J["press"][at], uj[at] * k, I["rho"][at], I["press"][at], ui[at] * k, n[at], scale * limit[at])
            p[at], s[at], fm[at], fe[at] = got
    live = p > 0
    mom = (size * fm)[:, None] * n
    energy = size * (fe + fm * (vf * n).sum(1))
    # the entropic switch of the energy flux
    smc = s.abs() / torch.minimum(I["cs"], J["cs"])
    fpm = p * size
    pdi, pdj = dwi * vi * vi * I["drk"] * p * vdr, dwj * vj * vj * J["drk"] * p * vdr
    old, new = fpm * (s + adv), 0.5 * (pdi - pdj + fpm * (fvi + fvj))
    ei, ej = I["press"] / I["rho"], J["press"] / J["rho"]
    oj, oi, nj, ni = -old + fpm * fvj, old - fpm * fvi, -new + fpm * fvj, new - fpm * fvi
    hot, cold = ei > 1.001 * ej, (ei <= 1.001 * ej) & (1.001 * ei < ej)
    rej_j, rej_i = (oj < 0) & (oj > nj), (oi < 0) & (oi > ni)
    no = torch.where(hot, (oj > 0) | rej_j, torch.where(cold, (oi > 0) | rej_i, rej_j | rej_i)) & (smc > 1e-3)
    use = ((smc < 0.5) | (leak > 1)) & ~no
    energy = energy + torch.where(use, new - old, torch.zeros_like(old))
    zero = torch.zeros_like(energy)
    return torch.where(live[:, None], mom, zero[:, None]), torch.where(live, energy, zero), signal


def exact(case, seed):
    """The pass of a lattice box whose radii are converged (kinds pass and noalloc); the other
    kinds iterate radii or step a timeline, and have no value apart from that iteration."""
    if case["kind"] not in ("pass", "noalloc"):
        return None
    side, kernel = case["side"], case["kernel"]
    f = _inputs(case, seed)
    n, h, pos, vel, mass, u = side ** 3, f["h"], f["pos"], f["vel"], f["mass"], f["u"]
    offsets = _offsets(_reach(side, kernel))
    if len({tuple(x % side for x in o) for o in offsets}) < len(offsets):
        return None  # a box too small for its offsets to be distinct
    zero = torch.zeros(n, dtype=F64, device=DEV)
    num, drn, dvs, t, fw, gh, ghd = zero.clone(), zero.clone(), zero.clone(), [zero.clone() for _ in range(6)], torch.zeros_like(pos), torch.zeros_like(pos), zero.clone()
    for o in offsets:
        dp = _separation(pos, side, o)
        r = dp.square().sum(1).sqrt()
        w, dw = _kernel(kernel, r, h)
        num += w
        drn -= 3 * w / h + r / h * dw
        if o == (0, 0, 0):
            continue
        for k, (a, b) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))):
            t[k] += w * dp[:, a] * dp[:, b]
        fw += w[:, None] * dp
        dvs -= dw * (dp * (vel - _shift(vel, side, o))).sum(1) / r
        gh += (dw / r)[:, None] * dp
        ghd += r / h * dw
    drk = drn * h / (3 * num)
    drk = torch.where(drk > -0.9, 1 / (1 + drk), torch.ones_like(drk))
    vol = 1 / num
    inv, cn = _inverse3(torch.stack(t, 1))
    trace = t[0] + t[1] + t[2]
    leak = (2 * vol[:, None] * (inv @ fw[:, :, None])[:, :, 0]).abs().sum(1) / 3
    fce = leak / (6 * vol * trace)
    if float(cn.max()) > 100 or float(fce.max()) > 0.35:
        return None  # the neighbour target would not be the plain one
    rho = mass * num
    if case.get("fd"):
        rho = rho / (1 + 4 * (3.0 / 16.0 if kernel == 3 else 1.0 / 6.0) * (gh / ghd[:, None]).square().sum(1))
    press = (GAMMA - 1) * u * rho
    cs = (GAMMA * press / rho).sqrt()
    q = torch.cat((rho[:, None], press[:, None], vel), 1)
    sums = torch.zeros(n, 3, 5, dtype=F64, device=DEV)
    top, low, dmax = torch.zeros_like(q), torch.zeros_like(q), h.clone()
    near = [o for o in offsets if o != (0, 0, 0)]
    for o in near:
        dp = _separation(pos, side, o)
        r = dp.square().sum(1).sqrt()
        mine, pair = r < h, r < torch.maximum(h, _shift(h, side, o))
        w = torch.where(mine, _kernel(kernel, r, h)[0], zero)
        d = torch.where(pair[:, None], _shift(q, side, o) - q, torch.zeros_like(q))
        sums -= (w[:, None] * dp)[:, :, None] * d[:, None, :]
        top, low, dmax = torch.maximum(top, d), torch.minimum(low, d), torch.maximum(dmax, torch.where(pair, r, zero))
    grad = (inv @ sums).transpose(1, 2)  # n x quantity x direction
    g = [_limit(grad[:, 0], top[:, 0], low[:, 0], h, 0.0, 0.25, rho, dmax), _limit(grad[:, 1], top[:, 1], low[:, 1], h, 0.1, 0.25, press, dmax)]
    g += [_limit(grad[:, 2 + c], top[:, 2 + c], low[:, 2 + c], h, 0.1, 0.25) for c in range(3)]
    grad_v = torch.cat(g[2:], 1)
    mine = dict(h=h, mass=mass, rho=rho, press=press, cs=cs, fce=fce, drk=drk, vel=vel, grad_rho=g[0], grad_p=g[1], grad_v=grad_v, inv=inv)
    mom, energy, signal = torch.zeros_like(pos), zero.clone(), cs.clone()
    for o in near:
        dp = _separation(pos, side, o)
        r = dp.square().sum(1).sqrt()
        at = torch.nonzero(r < torch.maximum(h, _shift(h, side, o))).reshape(-1)
        if not len(at):
            continue
        I = {k: v[at] for k, v in mine.items()}
        J = {k: _shift(v.reshape(n, -1), side, o).reshape(v.shape)[at] for k, v in mine.items()}
        fm, fe, sig = _force_of_pairs(kernel, I, J, dp[at], r[at])
        mom[at] += fm
        energy[at] += fe
        signal[at] = torch.maximum(signal[at], sig)
    return dict(h=h, rho=rho, press=press, grad_rho=g[0], grad_p=g[1], grad_v=grad_v, accel=mom / mass[:, None],
                dtu=(energy - (vel * mom).sum(1)) / mass, maxsig=signal)
