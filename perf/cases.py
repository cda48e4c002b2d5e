"""What this framework is timed on: the calls a user's program makes, over the range of grids that it makes them on.

Four ways in, each through public entry points:

* `run`      a resident grid advanced by `Hydro.run` from one output time to the next, with the state downloaded there
             (the snapshot that the program writes): 1-D tubes, 2-D and 3-D grids, dual energy, conduction, gravity
* `driver`   the same grid stepped by the routine-level calls that the Fortran driver makes, with the conservation sums
             that it writes every ten steps
* `batch`    an ensemble of small independent boxes, replayed as a graph by `Batch.run`
* `noalloc`  boxes in the caller's own device buffers, advanced by `run_noalloc`

A pass goes on from the state that the pass before left, as a run between two outputs does.
"""
import math

import numpy as np
import torch

from evora_amd.batch import Batch, run_noalloc
from evora_amd.hydro import FP32_MIXED, FP64, MODE_FUSED_EXACT, Hydro
from evora_amd.params import HydroParams

F64 = torch.float64


def _case(name, way, problem, nx, ny, nz, steps, precision="fp64", exact=False, solver=2, limiter=1, boundtype=2,
          cfl=0.4, atomic=True, mild=False, boxes=1, edge_lo=0, edge_hi=0, size_seed=0):
    return dict(name=name, way=way, problem=problem, nx=nx, ny=ny, nz=nz, steps=steps, precision=precision, exact=exact,
                solver=solver, limiter=limiter, boundtype=boundtype, cfl=cfl, atomic=atomic, mild=mild, boxes=boxes,
                edge_lo=edge_lo, edge_hi=edge_hi, size_seed=size_seed)


def listed():
    return [
        # The 1-D shock tube of 1000 cells (gamma 5/3, HLLC, CFL 0.8): the smallest grid in use, bound by launches.
        _case("sod_1000", "run", "sod", 1000, 1, 1, 100, boundtype=1, cfl=0.8),
        # The 2-D Kelvin-Helmholtz parameter file: 128 x 128, gamma 1.4, monotonized central.
        _case("kh2d_128", "run", "kh", 128, 128, 1, 100, limiter=2, atomic=False),
        # A large 2-D shear layer, ragged in both directions.
        _case("kh2d_4000x3001", "run", "kh", 4000, 3001, 1, 60),
        # A small 3-D blast stepped by the driver's own calls (primitive, bound, hydrostep, compevo, sweep).
        _case("driver_blast_64", "driver", "blast", 64, 64, 64, 40, boundtype=1),
        # An odd box in the form with the reference's arithmetic: HLL, van Leer, reflecting upper x.
        _case("exact_hll_197x101x131", "run", "blast", 197, 101, 131, 40, exact=True, solver=1, limiter=3, boundtype=3),
        # The headline: the HLLC point blast on 512^3, FP64 and FP32-mixed, in the caller's buffers.
        _case("blast_512", "noalloc", "blast", 512, 512, 512, 6, boundtype=1),
        _case("blast_512_mixed", "noalloc", "blast", 512, 512, 512, 8, precision="mixed", boundtype=1),
        # The supersonic field of a cosmological box with the dual-energy switch.
        _case("cosmo_256_dual", "run", "cosmo", 256, 256, 256, 30),
        # A hot blob with thermal conduction.
        _case("blob_256_conduction", "run", "blob", 256, 256, 256, 30),
        # A self-gravitating periodic box.
        _case("jeans_256_gravity", "run", "jeans", 256, 256, 256, 30),
        # The shock-cloud ensemble: boxes of uneven sizes in the caller's buffers, FP32-mixed.
        _case("ensemble_24_mixed", "noalloc", "cloud", 0, 0, 0, 10, precision="mixed", boundtype=1, boxes=24, edge_lo=64,
              edge_hi=192, size_seed=7),
        # Many small boxes as a replayed graph.
        _case("batch_32_small", "batch", "cloud", 0, 0, 0, 40, boundtype=1, boxes=32, edge_lo=16, edge_hi=48, size_seed=3),
    ]


def draw(rng):
    """One more case of the same ways and ranges; at most about 1e9 cell updates in a pass."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    opts = dict(solver=rng.choice([1, 2, 2]), limiter=rng.choice([1, 2, 3]), boundtype=rng.choice([1, 2, 3]))
    kind = rng.choice(["tube", "2d", "3d", "3d", "driver", "cosmo", "blob", "jeans", "noalloc", "ensemble", "batch"])
    if kind == "tube":
        c = _case("", "run", "sod", size(100, 4000), 1, 1, rng.randint(50, 150), boundtype=rng.choice([1, 3]), cfl=0.8,
                  solver=opts["solver"], limiter=opts["limiter"])
    elif kind == "2d":
        c = _case("", "run", "kh", size(60, 4000), size(60, 4000), 1, rng.randint(40, 100),
                  precision=rng.choice(["fp64", "mixed"]), atomic=rng.choice([True, False]), solver=opts["solver"],
                  limiter=opts["limiter"])
    elif kind in ("3d", "driver"):
        hi = 280 if kind == "3d" else 100
        c = _case("", "run" if kind == "3d" else "driver", rng.choice(["blast", "kh"]), size(24, hi), size(24, hi),
                  size(24, hi), rng.randint(20, 40), precision=rng.choice(["fp64", "fp64", "mixed"]), **opts)
        if c["problem"] == "kh":
            c["boundtype"] = 2
        if c["precision"] == "fp64":
            c["exact"] = rng.random() < 0.25
    elif kind in ("cosmo", "blob", "jeans"):
        n = [rng.choice([32, 64, 128, 256]) if rng.random() < 0.5 else size(32, 256) for _ in range(3)]
        c = _case("", "run", kind, n[0], n[1], n[2], rng.randint(10, 30), precision=rng.choice(["fp64", "mixed"]),
                  limiter=opts["limiter"] if kind != "cosmo" else 1)
    elif kind == "noalloc":
        c = _case("", "noalloc", "blast", size(64, 512), size(64, 400), size(64, 400), rng.randint(3, 8),
                  precision=rng.choice(["fp64", "mixed"]), solver=opts["solver"], boundtype=1)
    elif kind == "ensemble":
        c = _case("", "noalloc", "cloud", 0, 0, 0, rng.randint(4, 10), precision=rng.choice(["fp64", "mixed"]),
                  boundtype=1, boxes=rng.randint(3, 20), edge_lo=size(32, 64), edge_hi=size(80, 192),
                  size_seed=rng.randint(0, 999))
    else:
        c = _case("", "batch", "cloud", 0, 0, 0, rng.randint(20, 40), boundtype=1, boxes=rng.randint(8, 40),
                  edge_lo=size(12, 20), edge_hi=size(24, 56), size_seed=rng.randint(0, 999))
    del c["name"]
    if c["problem"] in ("blast", "kh", "cosmo", "jeans"):
        c["mild"], c["cfl"] = True, 0.3  # weaker flows: any box, limiter and boundary runs on without an error stop
    return c


# ---------------------------------------------------------------------------- the boxes of a case

def _params(case, n):
    nx, ny, nz = n
    prob = case["problem"]
    kw = dict(nx=nx, ny=ny, nz=nz, solver=case["solver"], limiter=case["limiter"], boundtype=case["boundtype"],
              cfl=case["cfl"], atomic=case["atomic"], tstart=0.0, tend=1e30)
    mid = 0.5 if prob == "blast" else 0.0
    for d, m in zip("xyz", n):  # cubic cells, the longest side 1; the blast is centred on the origin
        kw[d + "min"], kw[d + "max"] = -mid * m / max(n), (1 - mid) * m / max(n)
    if prob == "cosmo":
        kw.update(dualenergy=True, de_thresh=0.01)
    elif prob == "blob":
        kw.update(conduction=True, simplekappa=True)
    elif prob == "jeans":
        kw.update(gravity=True)
    return HydroParams(**kw)


def _sizes(case):
    """The grids of the case: one, or an ensemble of cubes and bricks drawn from its own seed."""
    if not case["edge_hi"]:
        return [(case["nx"], case["ny"], case["nz"])]
    rng = np.random.default_rng(case["size_seed"])
    lo, hi = math.log(case["edge_lo"]), math.log(case["edge_hi"])
    return [tuple(int(round(e)) for e in np.exp(rng.uniform(lo, hi, 3))) for _ in range(case["boxes"])]


def _initial(case, n, gen):
    """The box's initial state as q[6][nz][ny][nx] on the GPU in FP64: the problems of evora_amd.ics, with the seed in
    their noise, their phases and, for the shock-cloud boxes, Mach number and density contrast."""
    nx, ny, nz = n
    prob = case["problem"]
    c = _constants(case, n)
    g1, dev, shape = c["g1"], "cuda", (nz, ny, nx)
    # cell centres as shares of the box (x, y, z in 0..1) and their distances from its middle
    x, y, z = ((torch.arange(m, dtype=F64, device=dev) + 0.5) / m for m in n)
    x, y, z = x[None, None, :], y[None, :, None], z[:, None, None]
    r2 = sum(((s - 0.5) * m * c["dx"]) ** 2 for s, m in zip((x, y, z), n) if m > 1)

    def noise(a):
        return (torch.rand(shape, generator=gen, dtype=F64, device=dev) * 2 - 1) * a

    one = torch.ones(shape, dtype=F64, device=dev)
    vx = vy = vz = 0.0 * one
    extra = None
    if prob == "sod":
        left = (x < 0.5) & (one > 0)
        rho = torch.where(left, 1.0, 0.125) * (1 + noise(1e-3))
        p = torch.where(left, 1.0, 0.1) * one
    elif prob == "kh":
        inner = (y - 0.5).abs() < 0.25
        rho = torch.where(inner, 2.0, 1.0) * one
        vx = torch.where(inner, 0.5, -0.5) * one + noise(1e-4)
        bumps = torch.exp(-(y - 0.25) ** 2 / 0.005) + torch.exp(-(y - 0.75) ** 2 / 0.005)
        vy = 0.01 * torch.sin(4 * math.pi * x) * bumps * one + noise(1e-4)
        vz = noise(1e-4) if nz > 1 else vz
        p = 2.5 * one
    elif prob == "blast":
        rho = 1 + noise(0.01)
        p = (1e-2 if case["mild"] else 1e-5) * one
        inside = r2.sqrt() < 3.5 * c["dx"]
        e0 = 1.0 / (c["dx"] ** 3 * int(inside.sum()))
        extra = (inside, e0 * g1)
    elif prob == "cosmo":
        k = [torch.fft.fftfreq(m, 1.0 / m, dtype=F64, device=dev) for m in (nz, ny)]
        k.append(torch.fft.rfftfreq(nx, 1.0 / nx, dtype=F64, device=dev))
        kz, ky, kx = k[0][:, None, None], k[1][None, :, None], k[2][None, None, :]
        k2 = kx * kx + ky * ky + kz * kz
        k2[0, 0, 0] = 1.0
        white = torch.fft.rfftn(torch.randn(shape, generator=gen, dtype=F64, device=dev))
        amp = k2 ** (-2.5 / 4.0)
        amp[0, 0, 0] = 0.0
        delta = torch.fft.irfftn(white * amp, s=shape)
        delta = delta * (0.5 / delta.std())
        rho = (1 + delta).clamp_min(0.05)
        dk = torch.fft.rfftn(delta) / k2
        v = [torch.fft.irfftn(1j * m * dk, s=shape) for m in (kx, ky, kz)]
        scale = (1.5 if case["mild"] else 10.0) * math.sqrt(c["g"]) / float((v[0] ** 2 + v[1] ** 2 + v[2] ** 2).mean().sqrt())
        vx, vy, vz = (m * scale for m in v)
        p = rho.clone()
    elif prob == "blob":
        rho = 1 + noise(0.01)
        p = rho * (1000.0 + 2000.0 * torch.exp(-r2 / 0.04))
        vx, vy, vz = (noise(0.01 * math.sqrt(c["g"] * 1000.0)) for _ in range(3))
    elif prob == "jeans":
        rho = 1e6 * (1 + 0.1 * torch.cos(2 * math.pi * x) * torch.cos(2 * math.pi * y) + noise(0.01))
        length = 2.0 if case["mild"] else 0.5  # the Jeans length in box units: 0.5 collapses, 2 oscillates
        cs2 = length ** 2 * c["grav"] * 1e6 / (4 * math.pi ** 2)
        p = 1e6 * cs2 / c["g"] * one
        vx, vy, vz = (noise(0.01 * math.sqrt(cs2)) for _ in range(3))
    else:  # cloud: a Mach 3-30 shock towards a sphere 10-100 times denser than the gas around it
        r = torch.rand(2, generator=gen, dtype=F64, device=dev).tolist()
        mach, chi, g = 3 + 27 * r[0], 10 + 90 * r[1], c["g"]
        rho2 = (g + 1) * mach ** 2 / ((g - 1) * mach ** 2 + 2)
        p2 = (2 * g * mach ** 2 - (g - 1)) / (g + 1)
        post = (x < 0.1) & (one > 0)
        cloud = (x - 0.3) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2 < 0.01
        rho = torch.where(post, rho2, torch.where(cloud, chi, 1.0))
        vx = torch.where(post, mach * math.sqrt(g) * (1 - 1 / rho2), 0.0) * one
        p = torch.where(post, p2, 1.0) * one
    if extra is not None:
        p = torch.where(extra[0], extra[1], p)
    q = torch.empty((6,) + shape, dtype=F64, device=dev)
    q[0] = rho
    q[1] = rho * vx
    q[2] = rho * vy
    q[3] = rho * vz
    q[4] = 0.5 * rho * (vx * vx + vy * vy + vz * vz) + p / g1
    q[5] = p / rho ** g1
    return q


def _boxes(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return [_initial(case, n, gen) for n in _sizes(case)]


def _host(q):
    """q[6][nz][ny][nx] on the GPU as the host array of the reference's layout, (nz, ny, nx, 6)."""
    return q.permute(1, 2, 3, 0).contiguous().cpu().numpy()


# ---------------------------------------------------------------------------- one pass

def prepare(case, seed):
    sizes = _sizes(case)
    prec = FP32_MIXED if case["precision"] == "mixed" else FP64
    params = [_params(case, n).derive() for n in sizes]
    state = dict(case=case, params=params, prec=prec)
    if case["way"] in ("run", "driver"):
        state["h"] = h = Hydro(params[0], precision=prec, mode=MODE_FUSED_EXACT if case["exact"] else None)
        h.upload_q(_host(_boxes(case, seed)[0]))
        state["t"] = 0.0
    elif case["way"] == "batch":
        state["b"] = b = Batch(params, precision=prec)
        for i, q in enumerate(_boxes(case, seed)):
            b.upload_q(i, _host(q))
    else:
        kind = torch.float32 if prec == FP32_MIXED else F64
        q0 = torch.cat([q.to(kind).reshape(-1) for q in _boxes(case, seed)])
        n = len(sizes)
        state.update(q=(q0, torch.empty_like(q0)), side=np.zeros(n, np.int32), times=np.zeros(n),
                     tend=np.full(n, 1e30), steps=np.zeros(n, np.int32), go=np.ones(n, np.int32))
        torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return state


def _snapshot(state, q):
    """A downloaded state, time or sum in the precision that the form holds the state in: what the program would write."""
    q = torch.as_tensor(q, dtype=F64)
    return q.float() if state["prec"] == FP32_MIXED else q


def run(state):
    case, params = state["case"], state["params"]
    if case["way"] == "run":
        h = state["h"]
        state["t"], dt, done = h.run(case["steps"], t=state["t"], tend=1e30)
        out = dict(q=_snapshot(state, h.download_q()), t=_snapshot(state, state["t"]), dt=_snapshot(state, dt), done=done)
        if params[0].gravity:
            out["phi"] = torch.from_numpy(h.download_phi())
        return out
    if case["way"] == "driver":
        h, sums = state["h"], []
        for k in range(case["steps"]):
            h.primitive()
            h.bound()
            dt = h.hydrostep(1e99)
            h.compevo(dt)
            h.sweep(dt)
            state["t"] += dt
            if k % 10 == 9:
                sums.append(h.sums())
        return dict(q=_snapshot(state, h.download_q()), t=_snapshot(state, state["t"]),
                    sums=_snapshot(state, np.array(sums)))
    if case["way"] == "batch":
        b = state["b"]
        b.run(case["steps"], graph=True)
        t, dt, steps, _ = b.times()
        return dict(q=torch.cat([_snapshot(state, b.download_q(i)).reshape(-1) for i in range(b.n)]),
                    t=_snapshot(state, t), dt=_snapshot(state, dt))
    run_noalloc(params, state["q"][0].data_ptr(), state["q"][1].data_ptr(), state["side"], state["times"],
                state["tend"], state["steps"], state["go"], case["steps"], precision=state["prec"])
    # every running box has taken the same number of steps, so one buffer holds them all
    return dict(q=state["q"][int(state["side"][0])], t=_snapshot(state, state["times"].copy()))


def work(case):
    """Each step reads q and writes the new q (conduction and gravity: their pass too, which reads q and writes what it
    changes; the potential reads the density and writes phi), and the snapshot crosses to the host once.  Operations:
    additions, multiplications, divisions, roots and powers of the scheme for a cell, one each."""
    cells = sum(a * b * c for a, b, c in _sizes(case))
    dims = 1 if cells == case["nx"] else 2 if case["nz"] == 1 else 3
    e = 4 if case["precision"] == "mixed" else 8
    per, ops = 12 * e, 190 * dims + 10
    if case["problem"] == "blob":
        per, ops = per + 8 * e, ops + 60
    elif case["problem"] == "jeans":
        per, ops = per + 9 * e + 8 + (e + 8), ops + 45 + 2 * 2.5 * math.log2(max(cells, 2))
    host = 0 if case["way"] == "noalloc" else 48 * cells
    if case["problem"] == "jeans":
        host += 8 * cells
    return {"bytes": per * cells * case["steps"] + host, "flops": ops * cells * case["steps"]}


# ---------------------------------------------------------------------------- the same in plain torch, 64 bits

def _f32(x):
    return float(np.float32(x))


def _constants(case, n):
    """The constants of the step as the parameter file's rules give them (single-precision literals held in doubles)."""
    g = _f32(5.0 / 3.0) if case["atomic"] else _f32(1.4)
    pi = _f32(3.1415927)
    return dict(g=g, g1=g - 1.0, dx=1.0 / max(n), grav=8.38553911e-7, c_cond=_f32(0.1),
                kappa0=0.5 * 4.6e13 * 1e-20 / _f32(_f32(37.8) / _f32(40.0)), kf2=[pi / m for m in n],
                de_thresh1=1.0 - 0.01 if case["problem"] == "cosmo" else None)


def _ghosts(w, axis, bt):
    """Two ghost layers along `axis` (0 x, 1 y, 2 z) of w[m][nz][ny][nx]; an axis of one cell has it as every ghost."""
    dim, n = 3 - axis, w.shape[3 - axis]
    if n == 1:
        return w
    idx = [-2, -1] + list(range(n)) + [n, n + 1]
    src = [i % n if bt == 2 else (-1 - i if i < 0 else 2 * n - 1 - i if i >= n else i) for i in idx]
    out = w.index_select(dim, torch.tensor(src, device=w.device))
    if bt == 3 and axis == 0 and w.shape[0] == 5:
        out[1:4, :, :, -2:] *= -1
    return out


def _cut(w, axis, lo, hi):
    """w without its first `lo` and last `hi` layers along `axis`."""
    dim = 3 - axis
    return w.narrow(dim, lo, w.shape[dim] - lo - hi)


def _primitive(q, c):
    r = 1.0 / q[0]
    w = torch.empty((5,) + tuple(q.shape[1:]), dtype=q.dtype, device=q.device)
    w[0] = q[0]
    w[1:4] = q[1:4] * r
    kin = 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0]
    p = c["g1"] * (q[4] - kin)
    if c["de_thresh1"] is not None:
        pg = q[0] ** c["g1"]
        by_entropy = kin / q[4] > c["de_thresh1"]
        p = torch.where(by_entropy, q[5] * pg, p)
        q[4] = torch.where(by_entropy, kin + p / c["g1"], q[4])
        q[5] = torch.where(by_entropy, q[5], p / pg)
    w[4] = p
    return w


def _slope(l, m, r, limiter):
    a, b = m - l, r - m
    if limiter == 3:
        ab = a * b
        return torch.where(ab > 0, 2 * ab / torch.where(ab > 0, a + b, 1.0), 0.0)
    lo, hi = torch.minimum(a, b), torch.maximum(a, b)
    if limiter == 2:
        mid = 0.5 * (r - l)
        lo, hi = torch.minimum(2 * lo, mid), torch.maximum(2 * hi, mid)
    return torch.maximum(lo, hi.clamp_max(0.0))


def _conserved(w, c):
    ke = 0.5 * w[0] * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3])
    return torch.stack([w[0], w[0] * w[1], w[0] * w[2], w[0] * w[3], ke + w[4] / c["g1"], w[4] / w[0] ** c["g1"]])


def _flux(w, q, d):
    f = q * w[d]
    f[d] += w[4]
    f[4] += w[d] * w[4]
    return f


def _riemann(l, r, d, case, c):
    al, ar = (c["g"] * l[4] / l[0]).sqrt(), (c["g"] * r[4] / r[0]).sqrt()
    sl = torch.minimum(l[d] - al, r[d] - ar)
    sr = torch.maximum(l[d] + al, r[d] + ar)
    if case["solver"] == 1:
        ql, qr = _conserved(l, c), _conserved(r, c)
        fl, fr = _flux(l, ql, d), _flux(r, qr, d)
        mid = (sr * fl - sl * fr + sl * sr * (qr - ql)) / (sr - sl)
        return torch.where(sl > 0, fl, torch.where(sr < 0, fr, mid))
    kl, kr = l[0] * (sl - l[d]), r[0] * (sr - r[d])
    sm = (r[4] - l[4] + kl * l[d] - kr * r[d]) / (kl - kr)
    right = (sr < 0) | ((sm <= 0) & (sl <= 0))
    star = (sl <= 0) & (sr >= 0)
    w = torch.where(right, r, l)
    s, k = torch.where(right, sr, sl), torch.where(right, kr, kl)
    q = _conserved(w, c)
    f = _flux(w, q, d)
    qs = torch.empty_like(q)
    qs[0] = k / (s - sm)
    for i in (1, 2, 3):
        qs[i] = qs[0] * (sm if i == d else w[i])
    qs[4] = qs[0] * (q[4] / w[0] + (sm - w[d]) * (sm + w[4] / k))
    qs[5] = qs[0] * q[5] / w[0]
    return torch.where(star, f + s * (qs - q), f)


def _sweep(q, w, dt, case, c):
    """q after the unsplit step of size dt from its primitives w (MUSCL-Hancock, x then y then z differences)."""
    axes = [a for a in (0, 1, 2) if q.shape[3 - a] > 1]
    for a in axes:
        w = _ghosts(w, a, case["boundtype"])
    mid = w
    for a in axes:
        mid = _cut(mid, a, 1, 1)
    s, evo = {}, torch.zeros_like(mid)
    for a in axes:
        v = w
        for b in axes:
            if b != a:
                v = _cut(v, b, 1, 1)
        s[a] = _slope(_cut(v, a, 0, 2), mid, _cut(v, a, 2, 0), case["limiter"])
        t = mid[a + 1] * s[a]
        t[4] += c["g"] * mid[4] * s[a][a + 1]
        t[a + 1] += s[a][4] / mid[0]
        evo += t / c["dx"]
    evo *= -0.5 * dt
    for a in axes:
        hi, lo = mid + 0.5 * s[a] + evo, mid - 0.5 * s[a] + evo
        for b in axes:
            if b != a:
                hi, lo = _cut(hi, b, 1, 1), _cut(lo, b, 1, 1)
        f = _riemann(_cut(hi, a, 0, 1), _cut(lo, a, 1, 0), a + 1, case, c)
        q = q + dt / c["dx"] * (_cut(f, a, 0, 1) - _cut(f, a, 1, 0))
    return q


def _potential(rho, c):
    nz, ny, nx = rho.shape
    src = torch.fft.fftn((c["grav"] * (rho - rho.mean())).to(torch.complex128))
    sin2 = []
    for m, kf2 in zip((nx, ny, nz), c["kf2"]):
        half = max(m // 2, 1)
        k = torch.tensor([i if i < half else i - m for i in range(m)], dtype=F64, device=rho.device)
        sin2.append(torch.sin(kf2 * k) ** 2)
    den = sin2[2][:, None, None] + sin2[1][None, :, None] + sin2[0][None, None, :]
    den[0, 0, 0] = 1.0
    green = -(c["dx"] ** 2 / 4.0) / den
    green[0, 0, 0] = 0.0
    return torch.fft.ifftn(src * green).real


def _evolve(q, case, n, steps):
    c = _constants(case, n)
    t, phi, dts = 0.0, None, []
    for _ in range(steps):
        w = _primitive(q, c)
        a = (c["g"] * w[4] / w[0]).sqrt()
        v = min(float((c["dx"] / (w[d + 1].abs() + a)).min()) for d in range(3))
        dt = case["cfl"] * min(v, 1e6)
        if case["problem"] == "blob":
            dt = min(dt, c["c_cond"] * c["dx"] ** 2 * float((w[0] / (c["kappa0"] * (w[4] / w[0]) ** 2.5)).min()))
        del a
        q = _sweep(q, w, dt, case, c)
        del w
        t += dt
        dts.append(dt)
        axes = [d for d in (0, 1, 2) if q.shape[3 - d] > 1]
        if case["problem"] == "jeans":
            phi = _potential(q[0], c)
            f = [-(phi.roll(-1, 2 - d) - phi.roll(1, 2 - d)) * (0.5 / c["dx"]) if d in axes else 0.0 * phi
                 for d in range(3)]
            q[4] += dt * (q[1] * f[0] + q[2] * f[1] + q[3] * f[2])
            for d in range(3):
                q[1 + d] += dt * q[0] * f[d]
        if case["problem"] == "blob":
            temp = _primitive(q, c)[4:5] / q[0]
            de = torch.zeros_like(q[0])
            for d in axes:
                g = _cut(_ghosts(temp, d, case["boundtype"]), d, 1, 1)
                m = temp[0]
                de += dt / c["g1"] / c["dx"] ** 2 * ((_cut(g, d, 2, 0)[0] - m) - (m - _cut(g, d, 0, 2)[0]))
            q[5] += c["g1"] * de / q[0] ** c["g1"]
            q[4] += de
    return q, t, dts, phi


def exact(case, seed):
    sizes = _sizes(case)
    cells = sum(a * b * c for a, b, c in sizes)
    if cells * case["steps"] > 1.2e9 or len(sizes) * case["steps"] > 1400:
        return None  # over about 20 seconds
    mixed = case["precision"] == "mixed"
    wide = lambda v: torch.as_tensor(v, dtype=F64)  # noqa: E731
    out, times, last, phi = [], [], [], None
    sums = []
    for q, n in zip(_boxes(case, seed), sizes):
        q = q.float().double() if mixed else q
        if case["way"] == "driver":
            t, left = 0.0, case["steps"]
            while left:
                m = min(10, left)
                q, dt, dts, phi = _evolve(q, case, n, m)
                t, left = t + dt, left - m
                if m == 10:
                    sums.append([float(q[i].sum()) for i in (0, 4, 5)])
        else:
            q, t, dts, phi = _evolve(q, case, n, case["steps"])
        out.append(q)
        times.append(t)
        last.append(dts[-1])
    if case["way"] == "run":
        got = dict(q=torch.from_numpy(_host(out[0])), t=wide(times[0]), dt=wide(last[0]), done=None)
        if phi is not None:
            got["phi"] = phi.cpu()
        return got
    if case["way"] == "driver":
        return dict(q=torch.from_numpy(_host(out[0])), t=wide(times[0]), sums=wide(sums))
    if case["way"] == "batch":
        return dict(q=torch.cat([torch.from_numpy(_host(q)).reshape(-1) for q in out]), t=np.array(times),
                    dt=np.array(last))
    return dict(q=torch.cat([q.reshape(-1) for q in out]), t=np.array(times))
