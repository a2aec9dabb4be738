"""The measured work of the framework: reconstructions and the operators they
are made of, over the sizes that a user of the library meets.

Sizes come from the workloads of bench.py and its tests: slices of 128 to 1024
pixels from 90 to 720 angles (a batch of uneven slices is the flagship), 3-D
laminography volumes of 8 to 32 slices up to 511^2 and, padded as the 3-D
driver pads them, 29 x 721^2.  Operators are called through the C ABI on device
buffers, solvers through a resident Batch2D, the whole-solve driver and the
server on host arrays, as their callers do.

Solves run fewer iterations than a reconstruction does (5 to 20 instead of 20
to 100): an iteration costs the same throughout, and after five to ten CG
iterations rounding alone begins to move an under-sampled solution, so longer
solves could not be compared with anything.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

import laminocam_amd as lc
from laminocam_amd import _lib

DEV = "cuda"
PI = math.pi
TILT = -PI / 6          # laminography tilt of every 3-D case
N_SET = (128, 192, 256, 384, 512, 768, 1024)
ANG_SET = (90, 180, 360, 720)
EXACT_FLOPS = 2e14      # direct sums above this take too long in 64 bits


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one Toeplitz apply of a small slice: an opaque solver's inner call, all latency
        dict(name="apply2d_1x128", kind="apply2d", ns=1, n=128, nang=90, f64=False),
        # projecting an odd-sized stack on an odd detector (odd sizes are what the padding makes)
        dict(name="forward2d_4x511", kind="forward2d", ns=4, n=511, nang=360, nrad=511),
        # the right-hand side of a stack of the largest slices
        dict(name="backproj2d_8x1024", kind="backproj2d", ns=8, n=1024, nang=720, nrad=1024),
        # the flagship: 512 independent uneven slices solved together
        dict(name="batch_cg2d_512", kind="batch", solver="cg", slices=512, classes=28, n_min=128,
             n_max=1024, ragged=False, f64=False, iters=5, pick=4),
        # the same with TV regularisation, a smaller batch
        dict(name="batch_sb2d_64", kind="batch", solver="sb", slices=64, classes=12, n_min=128,
             n_max=1024, ragged=False, f64=False, iters=8, pick=5),
        # and in double precision, for solves that have to stay close to a 64-bit reference
        dict(name="batch_cg2d_f64_64", kind="batch", solver="cg", slices=64, classes=12, n_min=128,
             n_max=768, ragged=False, f64=True, iters=8, pick=6),
        # requests that arrive together at the server, sinograms in, solutions out (host arrays)
        dict(name="serve_2d_64", kind="serve", slices=64, classes=12, n_min=128, n_max=512,
             ragged=False, iters=5, pick=7),
        # projecting the padded laminography volume
        dict(name="forward3d_29x721", kind="forward3d", n1=29, n=721, nproj=360, nrows=89),
        # back-projection of a small and of a large scan
        dict(name="backproj3d_8x256", kind="backproj3d", n1=8, n=256, nproj=180, nrows=64),
        dict(name="backproj3d_32x511", kind="backproj3d", n1=32, n=511, nproj=720, nrows=128),
        # the laminography solve: CG on the padded volume
        dict(name="lamino_cg_29x721", kind="solve3d", solver="cg", n1=29, n=721, nproj=360,
             nrows=89, iters=10),
        # the whole laminography reconstruction on host arrays: padding, geometry, PSF,
        # back-projection, Split-Bregman, crop
        dict(name="mbir3d_21x511", kind="mbir3d", solver="sb", n1=21, n=511, nproj=360, nrows=64,
             iters=20),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["apply2d", "forward2d", "backproj2d", "batch", "batch", "serve", "forward3d",
                       "backproj3d", "solve3d", "mbir3d"])
    if kind in ("apply2d", "forward2d", "backproj2d"):
        n = _logint(rng, 64, 1024)
        ns = _logint(rng, 1, max(1, min(32, 8 * 1024 * 1024 // (n * n))))
        c = dict(kind=kind, ns=ns, n=n, nang=_logint(rng, 60, 720))
        if kind == "apply2d":
            return dict(c, f64=rng.random() < 0.3)
        return dict(c, nrad=rng.choice([n, n, n | 1, _logint(rng, max(64, n // 2), min(1024, 2 * n))]))
    if kind in ("batch", "serve"):
        f64 = kind == "batch" and rng.random() < 0.3
        n_max = rng.choice([128, 256, 512, 1024]) if kind == "batch" else rng.choice([128, 256, 512])
        top = min(512, int(24e6) // (n_max * n_max) + 1) // (4 if f64 else 1)
        c = dict(kind=kind, slices=_logint(rng, 1, max(2, min(64, top) if kind == "serve" else top)),
                 classes=rng.randint(1, 8), n_min=min(n_max, rng.choice([64, 128])), n_max=n_max,
                 ragged=rng.random() < 0.4, iters=rng.randint(3, 5), pick=rng.randrange(1 << 20))
        return c if kind == "serve" else dict(c, solver=rng.choice(["cg", "sb"]), f64=f64)
    n = _logint(rng, 64, 511)
    n1 = _logint(rng, 5, 32)
    c = dict(kind=kind, n1=n1, n=n, nproj=_logint(rng, 60, 720), nrows=rng.randint(n1, 4 * n1))
    if kind == "solve3d":
        return dict(c, solver=rng.choice(["cg", "sb"]), nproj=min(c["nproj"], 360), iters=rng.randint(4, 10))
    if kind == "mbir3d":
        n = _logint(rng, 64, 400) | 1
        return dict(c, solver=rng.choice(["cg", "sb"]), n=n, n1=_logint(rng, 5, 21) | 1,
                    nproj=min(c["nproj"], 360), nrows=c["nrows"] + (c["nrows"] & 1), iters=rng.randint(4, 12))
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _angles(nang, span=PI):
    return np.arange(nang, dtype=np.float64) * (span / nang)


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _noise(shape, seed, salt):
    return torch.randn(shape, generator=_gen(seed, salt), device=DEV, dtype=torch.float32)


def _ellipses(rs, n, k):
    """n phantoms of k ellipses: centre (cx, cy), semi-axes (a, b), rotation, value"""
    return (rs.uniform(-0.5, 0.5, (n, k)), rs.uniform(-0.5, 0.5, (n, k)), rs.uniform(0.05, 0.4, (n, k)),
            rs.uniform(0.05, 0.4, (n, k)), rs.uniform(0.0, PI, (n, k)), rs.uniform(0.0, 1.0, (n, k)))


def _phantoms2d(n, N, rs, k=10):
    """n random-ellipse slices of N x N on [-1, 1]^2"""
    ax = (torch.arange(N, device=DEV, dtype=torch.float32) + 0.5) * (2.0 / N) - 1.0
    out = torch.zeros((n, N, N), device=DEV)
    cols = [torch.as_tensor(p, device=DEV, dtype=torch.float32)[:, :, None, None] for p in _ellipses(rs, n, k)]
    for j in range(k):
        cx, cy, a, b, ph, v = (p[:, j] for p in cols)
        dx, dy = ax[None, None, :] - cx, ax[None, :, None] - cy
        xr, yr = dx * torch.cos(ph) + dy * torch.sin(ph), dy * torch.cos(ph) - dx * torch.sin(ph)
        out += v * ((xr / a) ** 2 + (yr / b) ** 2 <= 1.0)
    return out


def _sinograms2d(n, nang, nrad, seed, salt, k=10):
    """n noisy sinograms {nang, nrad} of random-ellipse phantoms (closed-form
    parallel projections, 1% noise), each divided by its maximum"""
    rs = np.random.default_rng((seed, salt))
    s = (torch.arange(nrad, device=DEV, dtype=torch.float32) + 0.5) * (2.0 / nrad) - 1.0
    th = torch.as_tensor(_angles(nang), device=DEV, dtype=torch.float32)[None, :, None]
    out = torch.zeros((n, nang, nrad), device=DEV)
    cols = [torch.as_tensor(p, device=DEV, dtype=torch.float32)[:, :, None, None] for p in _ellipses(rs, n, k)]
    for j in range(k):
        cx, cy, a, b, ph, v = (p[:, j] for p in cols)
        w2 = (a * torch.cos(th - ph)) ** 2 + (b * torch.sin(th - ph)) ** 2
        d = s - (cx * torch.cos(th) + cy * torch.sin(th))
        out += 2.0 * v * a * b * torch.sqrt(torch.clamp(w2 - d * d, min=0.0)) / w2
    out += 0.01 * out.amax(dim=(1, 2), keepdim=True) * _noise(out.shape, seed, salt + 1)
    return out / out.amax(dim=(1, 2), keepdim=True)


def _rot(theta, tilt=TILT):
    """columns 0 and 1 of the rotation of each projection (beta = 0): the
    detector's column and row directions as (x, y, z)"""
    ct, st, cg, sg = np.cos(theta), np.sin(theta), np.cos(tilt), np.sin(tilt)
    z = np.zeros_like(theta)
    u = np.stack([np.full_like(theta, cg), np.full_like(theta, -sg), z], 1)
    v = np.stack([ct * sg, ct * cg, -st], 1)
    return u, v


def _projections3d(n1, n, nproj, nrows, ncols, seed, k=12):
    """noisy projections {nproj, nrows, ncols} of a random-ellipsoid volume
    (closed form, 1% noise), divided by their maximum"""
    rs = np.random.default_rng((seed, 31))
    u, v = _rot(_angles(nproj, 2 * PI))
    half = np.array([n / 2.0, n / 2.0, n1 / 2.0])
    ctr = rs.uniform(-0.5, 0.5, (k, 3)) * half
    sem = rs.uniform(0.05, 0.4, (k, 3)) * half + 0.5
    val = rs.uniform(0.0, 1.0, k)
    cols = torch.arange(ncols, device=DEV, dtype=torch.float32) - (ncols - 1) / 2.0
    rows = torch.arange(nrows, device=DEV, dtype=torch.float32) - (nrows - 1) / 2.0
    out = torch.zeros((nproj, nrows, ncols), device=DEV)
    t = lambda a: torch.as_tensor(a, device=DEV, dtype=torch.float32)[:, None, None]
    for j in range(k):
        A = sem[j] ** 2
        suu, svv, suv = (u * u) @ A, (v * v) @ A, (u * v) @ A
        det = suu * svv - suv * suv
        dx = cols[None, None, :] - t(u @ ctr[j])
        dy = rows[None, :, None] - t(v @ ctr[j])
        q = (t(svv) * dx * dx - 2.0 * t(suv) * dx * dy + t(suu) * dy * dy) / t(det)
        out += t(2.0 * val[j] * np.prod(sem[j]) / np.sqrt(det)) * torch.sqrt(torch.clamp(1.0 - q, min=0.0))
    out += 0.01 * out.max() * _noise(out.shape, seed, 32)
    return out / out.max()


def _pow2(n):
    """transform sizes of the models here: few distinct plans"""
    return 1 << (n - 1).bit_length()


def _kaxis(m):
    return torch.fft.fftfreq(m, device=DEV, dtype=torch.float32) * (2 * PI)


def _rhs2d(n, N, nang, seed, salt):
    """right-hand sides of n slices: A^T A of a phantom with 1% of noise whose
    spectrum rises as the detector noise of a reconstruction does"""
    rs = np.random.default_rng((seed, salt))
    x = _phantoms2d(n, N, rs) / (N / 2.0)
    L = _pow2(N)
    k = torch.sqrt(_kaxis(L)[:, None] ** 2 + _kaxis(L)[None, :L // 2 + 1] ** 2)
    f = torch.fft.rfft2(_noise((n, L, L), seed, salt + 1)) * torch.sqrt(k)
    x += torch.fft.irfft2(f, s=(L, L))[:, :N, :N] * (0.01 / N)
    A = _toeplitz2d(N, nang, N)
    return torch.cat([A(x[i:i + 8].double()) for i in range(0, n, 8)])


def _rhs3d(n1, N, nproj, nrows, seed):
    """right-hand side of a 3-D volume, with A^T A modelled by its spectrum:
    every detector plane holds the (fixed) column direction u, so the samples
    are uniform along u and as dense as 1 / |k_perp| across it"""
    rs = np.random.default_rng((seed, 41))
    zz = (torch.arange(n1, device=DEV, dtype=torch.float32) + 0.5) * (2.0 / n1) - 1.0
    x = _phantoms2d(3, N, rs, 4)
    x = (x[0][None] * torch.exp(-4.0 * (zz - 0.2) ** 2)[:, None, None] + x[1][None] * (zz < 0)[:, None, None] +
         x[2][None] * (zz.abs() < 0.3)[:, None, None]) / (N / 2.0)
    s = (_pow2(2 * n1), _pow2(2 * N), _pow2(2 * N))
    kz, ky, kx = _kaxis(s[0])[:, None, None], _kaxis(s[1])[None, :, None], _kaxis(s[1])[None, None, :s[1] // 2 + 1].abs()
    cg, sg = math.cos(TILT), math.sin(TILT)
    par, perp = kx * cg - ky * sg, torch.sqrt(kz ** 2 + (kx * sg + ky * cg) ** 2)
    w = torch.where((par.abs() <= PI) & (perp <= PI), 2.0 * nproj * nrows / N / torch.clamp(perp, min=PI / nrows),
                    torch.zeros_like(perp))
    f = torch.fft.rfftn(x, s=s) * w
    f += 0.01 / N * torch.fft.rfftn(_noise((n1, N, N), seed, 42), s=s) * torch.sqrt(w)
    return torch.fft.irfftn(f, s=s)[:n1, :N, :N].contiguous()


def _problems(case):
    """the (N, angles) of every problem of a batch, in order: `classes` distinct
    pairs, each slice one of them; part of the plan, not of the inputs"""
    rs = np.random.default_rng(case["pick"])
    if case["ragged"]:
        lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
        pairs = [(int(round(math.exp(rs.uniform(lo, hi)))), int(rs.integers(60, 721)))
                 for _ in range(case["classes"])]
    else:
        ns = [v for v in N_SET if case["n_min"] <= v <= case["n_max"]]
        every = [(v, a) for v in ns for a in ANG_SET]
        pairs = [every[i] for i in rs.permutation(len(every))[:case["classes"]]]
    return sorted(pairs[i] for i in rs.integers(0, len(pairs), case["slices"]))


def _groups(probs):
    """(N, angles) -> its run of problems"""
    g = {}
    for i, key in enumerate(probs):
        g.setdefault(key, []).append(i)
    return sorted(g.items())


def _batch_rhs(case, seed):
    """per class: (N, angles), its problems, their right-hand sides in 64 bits
    (rounded to 32 for a 32-bit batch)"""
    out = []
    for j, ((N, nang), idx) in enumerate(_groups(_problems(case))):
        y = _rhs2d(len(idx), N, nang, seed, 100 + 10 * j)
        out.append(((N, nang), idx, y if case["f64"] else y.float().double()))
    return out


def _serve_inputs(case, seed):
    """sinograms and solver of every request (70% CG, 30% Split-Bregman)"""
    probs = _problems(case)
    sino = [None] * len(probs)
    for j, ((N, nang), idx) in enumerate(_groups(probs)):
        s = _sinograms2d(len(idx), nang, N, seed, 200 + 10 * j).cpu().numpy()
        for q, i in enumerate(idx):
            sino[i] = s[q:q + 1]
    rs = np.random.default_rng(case["pick"] + 1)
    sb = rs.uniform(size=len(probs)) < 0.3
    lam = rs.uniform(0.05, 0.2, len(probs))
    return probs, sino, sb, lam


def _volume3d(case, seed):
    rs = np.random.default_rng((seed, 51))
    p = _phantoms2d(3, case["n"], rs, 6)
    zz = (torch.arange(case["n1"], device=DEV, dtype=torch.float32) + 0.5) * (2.0 / case["n1"]) - 1.0
    vol = p[0][None] * torch.exp(-4.0 * zz ** 2)[:, None, None] + p[1][None] * (zz > 0)[:, None, None]
    return (vol + p[2][None] * (zz.abs() < 0.4)[:, None, None]).contiguous()


# ---------------------------------------------------------------------------
# state and pass
# ---------------------------------------------------------------------------
class _View:
    """a run of problems of a batch in the library's device memory, as torch can read it"""

    def __init__(self, batch, idx, which):
        self.batch = batch
        p0 = batch.device_ptr(idx[0], which)
        e = np.dtype(batch.dtype).itemsize
        n1, N, _ = shape = batch.shape(idx[0])
        step = batch.device_ptr(idx[1], which) - p0 if len(idx) > 1 else e * N * N
        assert len(idx) == 1 or all(batch.device_ptr(i, which) == p0 + j * step for j, i in enumerate(idx))
        if len(idx) > 1:
            shape = (len(idx), N, N)
        self.__cuda_array_interface__ = dict(shape=shape, typestr=np.dtype(batch.dtype).str, data=(p0, False),
                                             version=2, strides=(step, e * N, e))


def _view(batch, idx, which):
    return torch.as_tensor(_View(batch, idx, which), device=DEV)


def _dptr(t):
    return C.c_void_p(t.data_ptr())


def _grid3(case):
    return lc.PolarGrid(_angles(case["nproj"], 2 * PI), np.full(case["nproj"], TILT),
                        np.zeros(case["nproj"]), case["nrows"], case["n"])


def _resident(psfs, rhs, f64):
    """a batch with its right-hand sides set, and views of its solutions;
    rhs: (problems, their right-hand sides) per class"""
    b = lc.Batch2D(psfs, fp64=f64)
    for idx, y in rhs:
        _view(b, idx, b.Y).copy_(y)
    return b, [_view(b, idx, b.X) for idx, _ in rhs]


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("apply2d", "forward2d", "backproj2d"):
        ns, N, nang = case["ns"], case["n"], case["nang"]
        nrad = case.get("nrad", N)
        grid = lc.PolarGrid2D(_angles(nang), nrad)
        s["psf"] = lc.PointSpreadFunction2D(grid, N) if kind == "apply2d" else grid._geometry(N)
        if kind == "backproj2d":
            s["in"] = _sinograms2d(ns, nang, nrad, seed, 3)
            s["out"] = torch.empty((ns, N, N), device=DEV)
        else:
            s["in"] = _phantoms2d(ns, N, np.random.default_rng((seed, 5)))
            if case.get("f64"):
                s["in"] = s["in"].double()
            s["out"] = torch.empty((ns, nang, nrad), device=DEV) if kind == "forward2d" else torch.empty_like(s["in"])
    elif kind == "batch":
        rhs = _batch_rhs(case, seed)
        geo = {k: lc.PointSpreadFunction2D(lc.PolarGrid2D(_angles(k[1]), k[0]), k[0]) for k, _, _ in rhs}
        s["batch"], s["out"] = _resident([geo[k] for k in _problems(case)], [r[1:] for r in rhs], case["f64"])
    elif kind == "serve":
        probs, sino, sb, lam = _serve_inputs(case, seed)
        geo = {k: lc.PointSpreadFunction2D(lc.PolarGrid2D(_angles(k[1]), k[0]), k[0]) for k, _ in _groups(probs)}
        s["req"] = [(geo[k], sino[i], dict(solver="sb", lam=float(lam[i]), mu=10.0, outer=case["iters"], inner=1,
                                           zero_pad=True) if sb[i] else dict(solver="cg", max_iter=case["iters"]))
                    for i, k in enumerate(probs)]
        s["server"] = lc.Server(hbm_budget=64 << 30, lanes=4)
    elif kind == "forward3d":
        s["psf"] = lc.PointSpreadFunction(_grid3(case), (case["n1"], case["n"], case["n"]), lazy=True)
        s["in"] = _volume3d(case, seed)
        s["out"] = torch.empty((case["nproj"], case["nrows"], case["n"]), device=DEV)
    elif kind == "backproj3d":
        s["psf"] = lc.PointSpreadFunction(_grid3(case), (case["n1"], case["n"], case["n"]), lazy=True)
        s["in"] = _projections3d(case["n1"], case["n"], case["nproj"], case["nrows"], case["n"], seed)
        s["out"] = torch.empty((case["n1"], case["n"], case["n"]), device=DEV)
    elif kind == "solve3d":
        psf = lc.PointSpreadFunction(_grid3(case), (case["n1"], case["n"], case["n"]))
        s["batch"], s["out"] = _resident([psf], [([0], _rhs3d(case["n1"], case["n"], case["nproj"], case["nrows"], seed))],
                                          False)
    else:
        p = _projections3d(case["n1"], case["n"], case["nproj"], case["nrows"], case["n"], seed).cpu().numpy()
        s["data"] = [lc.Dataset(projs=p, angles=_angles(case["nproj"], 2 * PI), gamma=TILT)]
        reg = lc.Regularizer.SPLIT_BREGMAN if case["solver"] == "sb" else lc.Regularizer.UNCONSTRAINED
        s["par"] = lc.ReconParams(regularizer=reg, recon_dims=(case["n1"], case["n"], case["n"]),
                                  maxIters=case["iters"], tol=0.0, xtol=0.0)
    torch.cuda.synchronize()   # the library works on streams of its own
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("apply2d", "forward2d", "backproj2d"):
        p = s["psf"]
        lib = p.ctx.lib
        fn = dict(apply2d=lib.lc_sysmat2d_psf_f64 if case.get("f64") else lib.lc_sysmat2d_psf,
                  forward2d=lib.lc_forward2d, backproj2d=lib.lc_backproj2d)[kind]
        _lib.check(fn(p.ctx.handle, p.handle, _dptr(s["in"]), case["ns"], _dptr(s["out"]), _lib.LC_DEVICE_PTRS))
        return s["out"]
    if kind == "forward3d":
        p = s["psf"]
        _lib.check(p.lib.lc_forward3d(p.ctx.handle, p.handle, _dptr(s["in"]), _dptr(s["out"]), _lib.LC_DEVICE_PTRS))
        return s["out"]
    if kind == "backproj3d":
        p = s["psf"]
        _lib.check(p.lib.lc_backproj3d(p.ctx.handle, p.handle, _dptr(s["in"]), None, _dptr(s["out"]),
                                       _lib.LC_DEVICE_PTRS))
        return s["out"]
    if kind in ("batch", "solve3d"):
        b = s["batch"]
        if case["solver"] == "cg":
            b.cg(case["iters"], 1e-5, 1e-5)
        else:
            b.split_bregman(0.1, 10.0, case["iters"], 1, 1e-5, 1e-5, zero_pad=kind == "batch", x0_zero=True)
        return s["out"]
    if kind == "serve":
        srv = s["server"]
        tickets = [srv.submit(psf, sino=sino, borrow=True, **kw) for psf, sino, kw in s["req"]]
        return [srv.result(t, timeout=60.0)[0] for t in tickets]
    return lc.MBIR(s["data"], s["par"], graph=True)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _fft_flops(*dims):
    m = math.prod(dims)
    return 2.5 * m * math.log2(m)   # a real transform of m points


def _pad_size(n, f=np.float32(1.4142)):
    m = int(np.float32(n) * f)
    return m - 1 if m % 2 == 0 else m


def _solve_work(n1, N, iters, b, sb, vol):
    """n1 slices (vol: one volume) of N^2 elements of b bytes.  Per iteration x,
    r and p are read and written once (Split-Bregman: d and b, three components
    each, too) and A p is two transforms of the doubled size; the spectrum is
    read once per iteration (a batch counts it apart: its slices share it)"""
    n = n1 * N * N
    fft = _fft_flops(2 * n1, 2 * N, 2 * N) if vol else n1 * _fft_flops(2 * N, 2 * N)
    per = (6 + (12 if sb else 0)) * n + (4 * n if vol else 0)
    return b * (iters * per + 2 * n), iters * (2 * fft + 20 * n)


def _nufft_work(npts, dims):
    """eight cells per axis and point, and the transform of the doubled grid"""
    return 4.0 * npts * 8 ** len(dims) + 2 * _fft_flops(*(2 * d for d in dims))


def work(case):
    kind, n = case["kind"], case.get("n")
    if kind == "apply2d":
        b = 8 if case["f64"] else 4
        return {"bytes": b * (2 * case["ns"] * n * n + 2 * n * n), "flops": 2 * case["ns"] * _fft_flops(2 * n, 2 * n)}
    if kind in ("forward2d", "backproj2d"):
        npts = case["nang"] * case["nrad"]
        return {"bytes": 4 * case["ns"] * (n * n + npts), "flops": case["ns"] * _nufft_work(npts, (n, n))}
    if kind in ("forward3d", "backproj3d"):
        npts = case["nproj"] * case["nrows"] * n
        return {"bytes": 4 * (case["n1"] * n * n + npts), "flops": _nufft_work(npts, (case["n1"], n, n))}
    if kind == "solve3d":
        by, fl = _solve_work(case["n1"], n, case["iters"], 4, case["solver"] == "sb", True)
        return {"bytes": by, "flops": fl}
    if kind == "mbir3d":
        n1p, npad, nr = _pad_size(case["n1"]), _pad_size(n), _pad_size(case["nrows"])
        by, fl = _solve_work(n1p, npad, case["iters"], 4, case["solver"] == "sb", True)
        pts = case["nproj"] * nr * npad
        host = 4 * (case["nproj"] * case["nrows"] * n + case["n1"] * n * n)
        return {"bytes": by + 8 * pts + host,
                "flops": fl + _nufft_work(pts, (n1p, npad, npad)) + 40.0 * case["nproj"] * n1p * 2 * npad * npad}
    b = 8 if case.get("f64") else 4
    by = fl = 0
    probs = _problems(case)
    for N, nang in probs:
        q, w = _solve_work(1, N, case["iters"], b, case.get("solver") == "sb", False)
        by, fl = by + q, fl + w
        if kind == "serve":
            by, fl = by + 4 * nang * N, fl + _nufft_work(nang * N, (N, N))
    by += sum(2 * N * N * b * case["iters"] for (N, _), _ in _groups(probs))
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """about four times what each kind of case shows against exact().  A
    back-projection of many projections onto a small volume adds thousands of
    32-bit terms to the cells around the k-space centre"""
    kind = case["kind"]
    if kind == "apply2d":
        return {"rel": 5e-15 if case["f64"] else 7e-7}
    if kind in ("forward2d", "backproj2d", "forward3d"):
        return {"rel": 3.5e-6}
    if kind in ("backproj3d", "mbir3d"):
        return {"rel": 2.5e-5}
    return {"rel": 1e-10 if case.get("f64") else 1e-5}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
F64 = torch.float64


def _roll(a, d, axis):
    """out[k] = a[(k + d) mod n]"""
    return torch.roll(a, -d, axis)


def _shift(a, axes):
    for ax in axes:
        a = _roll(a, a.shape[ax] // 2, ax)
    return a


def _ishift(a, axes):
    for ax in axes:
        a = _roll(a, a.shape[ax] // 2 + a.shape[ax] % 2, ax)
    return a


def _lattice(n):
    return (torch.arange(n, device=DEV, dtype=F64) + 0.5) * (2 * PI / n) - PI


def _modes(n):
    return torch.arange(n, device=DEV, dtype=F64) - n // 2


def _cis(ph):
    return torch.cos(ph), torch.sin(ph)


def _exact_backproj(c, pts, dims, chunk):
    """Re sum_p c_p exp(i m.w_p) for every slice of c {ns, npts}; pts: (x, y, z or None)"""
    n1, n2, n3 = dims
    ns, npts = c.shape
    out = torch.zeros((ns, n1 * n2, n3), device=DEV, dtype=F64)
    for a in range(0, npts, chunk):
        q = slice(a, min(npts, a + chunk))
        er, ei = _cis(pts[0][q, None] * _modes(n3))
        yr, yi = _cis(pts[1][q, None] * _modes(n2))
        left = torch.complex(yr, yi)
        if pts[2] is not None:
            left = (torch.complex(*_cis(pts[2][q, None] * _modes(n1)))[:, :, None] * left[:, None, :]).reshape(-1, n1 * n2)
        for s in range(ns):
            w = left * c[s, q, None]
            out[s] += w.real.T @ er - w.imag.T @ ei
    return out.reshape(ns * n1, n2, n3)


def _exact_project(vol, pts, chunk):
    """sum_m f_m exp(-i m.w_p) of the slices vol {ns, n1, n2, n3}"""
    ns, n1, n2, n3 = vol.shape
    npts = pts[0].numel()
    out = torch.empty((ns, npts), device=DEV, dtype=torch.complex128)
    for a in range(0, npts, chunk):
        q = slice(a, min(npts, a + chunk))
        er, ei = _cis(pts[0][q, None] * _modes(n3))
        ey = torch.complex(*_cis(-pts[1][q, None] * _modes(n2)))
        for s in range(ns):
            v = vol[s].reshape(n1 * n2, n3).T
            t = torch.complex(er @ v, -(ei @ v)).reshape(-1, n1, n2)
            t = (t * ey[:, None, :]).sum(-1)
            if pts[2] is not None:
                t = t * torch.complex(*_cis(-pts[2][q, None] * _modes(n1)))
            out[s, q] = t.sum(-1)
    return out


def _points2d(nang, nrad):
    th = torch.as_tensor(_angles(nang), device=DEV)
    r = _lattice(nrad)
    return (torch.cos(th)[:, None] * r).reshape(-1), (torch.sin(th)[:, None] * r).reshape(-1), None


def _points3d(nproj, nrows, ncols):
    u, v = (torch.as_tensor(a, device=DEV) for a in _rot(_angles(nproj, 2 * PI)))
    qx, qy = _lattice(ncols)[None, None, :], _lattice(nrows)[None, :, None]
    p = [(u[:, a, None, None] * qx + v[:, a, None, None] * qy).reshape(-1) for a in range(3)]
    w = (p[0].abs() <= PI) & (p[1].abs() <= PI) & (p[2].abs() <= PI)
    return p, w.double()


def _exact_rhs2d(sino, N):
    ns, nang, nrad = sino.shape
    c = _ishift(torch.fft.fft(_shift(sino.to(torch.complex128), [-1]), dim=-1), [-1])
    return _exact_backproj(c.reshape(ns, -1), _points2d(nang, nrad), (1, N, N), 1 << 16) / nrad


def _exact_rhs3d(proj, dims):
    nproj, nrows, ncols = proj.shape
    c = _ishift(torch.fft.fft2(_shift(proj.to(torch.complex128), [-1, -2])), [-1, -2])
    pts, w = _points3d(nproj, nrows, ncols)
    chunk = max(64, (1 << 28) // (dims[0] * dims[1]))
    return _exact_backproj((c.reshape(1, -1) * w), pts, dims, chunk) / (nrows * ncols)


def _dirichlet(t, n):
    """sin(pi t) / sin(pi t / n)"""
    k = torch.round(t / n)
    d = t - k * n
    num = torch.sin(PI * (d - 2.0 * torch.round(d / 2.0)))
    den = torch.sin(d * (PI / n))
    r = torch.where(d == 0, torch.full_like(d, float(n)), num / torch.where(d == 0, torch.ones_like(d), den))
    return r if n % 2 else r * (1.0 - 2.0 * torch.remainder(k, 2.0))


def _toeplitz(us, ns, n1, N):
    """A^T A of N x N slices (n1 == 1) or an {n1, N, N} volume as a function;
    us: per lattice direction the vectors {count, 3} as (x, y, z), ns: its points"""
    mz = torch.arange(n1, device=DEV, dtype=F64)[:, None, None]
    m = torch.arange(-(N - 1), N, device=DEV, dtype=F64)
    P = torch.zeros((n1, 2 * N - 1, 2 * N - 1), device=DEV, dtype=F64)
    for i in range(len(us[0])):
        term = None
        for u, n in zip(us, ns):
            x, y, z = (float(a) for a in u[i])
            d = _dirichlet(mz * z + m[None, :, None] * y + m[None, None, :] * x, n)
            term = d if term is None else term * d
        P += term
    L, L1 = _pow2(2 * N), _pow2(2 * n1) if n1 > 1 else 1
    full = torch.zeros((L1, L, L), device=DEV, dtype=F64)
    idx = torch.remainder(m.long(), L)
    for z in range(n1):
        full[z][idx[:, None], idx[None, :]] = P[z]
        if z:
            full[L1 - z][idx[:, None], idx[None, :]] = P[z].flip(0, 1)
    K = torch.fft.rfftn(full) / float(N ** len(us))

    def apply(x):
        if n1 == 1:
            return torch.fft.irfft2(torch.fft.rfft2(x, s=(L, L)) * K, s=(L, L))[:, :N, :N]
        return torch.fft.irfftn(torch.fft.rfftn(x, s=(L1, L, L)) * K, s=(L1, L, L))[:n1, :N, :N]
    return apply


@functools.lru_cache(maxsize=48)
def _toeplitz2d(N, nang, nrad):
    th = _angles(nang)
    return _toeplitz([np.stack([np.cos(th), np.sin(th), np.zeros_like(th)], 1)], [nrad], 1, N)


def _toeplitz3d(nproj, nrows, ncols, n1, N):
    u, v = _rot(_angles(nproj, 2 * PI))
    return _toeplitz([u, v], [ncols, nrows], n1, N)


def _exact_cg(A, y, x, iters):
    r = y - A(x)
    p, rs = r, (r * r).sum()
    for _ in range(iters):
        Ap = A(p)
        al = rs / (p * Ap).sum()
        x, r = x + al * p, r - al * Ap
        rn = (r * r).sum()
        p, rs = r + rn / rs * p, rn
    return x


def _diff(u, axis, zero_pad):
    n = u.shape[axis]
    a = torch.zeros_like(u)
    if n > 1:
        a.narrow(axis, 0, n - 1).add_(u.narrow(axis, 1, n - 1))
        a.narrow(axis, 1, n - 1).sub_(u.narrow(axis, 0, n - 1))
    a *= 0.5
    if not zero_pad:
        keep = torch.zeros_like(u)
        keep[1:-1, 1:-1, 1:-1] = 1.0
        a *= keep
    return a


def _exact_sb(A, y, lam, mu, outer, zero_pad):
    grad = lambda u: [_diff(u, a, zero_pad) for a in range(3)]
    div = lambda g: sum(_diff(g[a], a, zero_pad) for a in range(3))
    op = lambda u: A(u) - mu * div(grad(u))
    x = torch.zeros_like(y)
    d, b = [torch.zeros_like(y) for _ in range(3)], [torch.zeros_like(y) for _ in range(3)]
    for _ in range(outer):
        x = _exact_cg(op, y - mu * div([p - q for p, q in zip(d, b)]), x, 1)
        g = grad(x)
        v = [p + q for p, q in zip(g, b)]
        sk = torch.sqrt(sum(q * q for q in v))
        sh = torch.clamp(sk - float(np.float32(lam) / np.float32(mu)), min=0.0) / (sk + 1e-8)
        d = [sh * q for q in v]
        b = [q - p for q, p in zip(v, d)]
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "apply2d":
        x = _phantoms2d(case["ns"], case["n"], np.random.default_rng((seed, 5))).double()
        return _toeplitz2d(case["n"], case["nang"], case["n"])(x)
    if kind == "forward2d":
        x = _phantoms2d(case["ns"], case["n"], np.random.default_rng((seed, 5))).double()
        c = _exact_project(x[:, None], _points2d(case["nang"], case["nrad"]), 1 << 16)
        c = _ishift(c.reshape(case["ns"], case["nang"], case["nrad"]), [-1])
        return _shift(torch.fft.ifft(c, dim=-1), [-1]).real.contiguous()
    if kind == "backproj2d":
        return _exact_rhs2d(_sinograms2d(case["ns"], case["nang"], case["nrad"], seed, 3).double(), case["n"])
    if kind in ("forward3d", "backproj3d"):
        n1, n, nproj, nrows = case["n1"], case["n"], case["nproj"], case["nrows"]
        if 4.0 * nproj * nrows * n * n * n * n1 > EXACT_FLOPS:
            return None
        if kind == "backproj3d":
            return _exact_rhs3d(_projections3d(n1, n, nproj, nrows, n, seed).double(), (n1, n, n))
        pts, w = _points3d(nproj, nrows, n)
        c = _exact_project(_volume3d(case, seed).double()[None], pts, max(64, (1 << 28) // (n1 * n)))
        c = _shift((c * w).reshape(nproj, nrows, n), [-1, -2])
        return _ishift(torch.fft.ifft2(c), [-1, -2]).real.contiguous()
    if kind == "batch":
        out = []
        for (N, nang), idx, y in _batch_rhs(case, seed):
            A = _toeplitz2d(N, nang, N)
            zero = torch.zeros_like(y[:1])
            out.append(torch.cat([_exact_cg(A, q, zero, case["iters"]) if case["solver"] == "cg" else
                                  _exact_sb(A, q, 0.1, 10.0, case["iters"], True) for q in y.split(1)]))
        return out
    if kind == "serve":
        probs, sino, sb, lam = _serve_inputs(case, seed)
        out = [None] * len(probs)
        for (N, nang), idx in _groups(probs):
            A = _toeplitz2d(N, nang, N)
            ys = _exact_rhs2d(torch.as_tensor(np.concatenate([sino[i] for i in idx]), device=DEV).double(), N)
            for j, i in enumerate(idx):
                q = ys[j:j + 1]
                out[i] = (_exact_sb(A, q, lam[i], 10.0, case["iters"], True) if sb[i] else
                          _exact_cg(A, q, torch.zeros_like(q), case["iters"])).cpu().numpy()
        return out
    n1, n, nproj, nrows = case["n1"], case["n"], case["nproj"], case["nrows"]
    if kind == "solve3d":
        y, ncols, crop = _rhs3d(n1, n, nproj, nrows, seed).double(), n, None
    else:
        dims, det = tuple(_pad_size(v) for v in (n1, n, n)), (_pad_size(nrows), _pad_size(n))
        if 4.0 * nproj * math.prod(det) * math.prod(dims) > EXACT_FLOPS:
            return None
        p = _projections3d(n1, n, nproj, nrows, n, seed)
        q = torch.zeros((nproj,) + det, device=DEV, dtype=F64)
        a, b = (det[0] - nrows) // 2, (det[1] - n) // 2
        q[:, a:a + nrows, b:b + n] = (p / p.max()).double()
        crop = [slice((dims[i] - v) // 2, (dims[i] - v) // 2 + v) for i, v in enumerate((n1, n, n))]
        (nrows, ncols), n1, n = det, dims[0], dims[1]
        y = _exact_rhs3d(q, dims)
    A = _toeplitz3d(nproj, nrows, ncols, n1, n)
    x = _exact_cg(A, y, torch.zeros_like(y), case["iters"]) if case["solver"] == "cg" else \
        _exact_sb(A, y, 0.1, 10.0, case["iters"], False)
    return x if crop is None else x[tuple(crop)].contiguous().cpu().numpy()
