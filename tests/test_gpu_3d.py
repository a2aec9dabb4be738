"""GPU parity of the 3-D laminography path against the FP64 oracle and the
committed golden vectors, through the C ABI: PointSpreadFunction and
sysmat(x, psf) (include/toeplitz.h:61-129), CG and Split-Bregman
(src/conjgrad.cpp:33-76, src/bregman.cpp:36-94), forward / backproj / NUFFT
sysmat (src/projection.cpp:42-131, src/gradient.cpp:32-41)."""
import os

import numpy as np
import pytest

from conftest import announce, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lc():
    import laminocam_amd
    return laminocam_amd


def lamino_angles(n, tilt_deg=-30.0, span=2 * np.pi):
    th = np.arange(n) * span / n
    return th, np.full(n, np.deg2rad(tilt_deg)), np.zeros(n)


# (recon dims, nproj, nrows, ncols, tilt): odd/even dims, PSF sizes 2^p 3^q,
# a single slice (M1 = 1), no tilt
SHAPES = [((5, 16, 16), 7, 9, 16, -30.0), ((3, 33, 33), 11, 12, 30, -30.0),
          ((8, 40, 40), 30, 16, 40, 20.0), ((1, 24, 24), 9, 6, 24, -30.0),
          ((6, 32, 32), 13, 10, 32, 0.0)]


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", SHAPES)
def test_kernel_hat3d_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"kernel_hat3d dims={dims} nproj={nproj}")
    th, ga, be = lamino_angles(nproj, tilt)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, nrows, ncols), dims)
    ref = orc64.psf3d(th, ga, be, nrows, ncols, dims, method=0)
    assert tuple(psf.dims()) == tuple(ref.dims)
    kh, kr = psf.kernel_hat(), ref.kernel_hat()
    assert kh.shape == kr.shape
    assert rel_l2(kh, kr) < 2e-6


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", SHAPES)
def test_toeplitz3d_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"toeplitz3d dims={dims} nproj={nproj}")
    rng = np.random.default_rng(sum(dims) + nproj)
    th, ga, be = lamino_angles(nproj, tilt)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, nrows, ncols), dims)
    x = rng.random(dims).astype(np.float32)   # float32: the FP32 operator
    y = psf.convolve(x)
    yr = orc64.psf3d(th, ga, be, nrows, ncols, dims, method=0).convolve(x)
    err = rel_l2(y, yr)
    print(f"toeplitz3d rel_l2 = {err:.3e}")
    assert err < 1e-5


@pytest.mark.parametrize("dims,nproj,nrows", [((3, 721, 721), 6, 8), ((2, 576, 576), 5, 6)])
def test_toeplitz3d_large_inplane_matches_oracle(lc, orc64, dims, nproj, nrows):
    # in-plane PSF lengths above 1024 (1458 as in the laminography volume,
    # 1152), which take the 512-thread row passes, on a short slice axis
    announce(f"toeplitz3d large in-plane dims={dims}")
    rng = np.random.default_rng(dims[1])
    th, ga, be = lamino_angles(nproj)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, nrows, dims[2]), dims)
    assert psf.dims()[1] > 1024
    x = rng.random(dims).astype(np.float32)
    y = psf.convolve(x)
    yr = orc64.psf3d(th, ga, be, nrows, dims[2], dims, method=0).convolve(x)
    err = rel_l2(y, yr)
    print(f"toeplitz3d {dims} rel_l2 = {err:.3e}")
    assert err < 1e-5


def test_toeplitz3d_lamino_size_symmetric_psd(lc):
    # the padded laminography volume of the 3-D configuration: 29 x 721 x 721
    # on 360 projections of 89 x 721 at 30 degrees tilt.  A^T A is symmetric and
    # positive semi-definite whatever the size (tests/test_adjoint.cpp)
    announce("toeplitz3d 29x721x721 symmetry")
    th, ga, be = lamino_angles(360)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, 89, 721), (29, 721, 721))
    assert tuple(psf.dims()) == (64, 1458, 1458)
    rng = np.random.default_rng(11)
    x = rng.standard_normal((29, 721, 721)).astype(np.float32)
    z = rng.standard_normal((29, 721, 721)).astype(np.float32)
    ax, az = psf.convolve(x), psf.convolve(z)
    lhs = float(np.vdot(ax.astype(np.float64), z))
    rhs = float(np.vdot(x.astype(np.float64), az))
    assert abs(lhs - rhs) <= 1e-4 * np.linalg.norm(ax) * np.linalg.norm(z)
    assert float(np.vdot(ax.astype(np.float64), x)) > 0.0


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", SHAPES[:3])
def test_cg3d_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"cg3d dims={dims}")
    rng = np.random.default_rng(5)
    th, ga, be = lamino_angles(nproj, tilt)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, nrows, ncols), dims)
    P = orc64.psf3d(th, ga, be, nrows, ncols, dims, method=0)
    xt = rng.random(dims)
    y = P.convolve(xt).astype(np.float32)
    x, rep = lc.cgsolver(psf, y, np.zeros(dims, np.float32), 5, 1e-12, 0.0)
    xr, rr = orc64.cgsolver(P, y, np.zeros(dims), 5, 1e-12, 0.0)
    assert rep["iters"] == rr["iters"]
    err = rel_l2(x, xr)
    print(f"cg3d rel_l2 = {err:.3e}")
    assert err < 1e-3


@pytest.mark.parametrize("zero_pad", [False, True])
def test_split_bregman3d_matches_oracle(lc, orc64, zero_pad):
    announce(f"split_bregman3d zero_pad={zero_pad}")
    dims = (5, 16, 16)
    rng = np.random.default_rng(8)
    th, ga, be = lamino_angles(9)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, 9, 16), dims)
    P = orc64.psf3d(th, ga, be, 9, 16, dims, method=0)
    y = P.convolve(rng.random(dims)).astype(np.float32)
    x, rep = lc.split_bregman(psf, y, np.zeros(dims, np.float32), 0.1, 10.0, 6, 1, 1e-12, 0.0,
                              zero_pad=zero_pad)
    xr, rr = orc64.split_bregman(P, y, np.zeros(dims), 0.1, 10.0, 6, 1, 1e-12, 0.0,
                                 boundary=1 if zero_pad else 0)
    err = rel_l2(x, xr)
    print(f"sb3d rel_l2 = {err:.3e}")
    assert err < 1e-3


def test_batch_mixed_2d_3d_same_alone_and_in_mix(lc):
    # a 3-D volume batched with 2-D stacks keeps its own CG scalars: its result
    # is bitwise the result of solving it alone
    announce("mixed 2-D / 3-D batch")
    rng = np.random.default_rng(21)
    dims = (6, 32, 32)
    th, ga, be = lamino_angles(13)
    p3 = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, 10, 32), dims)
    p2a = lc.PointSpreadFunction2D(lc.PolarGrid2D(np.arange(30) * np.pi / 30, 48), 48)
    p2b = lc.PointSpreadFunction2D(lc.PolarGrid2D(np.arange(20) * np.pi / 20, 32), 32)
    f32 = np.float32
    y3 = p3.convolve(rng.random(dims).astype(f32))
    y2a = p2a.convolve(rng.random((2, 48, 48)).astype(f32))
    y2b = p2b.convolve(rng.random((1, 32, 32)).astype(f32))
    mix = lc.Batch2D([p2a, p3, p2b], ns=[2, 0, 1])
    for i, y in enumerate([y2a, y3, y2b]):
        mix.set(i, mix.Y, y)
    mix.cg(8, 0.0, 0.0, graph=True)
    alone = lc.Batch2D([p3])
    alone.set(0, alone.Y, y3)
    alone.cg(8, 0.0, 0.0, graph=True)
    assert np.array_equal(mix.get(1, mix.X), alone.get(0, alone.X))
    single, _ = lc.cgsolver(p3, y3, np.zeros(dims, np.float32), 8, 0.0, 0.0)
    assert np.array_equal(single, alone.get(0, alone.X))


# ---------------------------------------------------------------- projectors
GOLDEN3 = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "golden3d.npz")
PROJ_TOL = 1e-4


def test_projectors3d_match_golden(lc):
    # brute-force NUDFT + numpy FFT restatement of the reference chain (odd,
    # non-2^p3^q detector: Bluestein path; rectangular volume)
    announce("projector3d golden")
    d = np.load(GOLDEN3)
    g = lc.PolarGrid(d["theta"], d["gamma"], d["beta"], int(d["det"][0]), int(d["det"][1]))
    fwd = lc.forward(d["vol"], g)
    assert fwd.shape == d["fwd"].shape
    assert rel_l2(fwd, d["fwd"]) < PROJ_TOL
    assert rel_l2(lc.backproj(d["proj"], g, tuple(d["dims"])), d["bp"]) < PROJ_TOL
    assert rel_l2(lc.backproj(d["proj"], g, tuple(d["dims"]), d["shifts"]), d["bp_shift"]) < PROJ_TOL


# (recon dims, nproj, nrows, ncols, tilt)
PSHAPES = [((6, 24, 24), 20, 16, 24, -30.0), ((5, 21, 19), 13, 11, 23, -30.0),
           ((9, 32, 32), 36, 13, 31, 20.0), ((1, 30, 30), 12, 8, 32, -30.0)]


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", PSHAPES)
def test_forward3d_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"forward3d dims={dims} det=({nrows},{ncols})")
    rng = np.random.default_rng(31 + nproj)
    th, ga, be = lamino_angles(nproj, tilt)
    vol = rng.random(dims)
    y = lc.forward(vol, lc.PolarGrid(th, ga, be, nrows, ncols))
    yr = orc64.forward3d(vol, th, ga, be, nrows, ncols, tol=1e-12)
    err = rel_l2(y, yr)
    print(f"forward3d rel_l2 = {err:.3e}")
    assert err < PROJ_TOL


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", PSHAPES)
def test_backproj3d_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"backproj3d dims={dims} det=({nrows},{ncols})")
    rng = np.random.default_rng(41 + nproj)
    th, ga, be = lamino_angles(nproj, tilt)
    proj = rng.standard_normal((nproj, nrows, ncols))
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    x = lc.backproj(proj, g, dims)
    xr = orc64.backproj3d(proj, th, ga, be, dims, tol=1e-12)
    err = rel_l2(x, xr)
    print(f"backproj3d rel_l2 = {err:.3e}")
    assert err < PROJ_TOL
    sh = rng.uniform(-2, 2, (nproj, 2))
    xs = lc.backproj(proj, g, dims, sh)
    xsr = orc64.backproj3d(proj, th, ga, be, dims, shifts=sh, tol=1e-12)
    assert rel_l2(xs, xsr) < PROJ_TOL


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", [((7, 36, 53), 90, 24, 53, -30.0),
                                                          ((16, 96, 96), 90, 32, 96, -30.0)])
def test_backproj3d_mid_size_matches_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    # fine grids (16, 72, 108) and (32, 192, 192): an odd number of spread bins
    # with a partial last bin, and many points per bin
    announce(f"backproj3d mid size dims={dims} det=({nrows},{ncols})")
    rng = np.random.default_rng(51 + nproj)
    th, ga, be = lamino_angles(nproj, tilt)
    proj = rng.standard_normal((nproj, nrows, ncols))
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    sh = rng.uniform(-2, 2, (nproj, 2))
    x = lc.backproj(proj, g, dims, sh)
    xr = orc64.backproj3d(proj, th, ga, be, dims, shifts=sh, tol=1e-9)
    err = rel_l2(x, xr)
    print(f"backproj3d rel_l2 = {err:.3e}")
    assert err < PROJ_TOL
    # deterministic: the same call gives the same bits
    assert np.array_equal(lc.backproj(proj, g, dims, sh), x)


# tilts per projection and the span of theta: one tilt over a full turn (opposite
# projections coincide: even and odd counts), two tilts, a tilt per projection
# (no two share a column direction) and for every two, and repeated angles
@pytest.mark.parametrize("kind,nproj", [("turn", 24), ("turn", 25), ("two", 24), ("each", 11), ("pairs", 26),
                                        ("repeat", 12), ("beta", 18)])
def test_psf3d_projection_groups_match_oracle(lc, orc64, kind, nproj):
    announce(f"psf3d groups {kind} nproj={nproj}")
    dims, nrows, ncols = (5, 22, 22), 9, 21
    th = np.arange(nproj) * (2 * np.pi / nproj)
    ga, be = np.full(nproj, -np.pi / 6), np.zeros(nproj)
    if kind == "two":
        ga[nproj // 2:] = 0.3
    elif kind == "each":
        ga = np.linspace(-0.6, 0.2, nproj)
    elif kind == "pairs":
        ga = np.linspace(-0.6, 0.2, nproj // 2)[np.arange(nproj) % (nproj // 2)]
    elif kind == "repeat":
        th = np.repeat(th[::3], 3)
    elif kind == "beta":
        be[:] = 0.2
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, be, nrows, ncols), dims)
    P = orc64.psf3d(th, ga, be, nrows, ncols, dims, method=0)
    x = np.random.default_rng(5).random(dims)
    ref = P.convolve(x)
    # FP32 operator: a few ulp of FP32; FP64 operator: phases of magnitude
    # pi |m| < 200 in FP64 (3e-14), times the denominators' margin
    assert rel_l2(psf.convolve(x.astype(np.float32)), ref) < 1e-6
    assert rel_l2(psf.convolve(x), ref) < 1e-12


# PSF sizes along z and along x / y with compiled line passes (16, 32, 64, 128,
# 192, 384) and with the run-time plan (24, 27, 36, 48), in both combinations
@pytest.mark.parametrize("dims", [(8, 24, 24), (12, 96, 96), (14, 64, 64), (16, 18, 18), (32, 180, 180)])
def test_psf3d_line_lengths_match_oracle(lc, orc64, dims):
    announce(f"psf3d line lengths {dims}")
    nproj, nrows, ncols = 7, 11, dims[2] + 1
    th = np.arange(nproj) * (np.pi / nproj)
    args = (th, np.full(nproj, -np.pi / 6), np.zeros(nproj))
    psf = lc.PointSpreadFunction(lc.PolarGrid(*args, nrows, ncols), dims)
    x = np.random.default_rng(8).random(dims)
    ref = orc64.psf3d(*args, nrows, ncols, dims, method=0).convolve(x)
    # as for the projection groups; phases of magnitude pi |m| < 700 (1e-13)
    assert rel_l2(psf.convolve(x.astype(np.float32)), ref) < 1e-6
    assert rel_l2(psf.convolve(x), ref) < 1e-11


# a sinogram of more points than the forward projector sorts at a time (2^27):
# the projections on either side of the boundary, and the last ones, against a
# grid of these alone
def test_forward3d_ranges_match_a_small_grid(lc):
    announce("forward3d in ranges")
    dims, nrows, ncols = (6, 16, 16), 48, 64
    per = (1 << 27) // (nrows * ncols)
    nproj = per + 70
    th = np.arange(nproj) * (2 * np.pi / nproj)
    ga = np.full(nproj, -np.pi / 6)
    vol = np.random.default_rng(7).random(dims).astype(np.float32)
    pick = np.r_[0:3, per - 3:per + 3, nproj - 3:nproj]
    all_of = lc.forward(vol, lc.PolarGrid(th, ga, np.zeros(nproj), nrows, ncols))[pick]
    few = lc.forward(vol, lc.PolarGrid(th[pick], ga[pick], np.zeros(len(pick)), nrows, ncols))
    assert rel_l2(all_of, few) < 1e-6   # the same FP32 operations per point


# a PSF large enough for runs of 32 values (the sizes above and several tilts take
# 16), the last run of a row partly empty; detectors of fewer rows than a run
# crosses have several removable zeros in one run
@pytest.mark.parametrize("tilts", [1, 2])
@pytest.mark.parametrize("nrows", [5, 40])
def test_psf3d_long_runs_match_oracle(lc, orc64, nrows, tilts):
    announce(f"psf3d long runs nrows={nrows} tilts={tilts}")
    dims, nproj = (9, 401, 401), 6
    th = np.arange(nproj) * (2 * np.pi / nproj)
    ga = np.repeat([-np.pi / 6, 0.3 if tilts == 2 else -np.pi / 6], nproj // 2)
    psf = lc.PointSpreadFunction(lc.PolarGrid(th, ga, np.zeros(nproj), nrows, 401), dims)
    x = np.random.default_rng(6).random(dims)
    ref = orc64.psf3d(th, ga, np.zeros(nproj), nrows, 401, dims, method=0).convolve(x)
    # as above; phases of magnitude pi |m| < 2200 (3e-13)
    assert rel_l2(psf.convolve(x.astype(np.float32)), ref) < 1e-6
    assert rel_l2(psf.convolve(x), ref) < 1e-11


# (recon dims, nproj, nrows, ncols): fine grids of 16 .. 81 cells per axis, two,
# three (24 and 27 cells) and more bins of 7 to 9 corners; the last one puts
# over 2048 points into its bins, in no multiple of a table of points
BIN_EDGES = [((8, 12, 13), 24, 11, 16), ((9, 13, 18), 24, 12, 15), ((12, 16, 40), 20, 16, 31),
             ((13, 27, 24), 20, 17, 30), ((6, 16, 16), 331, 13, 35)]


@pytest.mark.parametrize("dims,nproj,nrows,ncols", BIN_EDGES)
def test_projectors3d_bin_edges_match_oracle(lc, orc64, dims, nproj, nrows, ncols):
    announce(f"projectors3d bin edges dims={dims} det=({nrows},{ncols})")
    rng = np.random.default_rng(61 + nproj)
    th, ga, be = lamino_angles(nproj, -30.0)
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    vol, proj = rng.random(dims), rng.standard_normal((nproj, nrows, ncols))
    yr = orc64.forward3d(vol, th, ga, be, nrows, ncols, tol=1e-12)
    xr = orc64.backproj3d(proj, th, ga, be, dims, tol=1e-12)
    # the projectors' FP32 error: at most 9e-7 at these sizes
    assert rel_l2(lc.forward(vol, g), yr) < 3e-6
    ctx = lc.Context(0)
    try:
        psf = lc.PointSpreadFunction(g, dims, ctx=ctx, lazy=True)
        for shape in range(3):
            ctx.set_tuning3d(psf, shape)
            x = lc.backproj(proj, g, dims, ctx=ctx)
            err = rel_l2(x, xr)
            print(f"shape {shape}: rel_l2 = {err:.3e}")
            assert err < 3e-6
            assert np.array_equal(lc.backproj(proj, g, dims, ctx=ctx), x)
    finally:
        ctx.close()


# the forward projector interpolates few points in their own order and more in
# sorted order: (recon dims, nproj, nrows, ncols) with fine grids of 16 .. 81 cells
# per axis (two, three and more bins) on either side of that line, which for small
# volumes lies at 674 thousand points, with masked points in both
FORWARD_LINE = [((6, 16, 16), 331, 34, 59), ((6, 16, 16), 331, 34, 61), ((9, 13, 18), 400, 31, 57),
                ((12, 16, 40), 400, 31, 57), ((13, 27, 24), 300, 41, 58)]


@pytest.mark.parametrize("dims,nproj,nrows,ncols", FORWARD_LINE)
def test_forward3d_sorted_and_unsorted_match_oracle(lc, orc64, dims, nproj, nrows, ncols):
    announce(f"forward3d line dims={dims} points={nproj * nrows * ncols}")
    vol = np.random.default_rng(nproj + ncols).random(dims)
    th, ga, be = lamino_angles(nproj, -30.0)
    y = lc.forward(vol, lc.PolarGrid(th, ga, be, nrows, ncols))
    # the projectors' FP32 error is about 5e-7
    assert rel_l2(y, orc64.forward3d(vol, th, ga, be, nrows, ncols, tol=1e-12)) < 5e-6
    # the first projections alone are few points: the other kernel or the same one
    few = lc.forward(vol, lc.PolarGrid(th[:5], ga[:5], be[:5], nrows, ncols))
    assert rel_l2(few, y[:5]) < 1e-6


# Points on the lattice of the fine grid: without a tilt, with ncols = n and a
# fine grid of 2 n cells, every point's position along x is an odd whole number
# and that of detector column 1 is 3, whose footprint starts at the periodic
# edge (cell -1 or 0, as the FP64 position rounds); tilted, a detector row does
# so where theta = 90 degrees and nrows = 3 n1.  Every kernel has to take the same
# corner, or the whole column or row is lost (4e-3 and more of the norm).
LATTICE = [((8, 96, 96), 16, 16, 96, 0.0), ((8, 128, 128), 24, 32, 128, 0.0), ((6, 288, 288), 8, 12, 288, 0.0),
           ((8, 384, 384), 6, 16, 384, 0.0), ((32, 128, 128), 50, 128, 128, 0.0), ((16, 128, 128), 4, 48, 128, -30.0)]


@pytest.mark.parametrize("dims,nproj,nrows,ncols,tilt", LATTICE)
def test_projectors3d_lattice_points_match_oracle(lc, orc64, dims, nproj, nrows, ncols, tilt):
    announce(f"projectors3d lattice points dims={dims} det=({nrows},{ncols}) tilt={tilt}")
    rng = np.random.default_rng(dims[2] + nrows)
    th, ga, be = lamino_angles(nproj, tilt)
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    vol = rng.standard_normal(dims).astype(np.float32)
    proj = rng.standard_normal((nproj, nrows, ncols)).astype(np.float32)
    # the projectors' FP32 error is about 5e-7
    assert rel_l2(lc.forward(vol, g), orc64.forward3d(vol, th, ga, be, nrows, ncols, tol=1e-12)) < 5e-6
    xr = orc64.backproj3d(proj, th, ga, be, dims, tol=1e-12)
    sr = orc64.sysmat3d_nufft(vol, th, ga, be, nrows, ncols, tol=1e-12)
    ctx = lc.Context(0)
    try:
        psf = lc.PointSpreadFunction(g, dims, ctx=ctx, lazy=True)
        for shape in range(3):
            ctx.set_tuning3d(psf, shape)
            assert rel_l2(lc.backproj(proj, g, dims, ctx=ctx), xr) < 5e-6
            assert rel_l2(lc.sysmat(vol, g, ctx=ctx), sr) < 5e-6
    finally:
        ctx.close()


# points whose coordinates equal pi up to rounding (40 of them on this detector)
# are masked as the reference's FP64 operations mask them; rounded otherwise,
# the projectors are 4e-5 and more off
@pytest.mark.parametrize("dims", [(5, 40, 40), (6, 16, 20)])
def test_projectors3d_mask_ties_match_oracle(lc, orc64, dims):
    announce(f"projectors3d mask ties dims={dims}")
    nproj, nrows, ncols = 60, 30, 180
    rng = np.random.default_rng(dims[1])
    th, ga, be = lamino_angles(nproj, -30.0)
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    vol, proj = rng.standard_normal(dims), rng.standard_normal((nproj, nrows, ncols))
    # the projectors' FP32 error is about 5e-7
    assert rel_l2(lc.forward(vol, g), orc64.forward3d(vol, th, ga, be, nrows, ncols, tol=1e-12)) < 5e-6
    assert rel_l2(lc.backproj(proj, g, dims), orc64.backproj3d(proj, th, ga, be, dims, tol=1e-12)) < 5e-6


def test_backproj3d_bin_shapes_and_autotune(lc, orc64):
    # every choice of the spread (bins of more than 2048 points shared out among
    # teams of waves, or of more than 512 with choice 2) gives the oracle's
    # back-projection, deterministically; the autotuner installs one of them for
    # the grid's fine-grid shape
    dims, nproj, nrows, ncols = (16, 96, 96), 90, 32, 96
    announce(f"backproj3d bin shapes dims={dims}")
    rng = np.random.default_rng(77)
    th, ga, be = lamino_angles(nproj, -30.0)
    proj = rng.standard_normal((nproj, nrows, ncols))
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    sh = rng.uniform(-2, 2, (nproj, 2))
    xr = orc64.backproj3d(proj, th, ga, be, dims, shifts=sh, tol=1e-9)
    ctx = lc.Context(0)
    try:
        psf = lc.PointSpreadFunction(g, dims, ctx=ctx)
        xs = []
        for shape in range(3):
            ctx.set_tuning3d(psf, shape)
            assert ctx.get_tuning3d(psf) == shape
            x = lc.backproj(proj, g, dims, sh, ctx=ctx)
            err = rel_l2(x, xr)
            print(f"shape {shape}: rel_l2 = {err:.3e}")
            assert err < PROJ_TOL
            assert np.array_equal(lc.backproj(proj, g, dims, sh, ctx=ctx), x)
            xs.append(x)
        for x in xs[1:]:
            assert rel_l2(x, xs[0]) < 1e-5
        best, ms = ctx.autotune3d(psf)
        print(f"autotune3d: shape {best}, {ms:.3f} ms")
        assert best in (0, 1, 2) and ms > 0.0
        assert ctx.get_tuning3d(psf) == best
        assert np.array_equal(lc.backproj(proj, g, dims, sh, ctx=ctx), xs[best])
    finally:
        ctx.close()


def test_backproj3d_shift_count_mismatch(lc):
    # src/projection.cpp:105-108: std::invalid_argument
    th, ga, be = lamino_angles(4)
    g = lc.PolarGrid(th, ga, be, 4, 8)
    with pytest.raises(ValueError):
        lc.backproj(np.zeros((4, 4, 8)), g, (2, 8, 8), np.zeros((3, 2)))


@pytest.mark.parametrize("dims,nproj,nrows,ncols", [((4, 32, 32), 24, 16, 32), ((8, 48, 48), 60, 32, 48)])
def test_projectors3d_adjoint(lc, dims, nproj, nrows, ncols):
    # even detector dims: fftshift2 == ifftshift2, so backproj is the adjoint of forward
    announce(f"adjoint3d dims={dims}")
    rng = np.random.default_rng(2)
    th, ga, be = lamino_angles(nproj)
    g = lc.PolarGrid(th, ga, be, nrows, ncols)
    x = rng.random(dims)
    y = rng.standard_normal((nproj, nrows, ncols))
    lhs = float(np.vdot(lc.forward(x, g).astype(np.float64), y))
    rhs = float(np.vdot(x, lc.backproj(y, g, dims).astype(np.float64)))
    assert abs(lhs - rhs) <= 1e-5 * (abs(lhs) + abs(rhs))


@pytest.mark.parametrize("tilt", [0.0, -30.0])
def test_sysmat3d_nufft_matches_oracle_and_toeplitz(lc, orc64, tilt):
    # tests/test_sysmat_toeplitz.cpp:48-127: NUFFT sysmat == Toeplitz sysmat when
    # the detector matches the image (nrows * ncols = n2 * n3)
    announce(f"sysmat3d nufft tilt={tilt}")
    rng = np.random.default_rng(4)
    dims = (5, 16, 16)
    th, ga, be = lamino_angles(9, tilt)
    g = lc.PolarGrid(th, ga, be, 16, 16)
    x = rng.random(dims)
    y1 = lc.sysmat(x, g)
    assert rel_l2(y1, orc64.sysmat3d_nufft(x, th, ga, be, 16, 16, tol=1e-12)) < PROJ_TOL
    y2 = lc.sysmat(x, lc.PointSpreadFunction(g, dims))
    assert rel_l2(y1, y2) < PROJ_TOL


def test_projectors3d_lamino_size(lc):
    # the laminography configuration's shapes: volume 29 x 721 x 721,
    # 360 projections of 89 x 721 (Bluestein on both detector axes); adjoint
    # pairing holds up to the odd-length shift convention, so check the
    # forward/backward sizes and finiteness plus linearity
    announce("projectors3d 29x721x721 / 360x89x721")
    th, ga, be = lamino_angles(360)
    g = lc.PolarGrid(th, ga, be, 89, 721)
    rng = np.random.default_rng(6)
    x = rng.random((29, 721, 721)).astype(np.float32)
    p = lc.forward(x, g)
    assert p.shape == (360, 89, 721) and np.all(np.isfinite(p))
    p2 = lc.forward(2.0 * x, g)
    assert rel_l2(p2, 2.0 * p) < 1e-6
    b = lc.backproj(p, g, (29, 721, 721))
    assert b.shape == (29, 721, 721) and np.all(np.isfinite(b))
    assert float(np.vdot(b.astype(np.float64), x)) > 0.0
