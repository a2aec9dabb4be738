// 3-D laminography NUFFT projectors on gfx950: forward, backproj (with
// optional centre-of-rotation shifts) and the NUFFT normal operator
// (src/projection.cpp:42-131, src/gradient.cpp:32-41).
//
//   forward(x)  = Re(ifftshift2(ifft2(fftshift2(w . T2 x)))) / (nrows ncols)
//   backproj(y) = Re(T1(w . e^{-i(qx dx + qy dy)} . ifftshift2(fft2(fftshift2 y)))) / (nrows ncols)
//   sysmat(x)   = Re(T1(T2 x)) / (nrows ncols)                (no mask)
// T1/T2: type-1/type-2 NUFFT on the grid R_i (qX_k, qY_j, 0), modes {n1,n2,n3}
// with m_x <-> n3, m_y <-> n2, m_z <-> n1 (include/nufft.h:37-58); w = 0 where
// any coordinate exceeds pi (include/polar_grid.h:80-86).
//
// Method as in 2-D: exponential-of-semicircle kernel, width 8, fine grid 2n
// per axis (2^p 3^q, at least 16), centred so points map to cells without a
// shift; the (-1)^m phase and 1/psi_hat sit in per-axis correction factors.
//   type 1: deterministic sorted-bin spreading -> fine grid, then one pruned
//           FFT pass per axis (x, y, z), deconvolution in each pass;
//   type 2: the reverse passes, then 8x8x8 interpolation of the points, sorted
//           where there are enough of them.
// Detector transforms are line FFTs along x then y with the reference's shift
// index maps; widths that are not 2^p 3^q use Bluestein's algorithm with an
// FP64-built chirp and chirp spectrum.
#include <cmath>
#include <complex>

#include <rocprim/device/device_radix_sort.hpp>

#include "lc_engine.hpp"

namespace lc {

extern __shared__ __align__(16) char lc_smem[];

namespace {

constexpr int W3 = 8;                       // kernel width (cells)
constexpr int LN_NT = 256, LN_ME = 32;      // line passes: NT * ME complex in LDS

// The compiled line passes hold NT * LN_ME_CT values per block (32 KiB), so
// a CU holds five blocks.
constexpr int LN_ME_CT = 16;
template <typename F> bool with_line_len(int L, F &&f) { return with_ct_len(L, f); }

// exp(beta (sqrt(1 - z^2) - 1)) for |z| < 1, else 0.  The hardware square
// root (within 1 ulp; s lies in (0, 1]) instead of the correctly rounded
// sequence: one instruction instead of about fifteen, a relative weight
// error near 1e-6, inside the kernel's own approximation error
__device__ __forceinline__ float es3(float z, float beta) {
    const float s = 1.0f - z * z;
    return s > 0.0f ? __expf(beta * (__builtin_amdgcn_sqrtf(s) - 1.0f)) : 0.0f;
}

// a modulo n for a in [-n, 2 n)
__device__ __forceinline__ int wrapi(int a, int n) {
    a += a < 0 ? n : 0;
    return a - (a >= n ? n : 0);
}

// a / b for inv = 1.0 / b: the FP64 product is within one of the quotient
__device__ __forceinline__ unsigned div_by(unsigned a, unsigned b, double inv) {
    const unsigned q = (unsigned)((double)a * inv);
    const int r = (int)(a - q * b);
    return r < 0 ? q - 1 : r >= (int)b ? q + 1 : q;
}

struct Grid3 {
    int nproj, nrows, ncols;
    int nf[3];          // fine grid (z, y, x)
    double dX, dY;      // lattice steps 2 pi / ncols, 2 pi / nrows
    double icols, irows;   // 1 / ncols, 1 / nrows
    float beta;
    int mask;           // 1: drop points with any |coordinate| > pi
};

// A point's position is rounded alike in every kernel: its fused multiply-adds are
// explicit.  Positions that are whole numbers up to rounding are common (an
// untilted scan with ncols = n has no others along x), and kernels that let the
// compiler fuse these products each in its own way took different corners for
// them, on the two sides of the periodic edge at worst.
__device__ __forceinline__ double lattice_coord(int k, double step) {   // (k + 1/2) step - pi
    return __builtin_fma((double)k + 0.5, step, -M_PI);
}
__device__ __forceinline__ void point3(const double *rot, int p, int j, int k, const Grid3 &g,
                                       double &x, double &y, double &z) {
    const double *r = rot + 6 * (int64_t)p;
    const double qx = lattice_coord(k, g.dX), qy = lattice_coord(j, g.dY);
    x = __builtin_fma(qy, r[3], qx * r[0]);
    y = __builtin_fma(qy, r[4], qx * r[1]);
    z = __builtin_fma(qy, r[5], qx * r[2]);
}

// the reference's mask (include/polar_grid.h:80-86): some coordinates equal pi up
// to rounding, so by its own operations, of which none is fused
__device__ __forceinline__ bool inside_pi(const double *rot, int p, int j, int k, const Grid3 &g) {
#pragma clang fp contract(off)
    const double *r = rot + 6 * (int64_t)p;
    const double qx = ((double)k + 0.5) * g.dX - M_PI, qy = ((double)j + 0.5) * g.dY - M_PI;
    const double x = qx * r[0] + qy * r[3], y = qx * r[1] + qy * r[4], z = qx * r[2] + qy * r[5];
    return fabs(x) <= M_PI && fabs(y) <= M_PI && fabs(z) <= M_PI;
}

// ---------------------------------------------------------------------------
// Points by bins of footprint corners.  A point's corner is its first
// footprint cell, ceil(g - W3/2) per axis, taken modulo nf.  Every axis is cut
// into nb bins of corners, bin i starting at floor(i nf / nb): an even number
// of bins of 7 to BE cells (three bins where no even number gives such widths:
// nf = 24 and 27), so that the footprints of one bin lie in a region of 16
// cells along each axis, and the regions of two bins an even distance apart
// are disjoint, around the periodic wrap too.  k_bin_keys
// gives every point its bin and, below it, its corner's row in the bin; a
// stable radix sort (rocPRIM) orders the points, keeping point order where
// the keys agree; k_bin_ranges marks each bin's run.
// ---------------------------------------------------------------------------
constexpr int RGN = 16;                     // region cells along an axis: the edge of an MFMA tile
constexpr int BE = RGN - W3 + 1;            // most corner cells of a bin along an axis
constexpr int YB = 4;                       // key bits of a corner's row in its bin
constexpr int TEAMS = 4;                    // teams of a heavy bin (their tables fill the LDS)
static_assert(RGN % 8 == 0 && BE < 1 << YB, "rows go to four waves in turn; a row index fits its key bits");

// The spread's choices, per fine-grid shape (nufft3d_autotune): a bin of more
// than HEAVY points is spread by several teams of waves.  2048 is the default;
// 512 wins where the fullest bins of a phase are its time, and loses where the
// phases are long (back-projection, us, 2048 / 512: 8 x 256^2 from 180 x 64 rows
// 1417 / 1182, 16 x 128^2 from 360 x 48 1903 / 1568, 128^3 from 360 x 128 3093 /
// 2744; 32 x 256^2 from 720 x 96 4687 / 5281, 32 x 511^2 from 720 x 128 9832 /
// 11404).  Choice 1, once bins of 25 rows (2.0 to 3.4 times the default's time
// over twelve scans), is the default too.
constexpr int N_SHAPES3 = 3;
template <typename F> void with_heavy3(int i, F &&f) {
    if (i == 2) f(std::integral_constant<unsigned, 512>{});
    else f(std::integral_constant<unsigned, 2048>{});
}

// bins along an axis of nf >= 16 cells
__host__ __device__ constexpr int bins_along(int nf) {
    int nb = 2 * ((nf + 2 * BE - 1) / (2 * BE));
    return nf / nb >= W3 - 1 ? nb : 3;
}

struct Bins3 {
    int nb[3];          // bins per axis
};
__device__ __forceinline__ int bin_first(int i, int nf, int nb) { return (int)((int64_t)i * nf / nb); }
// the bin of corner l: the largest i with bin_first(i) <= l
__device__ __forceinline__ int bin_of(int l, int nf, int nb) { return (int)(((int64_t)(l + 1) * nb - 1) / nf); }

// fine-grid position g, footprint corner l (unwrapped) of point (p, j, k).
// The columns of a rotation are orthonormal, so a coordinate is at most
// sqrt(2) pi in size and a corner lies in [-nf, 2 nf).
struct Corner3 {
    double gz, gy, gx;
    int lz, ly, lx;
    bool ok;    // false: dropped by the mask
};
__device__ __forceinline__ Corner3 corner3(const double *rot, int p, int j, int k, const Grid3 &g) {
    Corner3 c;
    double x, y, z;
    point3(rot, p, j, k, g, x, y, z);
    c.ok = !g.mask || inside_pi(rot, p, j, k, g);
    const double hw = 0.5 * W3;
    c.gz = __builtin_fma(z, g.nf[0] / (2.0 * M_PI), 0.5 * g.nf[0]);
    c.gy = __builtin_fma(y, g.nf[1] / (2.0 * M_PI), 0.5 * g.nf[1]);
    c.gx = __builtin_fma(x, g.nf[2] / (2.0 * M_PI), 0.5 * g.nf[2]);
    c.lz = (int)ceil(c.gz - hw);
    c.ly = (int)ceil(c.gy - hw);
    c.lx = (int)ceil(c.gx - hw);
    return c;
}
__device__ __forceinline__ Corner3 corner3(const double *rot, unsigned pt, const Grid3 &g) {
    const unsigned pj = div_by(pt, (unsigned)g.ncols, g.icols);
    const int k = (int)(pt - pj * (unsigned)g.ncols);
    const int p = (int)div_by(pj, (unsigned)g.nrows, g.irows), j = (int)(pj - (unsigned)p * (unsigned)g.nrows);
    return corner3(rot, p, j, k, g);
}

// key[i]: bin << YB | corner row in the bin of point i, or nbins << YB (sorted
// last) for a point the mask drops, whose value in `drop` (if given) becomes
// 0; val[i] = i
__global__ void k_bin_keys(const double *__restrict__ rot, Grid3 g, Bins3 bn, unsigned *__restrict__ key,
                           unsigned *__restrict__ val, int64_t npts, unsigned nbins, float2 *__restrict__ drop) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npts) return;
    const Corner3 c = corner3(rot, (unsigned)i, g);
    unsigned b = nbins << YB;
    if (c.ok) {
        const int lz = wrapi(c.lz, g.nf[0]), ly = wrapi(c.ly, g.nf[1]), lx = wrapi(c.lx, g.nf[2]);
        const int bz = bin_of(lz, g.nf[0], bn.nb[0]), by = bin_of(ly, g.nf[1], bn.nb[1]),
                  bx = bin_of(lx, g.nf[2], bn.nb[2]);
        b = (unsigned)(((int64_t)bz * bn.nb[1] + by) * bn.nb[2] + bx) << YB |
            (unsigned)(ly - bin_first(by, g.nf[1], bn.nb[1]));
    } else if (drop) {
        drop[i] = make_float2(0.f, 0.f);
    }
    key[i] = b;
    val[i] = (unsigned)i;
}

// [start[b], end[b]) is bin b's run in the sorted keys (start = end = 0 when
// empty: both arrays cleared first)
__global__ void k_bin_ranges(const unsigned *__restrict__ skey, int64_t n, unsigned *__restrict__ start,
                             unsigned *__restrict__ end, unsigned nbins) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned b = skey[i] >> YB;
    if (b >= nbins) return;
    if (i == 0 || (skey[i - 1] >> YB) != b) start[b] = (unsigned)i;
    if (i == n - 1 || (skey[i + 1] >> YB) != b) end[b] = (unsigned)(i + 1);
}

// launch phases along an axis: two (even and odd bins), or one per bin of three
__host__ __device__ constexpr int phases_along(int nb) { return nb == 3 ? 3 : 2; }

// the bins in launch order: grouped by phase (bins that may add to the grid
// side by side), fullest first inside a phase, so a phase's long-running
// dense bins start first and its tail is short.  key = phase << 26 |
// (2^26 - 1 - count), val = bin
constexpr int ORDER_BITS = 31;
__global__ void k_bin_order_keys(const unsigned *__restrict__ bstart, const unsigned *__restrict__ bend,
                                 Bins3 bn, unsigned *__restrict__ key, unsigned *__restrict__ val,
                                 unsigned nbins) {
    const unsigned b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbins) return;
    const unsigned bx = b % bn.nb[2], by = (b / bn.nb[2]) % bn.nb[1], bz = b / (bn.nb[2] * bn.nb[1]);
    const unsigned py = phases_along(bn.nb[1]), px = phases_along(bn.nb[2]);
    const unsigned ph = ((bz % phases_along(bn.nb[0])) * py + by % py) * px + bx % px;
    const unsigned cnt = min(bend[b] - bstart[b], (1u << 26) - 1);
    key[b] = (ph << 26) | ((1u << 26) - 1 - cnt);
    val[b] = b;
}

// include/fft.h:53-74 (phase_shift2d): detector spectrum C[p][j][k] *=
// exp(-i (qx_k dx_p + qy_j dy_p)), qx_k = (k + 1/2) 2 pi / ncols - pi,
// qy_j = (j + 1/2) 2 pi / nrows - pi; once per point, before the spread
__global__ void k_phase_shift3d(float2 *__restrict__ C, const double *__restrict__ shifts, Grid3 g,
                                int64_t np) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int64_t pj = i / g.ncols;
    const int kk = (int)(i - pj * g.ncols);
    const int pp = (int)(pj / g.nrows), jj = (int)(pj - (int64_t)pp * g.nrows);
    const double qx = lattice_coord(kk, g.dX), qy = lattice_coord(jj, g.dY);
    double s, c;
    sincos(qx * shifts[2 * pp] + qy * shifts[2 * pp + 1], &s, &c);
    const float cr = (float)c, si = (float)-s;
    const float2 cv = C[i];
    C[i] = make_float2(cv.x * cr - cv.y * si, cv.x * si + cv.y * cr);
}

// ---------------------------------------------------------------------------
// Both directions run on the matrix cores.  With wz, wy, wx a point's 8 weights
// per axis, placed at its corner in 16 slots that are zero elsewhere,
//   spread:  R[z][y][x]  = sum_p (wz_p[z] wy_p[y]) (c_p wx_p[x])   K = points
//   interp:  G[p][x]     = sum_{y,z} (wz_p[z] wy_p[y]) F[z][y][x]  K = (z, y)
//            c_p         = sum_x wx_p[x] G[p][x]
// so each region row y is one 16 x 16 FP32 MFMA tile (v_mfma_f32_16x16x4_f32:
// lane l holds A[l & 15][l >> 4], B[l >> 4][l & 15] and, in register q,
// D[4 (l >> 4) + q][l & 15]), once for the real and once for the imaginary
// part.  A block's four waves take the rows y = w, w + 4, ...; the points of a
// bin come in corner-row order, so a group of consecutive points touches 8 or
// 9 rows, and a wave skips the others.  A group's other weights are zeros:
// half the products along z and along x are wasted, which the matrix rate
// (twice the vector FMA rate, with no LDS access per cell) more than pays for.
// Weights are computed once per point into LDS tables of BATCH points.
// Measured: interpolating 23.1 M points (360 x 89 x 721 on 29 x 721^2) takes
// 3.7 ms against 22.0 ms with a wave per point reading its 512 cells through
// L1; spreading 47 M points (720 x 128 x 511 on 32 x 511^2) 6.8 ms against 13.5
// ms with a wave per bin adding each point's cells to an LDS copy of a 4 x 4 x
// 8 bin's region, and 2.9 M points (8 x 256^2) 1.15 against 2.61 ms.  Four waves
// per SIMD (128 registers) matter: with three the spread takes 20% longer.
// ---------------------------------------------------------------------------
using f32x4 = __attribute__((ext_vector_type(4))) float;
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
constexpr int BATCH = 128;                  // points per table; two threads fill a point's slots

// footprint corner of a point relative to its bin (inside it: corner3 gives
// every kernel the same corner), and the offset of its cell W3 / 2 from the
// point, in [0, 1), per axis (the weights' arguments are exact integers away
// from it: the largest weights get the smallest rounding)
template <typename T> struct Foot {
    int t[3];
    T f[3];
};
template <typename T>
__device__ __forceinline__ Foot<T> foot3(const double *rot, unsigned pt, const Grid3 &g, const int s[3]) {
    const Corner3 c = corner3(rot, pt, g);
    Foot<T> q;
    q.t[0] = wrapi(c.lz, g.nf[0]) - s[0];
    q.t[1] = wrapi(c.ly, g.nf[1]) - s[1];
    q.t[2] = wrapi(c.lx, g.nf[2]) - s[2];
    q.f[0] = (T)((double)(c.lz + W3 / 2) - c.gz);
    q.f[1] = (T)((double)(c.ly + W3 / 2) - c.gy);
    q.f[2] = (T)((double)(c.lx + W3 / 2) - c.gx);
    return q;
}

// the slots congruent to 4 h .. 4 h + 3 modulo 8 of one axis's `slots` slots:
// put(slot, weight), where one slot of each residue lies in the footprint
template <int SLOTS, typename T, typename F>
__device__ __forceinline__ void axis_weights(int t, T f, int h, float beta, F &&put) {
    const float ihw = 1.0f / (0.5f * W3);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * h + i, d = (r - t) & (W3 - 1), slot = t + d;
        const float w = es3((float)((T)(d - W3 / 2) + f) * ihw, beta);
#pragma unroll
        for (int s = 0; s < SLOTS; s += W3) put(r + s, r + s == slot ? w : 0.f);
    }
}
// smallest and largest corner row of the groups of G consecutive lanes
template <int G> __device__ __forceinline__ void group_rows(int ty, bool ok, int &lo, int &hi) {
    // (a corner's row lies in its bin: the bounds change no value, but the spread of
    // 8 x 256^2 from 180 x 64 rows takes 1400 us with them and 1413 without)
    ty = min(max(ty, 0), 63);
    lo = ok ? ty : 127;
    hi = ok ? ty : 0;
#pragma unroll
    for (int o = 1; o < G; o <<= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
}
// v summed over its row of 16 lanes (every lane gets the sum)
__device__ __forceinline__ float row_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, true));   // row_ror:1
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true));
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
}
// first and last of wave w's rows (row w + 4 q -> q) that a group with corner
// rows lo .. hi touches
__device__ __forceinline__ int first_row(int lo, int w) { return max(0, (lo - w + 3) >> 2); }
__device__ __forceinline__ int last_row(int hi, int w) { return (hi + W3 - 1 - w) >> 2; }

// value of v in lane `lane` (uniform lane index: a scalar broadcast, no LDS)
__device__ __forceinline__ float rl_f32(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double rl_f64(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// type 2 of few points, in their own order: a wave per 64 points.  Lane l first
// finds the footprint of point l; then the wave takes the points in turn with
// its lanes over the 8 x 8 (y, x) footprint, walking the 8 z planes, and sums
// the 64 lanes in a fixed order.  Bound by the 4 KB per point through L1, but
// free of the sort (see interp_direct).
__global__ void __launch_bounds__(256)
k_interp3d_direct(const float2 *__restrict__ F, float2 *__restrict__ C, const double *__restrict__ rot,
                  unsigned npts, Grid3 g) {
    static_assert(W3 == 8, "the lane layout assumes a footprint of 8 per axis");
    const int lane = threadIdx.x & 63;
    const unsigned base = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64;
    if (base >= npts) return;   // whole wave
    const Corner3 c = corner3(rot, min(base + lane, npts - 1), g);
    const float ihw = 1.0f / (0.5f * W3);
    const int iy = lane >> 3, ix = lane & 7;
    const int nloc = (int)min(npts - base, 64u);
    float2 res = make_float2(0.f, 0.f);
    for (int j = 0; j < nloc; ++j) {
        if (!__builtin_amdgcn_readlane(c.ok ? 1 : 0, j)) continue;   // masked point: 0
        const int z0 = __builtin_amdgcn_readlane(c.lz, j), y0 = __builtin_amdgcn_readlane(c.ly, j),
                  x0 = __builtin_amdgcn_readlane(c.lx, j);
        // lane (iy, ix) holds the y weight of row iy, the x weight of column
        // ix, and the z weight of plane ix (read by every lane in the z walk)
        const float wz = es3((float)((double)(z0 + ix) - rl_f64(c.gz, j)) * ihw, g.beta);
        const float wy = es3((float)((double)(y0 + iy) - rl_f64(c.gy, j)) * ihw, g.beta);
        const float wx = es3((float)((double)(x0 + ix) - rl_f64(c.gx, j)) * ihw, g.beta);
        const int yy = wrapi(y0 + iy, g.nf[1]), xx = wrapi(x0 + ix, g.nf[2]);
        float rr = 0.f, ri = 0.f;
#pragma unroll
        for (int a = 0; a < W3; ++a) {
            const float wza = rl_f32(wz, a);
            const float2 v = F[((int64_t)wrapi(z0 + a, g.nf[0]) * g.nf[1] + yy) * g.nf[2] + xx];
            rr += wza * v.x;
            ri += wza * v.y;
        }
        const float w = wy * wx;
        float sr = w * rr, si = w * ri;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            sr += __shfl_xor(sr, off, 64);
            si += __shfl_xor(si, off, 64);
        }
        if (lane == j) res = make_float2(sr, si);
    }
    if (base + lane < npts) C[base + lane] = res;
}

// type 2: a block takes `chunk` consecutive sorted points; for each bin among
// them the waves load their rows of the region into registers (they stay there
// for all the bin's points).  Every point's sum depends on that point alone.
// Masked points (sorted last) are not read.
constexpr int XS = 20;                      // row stride of the x table
__global__ void __launch_bounds__(256, 4)
k_interp3d(const float2 *__restrict__ F, float2 *__restrict__ C, const double *__restrict__ rot,
           const unsigned *__restrict__ skey, const unsigned *__restrict__ sval,
           const unsigned *__restrict__ bend, unsigned npts, unsigned nbins, unsigned chunk, Grid3 g, Bins3 bn) {
    __shared__ float Zt[BATCH * RGN], Yt[BATCH * RGN], Xt[BATCH * XS];   // [group][slot][16 points], x: [point][slot]
    __shared__ float2 part[4][BATCH];
    __shared__ int meta[BATCH / 16];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = threadIdx.x & (BATCH - 1), h = threadIdx.x >> 7;
    const int n = lane & 15, k4 = lane >> 4;
    unsigned a = blockIdx.x * chunk;
    const unsigned stop = min(npts, a + chunk);
    while (a < stop) {
        const unsigned bin = __builtin_amdgcn_readfirstlane(skey[a] >> YB);
        if (bin >= nbins) return;   // the masked points: all of the rest (the whole block agrees)
        const unsigned e = min(stop, bend[bin]);
        const int b[3] = {(int)(bin / (unsigned)(bn.nb[1] * bn.nb[2])), (int)(bin / (unsigned)bn.nb[2]) % bn.nb[1],
                          (int)(bin % (unsigned)bn.nb[2])};
        int s[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) s[i] = bin_first(b[i], g.nf[i], bn.nb[i]);
        // lane (k4, n): x = n, z = 4 j + k4 of row y = w + 4 q
        float fr[4][4], fi[4][4];
        {
            int xx = s[2] + n;
            xx -= xx >= g.nf[2] ? g.nf[2] : 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int yy = s[1] + w + 4 * q;
                yy -= yy >= g.nf[1] ? g.nf[1] : 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    int zz = s[0] + 4 * j + k4;
                    zz -= zz >= g.nf[0] ? g.nf[0] : 0;
                    const float2 v = F[((int64_t)zz * g.nf[1] + yy) * g.nf[2] + xx];
                    fr[q][j] = v.x;
                    fi[q][j] = v.y;
                }
            }
        }
        unsigned next = sval[min(a + p, e - 1)];   // this thread's point of the coming table
        for (; a < e; a += BATCH) {
            const int cnt = (int)min(e - a, (unsigned)BATCH);
            const bool ok = p < cnt;
            const unsigned pt = next;
            next = sval[min(a + BATCH + p, e - 1)];
            if ((p & 64) < cnt) {   // (a wave whose points all lie past the end has none to place)
                const Foot<double> ft = foot3<double>(rot, pt, g, s);
                float *zt = Zt + (p >> 4) * 256 + (p & 15), *yt = Yt + (p >> 4) * 256 + (p & 15), *xt = Xt + p * XS;
                axis_weights<RGN>(ft.t[0], ft.f[0], h, g.beta, [&](int sl, float v) { zt[16 * sl] = v; });
                axis_weights<RGN>(ft.t[1], ft.f[1], h, g.beta, [&](int sl, float v) { yt[16 * sl] = v; });
                axis_weights<RGN>(ft.t[2], ft.f[2], h, g.beta, [&](int sl, float v) { xt[sl] = v; });
                int lo, hi;
                group_rows<16>(ft.t[1], ok, lo, hi);
                if ((threadIdx.x & 15) == 0 && h == 0) meta[p >> 4] = lo | hi << 8;
            }
            __syncthreads();
            const int ng = (cnt + 15) >> 4;
            const int mt = meta[lane & 7];
            for (int gr = 0; gr < ng; ++gr) {
                const int m = __builtin_amdgcn_readlane(mt, gr);
                const int q0 = first_row(m & 255, w), q1 = last_row(m >> 8, w);
                float zw[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) zw[j] = Zt[gr * 256 + (4 * j + k4) * 16 + n];
                // even and odd rows apart: each matrix instruction is a chain
                // of rounded FMAs, and shorter chains round less
                f32x4 ar[2], ai[2];
                ar[0] = ar[1] = ai[0] = ai[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (q < q0 || q > q1) continue;
                    const float wy = Yt[gr * 256 + (w + 4 * q) * 16 + n];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float av = zw[j] * wy;
                        ar[q & 1] = mfma4(av, fr[q][j], ar[q & 1]);
                        ai[q & 1] = mfma4(av, fi[q][j], ai[q & 1]);
                    }
                }
                ar[0] += ar[1];
                ai[0] += ai[1];
                // register q: point 4 k4 + q, x = n; summed over x in the 16 lanes
                const float *xw = Xt + (gr * 16 + 4 * k4) * XS + n;
                float2 o = make_float2(0.f, 0.f);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float wx = xw[q * XS];
                    const float vr = row_sum(ar[0][q] * wx), vi = row_sum(ai[0][q] * wx);
                    if (n == q) o = make_float2(vr, vi);
                }
                if (n < 4) part[w][gr * 16 + 4 * k4 + n] = o;
            }
            __syncthreads();
            if (h == 0 && ok) {
                const float2 v0 = part[0][p], v1 = part[1][p], v2 = part[2][p], v3 = part[3][p];
                C[pt] = make_float2((v0.x + v1.x) + (v2.x + v3.x), (v0.y + v1.y) + (v2.y + v3.y));
            }
        }
        a = e;
    }
}

// Bins of more than HEAVY points are spread by TEAMS teams of four
// waves, each taking a consecutive part of the bin's points; their sums are
// added in team order.  Whether a bin is heavy depends only on its own count.

// LDS of one team: tables [point][slot] of wz, c wx (re, im) and wy (its rows
// reordered to [wave][row / 4]), the row strides padded against bank conflicts,
// and the point groups' rows
constexpr int ZS = RGN + 1;
struct alignas(16) SpreadLds {
    float z[BATCH * ZS], xr[BATCH * ZS], xi[BATCH * ZS];
    alignas(16) float y[BATCH * (RGN + 4)];   // read four rows at a time
    int meta[BATCH / 4];
};

// type 1: adds bin `bin`'s points to the fine grid F with NT teams of four waves
template <int NT>
__device__ __forceinline__ void spread3_bin(const float2 *__restrict__ C, float2 *__restrict__ F,
                                            const double *__restrict__ rot, const unsigned *__restrict__ sval,
                                            int bin, unsigned s0, unsigned s1, const Grid3 &g, const Bins3 &bn,
                                            SpreadLds *lds) {
    constexpr int NQ = RGN / 4, YS = RGN + 4;
    const int b[3] = {bin / (bn.nb[1] * bn.nb[2]), (bin / bn.nb[2]) % bn.nb[1], bin % bn.nb[2]};
    int s[3], ext[3];   // the region's first cell and extent (the bin's corners + W3 - 1)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        s[i] = bin_first(b[i], g.nf[i], bn.nb[i]);
        ext[i] = bin_first(b[i] + 1, g.nf[i], bn.nb[i]) - s[i] + W3 - 1;
    }
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const int team = NT == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int p = threadIdx.x & (BATCH - 1), h = (threadIdx.x >> 7) & 1;
    const int n = lane & 15, k4 = lane >> 4;
    SpreadLds &L = lds[team];
    // sums over the batches so far (tr, ti) and within one: two levels keep the
    // chains of rounded additions short where a bin holds thousands of points
    f32x4 tr[NQ], ti[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) tr[q] = ti[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    // team t takes the t-th part of the bin's points, in order; every team
    // runs the same number of batches
    const unsigned per = ((s1 - s0 + NT - 1) / NT + BATCH - 1) / BATCH * BATCH;
    const unsigned ws = min(s1, s0 + team * per), we = min(s1, ws + per);
    const int nit = (int)(per / BATCH);
    // the next batch's points are fetched during this one
    auto index = [&](int it) -> unsigned {
        const unsigned i = ws + (unsigned)it * BATCH + p;
        return sval[i < we ? i : s0];
    };
    unsigned pt = index(0), ptn = nit > 1 ? index(1) : pt;
    float2 cv = C[pt];
    for (int it = 0; it < nit; ++it) {
        const unsigned base = ws + (unsigned)it * BATCH;
        const int cnt = base < we ? (int)min(we - base, (unsigned)BATCH) : 0;
        const bool ok = p < cnt;
        if ((p & 64) < cnt) {   // (a wave whose points all lie past the end has none to place)
            const Foot<float> ft = foot3<float>(rot, pt, g, s);
            float *zt = L.z + p * ZS, *xr = L.xr + p * ZS, *xi = L.xi + p * ZS, *yt = L.y + p * YS;
            const float cr = ok ? cv.x : 0.f, ci = ok ? cv.y : 0.f;
            // past the last point every product is 0 x a stored weight
            axis_weights<RGN>(ft.t[0], ft.f[0], h, g.beta, [&](int sl, float v) { zt[sl] = ok ? v : 0.f; });
            axis_weights<RGN>(ft.t[1], ft.f[1], h, g.beta,
                                  [&](int sl, float v) { yt[(sl & 3) * NQ + (sl >> 2)] = v; });
            axis_weights<RGN>(ft.t[2], ft.f[2], h, g.beta, [&](int sl, float v) {
                xr[sl] = v * cr;
                xi[sl] = v * ci;
            });
            int lo, hi;
            group_rows<4>(ft.t[1], ok, lo, hi);
            if ((p & 3) == 0 && h == 0) L.meta[p >> 2] = lo | hi << 8;
        }
        __syncthreads();
        pt = ptn;
        cv = C[pt];
        if (it + 2 < nit) ptn = index(it + 2);
        const int mt = L.meta[lane & 31];
        const int ng = (cnt + 3) >> 2;
        const float *zl = L.z + k4 * ZS + n, *xrl = L.xr + k4 * ZS + n, *xil = L.xi + k4 * ZS + n;
        const float *yl = L.y + k4 * YS + w * NQ;
        f32x4 ar[NQ], ai[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) ar[q] = ai[q] = f32x4{0.f, 0.f, 0.f, 0.f};
        // the next group's operands are read during this one's products
        float zw = zl[0], br = xrl[0], bi = xil[0];
        f32x4 wy[NQ / 4];
#pragma unroll
        for (int q = 0; q < NQ / 4; ++q) wy[q] = *reinterpret_cast<const f32x4 *>(yl + 4 * q);
        for (int gr = 0; gr < ng; ++gr) {
            const int gn = min(gr + 1, BATCH / 4 - 1);
            const float zn = zl[gn * 4 * ZS], brn = xrl[gn * 4 * ZS], bnx = xil[gn * 4 * ZS];
            f32x4 wyn[NQ / 4];
#pragma unroll
            for (int q = 0; q < NQ / 4; ++q) wyn[q] = *reinterpret_cast<const f32x4 *>(yl + gn * 4 * YS + 4 * q);
            const int m = __builtin_amdgcn_readlane(mt, gr);
            const int q0 = first_row(m & 255, w), q1 = last_row(m >> 8, w);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                if (q < q0 || q > q1) continue;
                const float av = zw * wy[q / 4][q % 4];
                ar[q] = mfma4(av, br, ar[q]);
                ai[q] = mfma4(av, bi, ai[q]);
            }
            zw = zn;
            br = brn;
            bi = bnx;
#pragma unroll
            for (int q = 0; q < NQ / 4; ++q) wy[q] = wyn[q];
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            tr[q] += ar[q];
            ti[q] += ai[q];
        }
        __syncthreads();
    }
    // register i of row slot q: cell (z, y, x) = (4 k4 + i, w + 4 q, n)
    int xx = s[2] + n;
    xx -= xx >= g.nf[2] ? g.nf[2] : 0;
    auto cell = [&](int q, int i, bool &in) -> float2 * {
        const int y = w + 4 * q, z = 4 * k4 + i;
        in = y < ext[1] && z < ext[0] && n < ext[2];
        int yy = s[1] + y, zz = s[0] + z;
        yy -= yy >= g.nf[1] ? g.nf[1] : 0;
        zz -= zz >= g.nf[0] ? g.nf[0] : 0;
        return F + ((int64_t)zz * g.nf[1] + yy) * g.nf[2] + xx;
    };
    if constexpr (NT == 1) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            float2 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bool in;
                const float2 *f = cell(q, i, in);
                if (in) v[i] = *f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                bool in;
                float2 *f = cell(q, i, in);
                if (in) *f = make_float2(v[i].x + tr[q][i], v[i].y + ti[q][i]);
            }
        }
    } else {
        // row slot by row slot through LDS (the tables' space): team q mod
        // NT adds the teams' sums in team order
        f32x4 *ex = reinterpret_cast<f32x4 *>(lds);   // [team][wave][re, im][lane]
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            ex[((team * 4 + w) * 2) * 64 + lane] = tr[q];
            ex[((team * 4 + w) * 2 + 1) * 64 + lane] = ti[q];
            __syncthreads();
            if (q % NT == team) {
                f32x4 sr = ex[(w * 2) * 64 + lane], si = ex[(w * 2 + 1) * 64 + lane];
                for (int t = 1; t < NT; ++t) {
                    sr += ex[((t * 4 + w) * 2) * 64 + lane];
                    si += ex[((t * 4 + w) * 2 + 1) * 64 + lane];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bool in;
                    float2 *f = cell(q, i, in);
                    if (in) {
                        const float2 v = *f;
                        *f = make_float2(v.x + sr[i], v.y + si[i]);
                    }
                }
            }
            __syncthreads();
        }
    }
}

// one block per light bin of this phase (order: the phase's bins, fullest first)
template <unsigned HEAVY>
__global__ void __launch_bounds__(256, 4)
k_spread3d_bin(const float2 *__restrict__ C, float2 *__restrict__ F, const double *__restrict__ rot,
               const unsigned *__restrict__ sval, const unsigned *__restrict__ bstart,
               const unsigned *__restrict__ bend, const unsigned *__restrict__ order, Grid3 g, Bins3 bn) {
    const int bin = __builtin_amdgcn_readfirstlane(order[blockIdx.x]);
    const unsigned s0 = bstart[bin], s1 = bend[bin];
    if (s0 >= s1 || s1 - s0 > HEAVY) return;   // empty, or a heavy bin
    spread3_bin<1>(C, F, rot, sval, bin, s0, s1, g, bn, reinterpret_cast<SpreadLds *>(lc_smem));
}

// the phase's heavy bins (a prefix of its order): each block takes bins
// j, j + gridDim.x, ... until the first light one
template <unsigned HEAVY>
__global__ void __launch_bounds__(256 * TEAMS)
k_spread3d_bin_heavy(const float2 *__restrict__ C, float2 *__restrict__ F, const double *__restrict__ rot,
                     const unsigned *__restrict__ sval, const unsigned *__restrict__ bstart,
                     const unsigned *__restrict__ bend, const unsigned *__restrict__ order, unsigned nphase,
                     Grid3 g, Bins3 bn) {
    for (unsigned j = blockIdx.x; j < nphase; j += gridDim.x) {
        const int bin = __builtin_amdgcn_readfirstlane(order[j]);
        const unsigned s0 = bstart[bin], s1 = bend[bin];
        if (s1 - s0 <= HEAVY) break;   // the order is fullest first: the rest are light
        spread3_bin<TEAMS>(C, F, rot, sval, bin, s0, s1, g, bn, reinterpret_cast<SpreadLds *>(lc_smem));
    }
}

__global__ void k_zero_u32(unsigned *p, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

__global__ void k_zero2(float2 *p, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = make_float2(0.f, 0.f);
}

// ---------------------------------------------------------------------------
// pruned line passes between the fine grid and the modes along one axis.
// Array (outer, L, inner); row mode when inner == 1 (nl lines per block),
// otherwise column mode with B consecutive inner indices per block.
// DIR 1 (type 1): in (outer, nf, inner) -> FFT+ -> out (outer, nm, inner),
//                 out[a] = X[m_a mod nf] * corr[a] (* scale, real part if ROUT)
// DIR 2 (type 2): in (outer, nm, inner) (* corr, real if RIN) placed at
//                 m_a mod nf, zeros elsewhere -> FFT- -> out (outer, nf, inner)
// ---------------------------------------------------------------------------
// one FFT of nl lines in LDS: row layout (rowm) or nl = 1 << lsh interleaved
// lines; LC > 0: length LC compiled (unrolled stages), else the runtime plan
template <int SIGN, int NT, int MAXE, int LC>
__device__ __forceinline__ void line_fft(float2 *buf, bool rowm, int nl, int lsh, int L, const FftPlan &plan,
                                         const float2 *__restrict__ tw) {
    if constexpr (LC > 0) {
        if (rowm) fft_lds_ct<float, LC, SIGN, NT, MAXE, false>(buf, nl, 0, tw);
        else fft_lds_ct<float, LC, SIGN, NT, MAXE, true>(buf, nl, lsh, tw);
    } else {
        if (rowm) fft_lds<float, SIGN, NT, MAXE, false>(buf, nl, L, plan, tw);
        else fft_lds<float, SIGN, NT, MAXE, true>(buf, nl, 0, plan, tw);
    }
}

__device__ __forceinline__ int m2f(int a, int nm, int nf) {
    const int m = a - nm / 2;
    return m < 0 ? m + nf : m;
}

template <int DIR, bool RIN, bool ROUT, int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_nu_axis(const void *__restrict__ vin, void *__restrict__ vout, int64_t outer, int64_t inner,
          int nf, int nm, int nl, int lsh, const float *__restrict__ corr, float scale, FftPlan plan,
          const float2 *__restrict__ tw) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) nf = LC;
    const int Lin = DIR == 1 ? nf : nm, Lout = DIR == 1 ? nm : nf;
    const bool rowm = inner == 1;
    int64_t o0, i0;
    int nloc;
    if (rowm) {
        o0 = (int64_t)blockIdx.x * nl;
        i0 = 0;
        nloc = (int)min((int64_t)nl, outer - o0);
    } else {
        o0 = blockIdx.y;
        i0 = (int64_t)blockIdx.x * nl;
        nloc = (int)min((int64_t)nl, inner - i0);
    }
    // element e of local line l: address of (o, e, i)
    auto addr = [&](int l, int e, int L) -> int64_t {
        return rowm ? (o0 + l) * L + e : (o0 * L + e) * inner + i0 + l;
    };
    auto lds = [&](int l, int e) -> int { return rowm ? lds_row(l, e, nf) : lds_col(l, e, nl); };
    if (DIR == 2) {
        for (int idx = threadIdx.x; idx < nl * nf; idx += NT)
            buf[rowm ? swz(idx) : swz(idx)] = make_float2(0.f, 0.f);
        __syncthreads();
    }
    for (int idx = threadIdx.x; idx < nl * Lin; idx += NT) {
        int l, e;
        if (rowm) { l = idx / Lin; e = idx - l * Lin; }
        else { e = idx / nl; l = idx - e * nl; }
        if (l >= nloc) continue;
        const int64_t q = addr(l, e, Lin);
        float2 v = RIN ? make_float2(reinterpret_cast<const float *>(vin)[q], 0.f)
                       : reinterpret_cast<const float2 *>(vin)[q];
        if (DIR == 1) {
            buf[lds(l, e)] = v;
        } else {
            const float c = corr[e];
            buf[lds(l, m2f(e, nm, nf))] = make_float2(v.x * c, v.y * c);
        }
    }
    if (DIR == 1) {
        // lines beyond nloc hold stale LDS: clear them so the FFT reads zeros
        for (int idx = threadIdx.x; idx < nl * nf; idx += NT) {
            int l, e;
            if (rowm) { l = idx / nf; e = idx - l * nf; }
            else { e = idx / nl; l = idx - e * nl; }
            if (l >= nloc) buf[lds(l, e)] = make_float2(0.f, 0.f);
        }
    }
    __syncthreads();
    line_fft<DIR == 1 ? 1 : -1, NT, MAXE, LC>(buf, rowm, nl, lsh, nf, plan, tw);
    for (int idx = threadIdx.x; idx < nl * Lout; idx += NT) {
        int l, e;
        if (rowm) { l = idx / Lout; e = idx - l * Lout; }
        else { e = idx / nl; l = idx - e * nl; }
        if (l >= nloc) continue;
        const int64_t q = addr(l, e, Lout);
        if (DIR == 1) {
            const float2 v = buf[lds(l, m2f(e, nm, nf))];
            const float c = corr[e] * scale;
            if (ROUT) reinterpret_cast<float *>(vout)[q] = v.x * c;
            else reinterpret_cast<float2 *>(vout)[q] = make_float2(v.x * c, v.y * c);
        } else {
            reinterpret_cast<float2 *>(vout)[q] = buf[lds(l, e)];
        }
    }
}

// ---------------------------------------------------------------------------
// detector line transform along one axis with the reference shift maps:
// buf[k] = in[(k + din) mod n]; X = DFT_sign(buf); out[k] = X[(k + dout) mod n]
// Stockham when n is 2^p 3^q, else Bluestein of length Lb:
// X_m = a_m sum_k (x_k a_k) b_{m-k},  a_k = e^{s i pi k^2/n},  b_k = conj(a_k)
// computed as a_m * FFT+(FFT-(x a) * bhat) with bhat = FFT-(b) / Lb.
// ---------------------------------------------------------------------------
template <bool RIN, bool ROUT, int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_det_axis(const void *__restrict__ vin, void *__restrict__ vout, int64_t outer, int64_t inner,
           int n, int nl, int lsh, int din, int dout, int sign, float scale, int blue, FftPlan plan,
           const float2 *__restrict__ tw, const float2 *__restrict__ chirp,
           const float2 *__restrict__ bhat) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    const int L = LC > 0 ? LC : blue ? plan.L : n;
    const bool rowm = inner == 1;
    int64_t o0, i0;
    int nloc;
    if (rowm) {
        o0 = (int64_t)blockIdx.x * nl;
        i0 = 0;
        nloc = (int)min((int64_t)nl, outer - o0);
    } else {
        o0 = blockIdx.y;
        i0 = (int64_t)blockIdx.x * nl;
        nloc = (int)min((int64_t)nl, inner - i0);
    }
    auto addr = [&](int l, int e) -> int64_t {
        return rowm ? (o0 + l) * n + e : (o0 * n + e) * inner + i0 + l;
    };
    auto lds = [&](int l, int e) -> int { return rowm ? lds_row(l, e, L) : lds_col(l, e, nl); };
    for (int idx = threadIdx.x; idx < nl * L; idx += NT) {
        int l, e;
        if (rowm) { l = idx / L; e = idx - l * L; }
        else { e = idx / nl; l = idx - e * nl; }
        float2 v = make_float2(0.f, 0.f);
        if (l < nloc && e < n) {
            int src = e + din;
            if (src >= n) src -= n;
            const int64_t q = addr(l, src);
            v = RIN ? make_float2(reinterpret_cast<const float *>(vin)[q], 0.f)
                    : reinterpret_cast<const float2 *>(vin)[q];
            if (blue) {
                float2 a = chirp[e];
                if (sign < 0) a.y = -a.y;
                v = cmul(v, a);
            }
        }
        buf[lds(l, e)] = v;
    }
    __syncthreads();
    if (!blue) {
        if (sign < 0) line_fft<-1, NT, MAXE, LC>(buf, rowm, nl, lsh, L, plan, tw);
        else line_fft<1, NT, MAXE, LC>(buf, rowm, nl, lsh, L, plan, tw);
    } else {
        line_fft<-1, NT, MAXE, LC>(buf, rowm, nl, lsh, L, plan, tw);
        const float2 *bh = bhat + (sign < 0 ? 0 : L);
        for (int idx = threadIdx.x; idx < nl * L; idx += NT) {
            int l, e;
            if (rowm) { l = idx / L; e = idx - l * L; }
            else { e = idx / nl; l = idx - e * nl; }
            float2 *p = buf + lds(l, e);
            *p = cmul(*p, bh[e]);
        }
        __syncthreads();
        line_fft<1, NT, MAXE, LC>(buf, rowm, nl, lsh, L, plan, tw);
    }
    for (int idx = threadIdx.x; idx < nl * n; idx += NT) {
        int l, e;
        if (rowm) { l = idx / n; e = idx - l * n; }
        else { e = idx / nl; l = idx - e * nl; }
        if (l >= nloc) continue;
        int m = e + dout;
        if (m >= n) m -= n;
        float2 v = buf[lds(l, m)];
        if (blue) {
            float2 a = chirp[m];
            if (sign < 0) a.y = -a.y;
            v = cmul(v, a);
        }
        const int64_t q = addr(l, e);
        if (ROUT) reinterpret_cast<float *>(vout)[q] = v.x * scale;
        else reinterpret_cast<float2 *>(vout)[q] = make_float2(v.x * scale, v.y * scale);
    }
}

bool smooth23(int64_t n) { return is_2_3_smooth(n); }

int fine_size(int64_t n) {
    int64_t f = std::max<int64_t>(2 * n, 2 * W3);
    while (!smooth23(f)) ++f;
    return (int)f;
}

} // namespace

int nufft3d_fine_n(int64_t n) { return fine_size(n); }

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
void det_line_init(Ctx &c, DetLine &d, int n) {
    d.n = n;
    if (n <= LN_NT * LN_ME && fft_make_plan(n, d.plan)) {
        d.blue = false;
        return;
    }
    // any L >= 2n - 1 gives the exact DFT: the smallest 2^p 3^q, or a length
    // with a compiled line FFT when one is within 25% of it
    int64_t L = 2 * (int64_t)n - 1;
    while (!is_2_3_smooth(L)) ++L;
    for (int cl = (int)(2 * (int64_t)n - 1); cl <= L + L / 4 && cl <= 2048; ++cl)
        if (with_line_len(cl, [](auto) {})) {
            L = cl;
            break;
        }
    LC_REQUIRE(L <= LN_NT * LN_ME, "detector transform: width too large");
    LC_REQUIRE(fft_make_plan((int)L, d.plan), "detector transform: no Bluestein length");
    d.blue = true;
    // chirp a_k = e^{+i pi k^2 / n} (the kernel conjugates it for sign -1); bhat
    // for sign s is FFT-(b) / L with b_k = conj(a_k^s) on k and L - k (L >= 2n - 1,
    // so the two runs do not meet), [sign -1 | sign +1]: b is even, so the sign +1
    // table is the conjugate of the sign -1 one
    std::vector<std::complex<double>> ch64, bh64;
    bluestein_tables(n, (int)L, ch64, bh64);
    std::vector<float2> ch(n), bh(2 * L);
    for (int k = 0; k < n; ++k) ch[k] = make_float2((float)ch64[k].real(), (float)ch64[k].imag());
    for (int64_t m = 0; m < L; ++m) {
        bh[m] = make_float2((float)bh64[m].real(), (float)bh64[m].imag());
        bh[L + m] = make_float2((float)bh64[m].real(), (float)-bh64[m].imag());
    }
    d.chirp.alloc(sizeof(float2) * n);
    d.bhat.alloc(sizeof(float2) * 2 * L);
    LC_HIP(hipMemcpyAsync(d.chirp.as(), ch.data(), sizeof(float2) * n, hipMemcpyHostToDevice, c.stream()));
    LC_HIP(hipMemcpyAsync(d.bhat.as(), bh.data(), sizeof(float2) * 2 * L, hipMemcpyHostToDevice, c.stream()));
    c.sync();
}

void nufft3d_init(Ctx &c, Geom3D &g) {
    Nufft3D &u = g.nu;
    const int64_t nm[3] = {g.n1, g.n2, g.n3};
    const double beta = 2.30 * W3;
    u.beta = beta;
    std::vector<float> corr;
    for (int a = 0; a < 3; ++a) {
        u.nf[a] = fine_size(nm[a]);
        LC_REQUIRE(u.nf[a] <= LN_NT * LN_ME, "3-D NUFFT: fine grid too large");
        LC_REQUIRE(fft_make_plan(u.nf[a], u.plan[a]), "3-D NUFFT: fine size not 2^p 3^q");
        u.coff[a] = (int)corr.size();
        corr.resize(corr.size() + nm[a]);
        es_correction((int)nm[a], u.nf[a], W3, beta, corr.data() + u.coff[a]);
    }
    u.corr.alloc(sizeof(float) * corr.size());
    LC_HIP(hipMemcpyAsync(u.corr.as(), corr.data(), sizeof(float) * corr.size(), hipMemcpyHostToDevice,
                          c.stream()));
    c.sync();
    det_line_init(c, u.det_x, (int)g.ncols);
    det_line_init(c, u.det_y, (int)g.nrows);
    u.ready = true;
}

namespace {

Grid3 grid3(const Geom3D &g, bool mask) {
    Grid3 r;
    r.nproj = (int)g.nproj;
    r.nrows = (int)g.nrows;
    r.ncols = (int)g.ncols;
    for (int a = 0; a < 3; ++a) r.nf[a] = g.nu.nf[a];
    r.dX = 2.0 * M_PI / (double)g.ncols;
    r.dY = 2.0 * M_PI / (double)g.nrows;
    r.icols = 1.0 / (double)g.ncols;
    r.irows = 1.0 / (double)g.nrows;
    r.beta = (float)g.nu.beta;
    r.mask = mask ? 1 : 0;
    return r;
}

struct Work3 {
    float2 *C, *F, *V1, *V2;
    // the points' keys and indices (unsorted, sorted), the bins' runs, the
    // bins' launch order and the sorts' scratch
    unsigned *key_a, *key_b, *val_a, *val_b, *bstart, *bend;
    unsigned *okey_a, *okey_b, *oval_a, *order;
    void *sort_tmp;
    size_t sort_bytes;
};

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

Bins3 bins_of(const int nf[3]) {
    const Bins3 bn{{bins_along(nf[0]), bins_along(nf[1]), bins_along(nf[2])}};
    for (int a = 0; a < 3; ++a)
        LC_REQUIRE(nf[a] >= RGN && ceil_div(nf[a], bn.nb[a]) <= BE, "3-D NUFFT: no bins for this fine grid");
    return bn;
}
unsigned count_of(const Bins3 &bn) { return (unsigned)bn.nb[0] * bn.nb[1] * bn.nb[2]; }

// bits of the sort key: bins 0 .. nbins - 1 and nbins for dropped points, above
// the bits of the corner row
int key_bits(unsigned nbins) {
    int b = 1;
    while (b < 32 && (1ull << b) <= nbins) ++b;
    LC_REQUIRE(b + YB <= 32, "3-D NUFFT: too many bins");
    return b + YB;
}

size_t sort_tmp_bytes(int64_t npts, unsigned nbins) {
    size_t tb = 0, to = 0;
    LC_HIP(rocprim::radix_sort_pairs(nullptr, tb, (unsigned *)nullptr, (unsigned *)nullptr, (unsigned *)nullptr,
                                     (unsigned *)nullptr, (size_t)npts, 0, 32, (hipStream_t)0));
    LC_HIP(rocprim::radix_sort_pairs(nullptr, to, (unsigned *)nullptr, (unsigned *)nullptr, (unsigned *)nullptr,
                                     (unsigned *)nullptr, (size_t)nbins, 0, ORDER_BITS, (hipStream_t)0));
    return std::max(tb, to);
}

// bytes of the sorted points' buffers
size_t spread_bytes(int64_t npts, const int nf[3]) {
    const unsigned nbins = count_of(bins_of(nf));
    return 4 * align256(sizeof(unsigned) * (size_t)npts) + 6 * align256(sizeof(unsigned) * (size_t)nbins) +
           align256(sort_tmp_bytes(npts, nbins));
}

// projections that the forward projector sorts at a time: up to 2^27 points
// (2 GiB of keys and indexes; the 23 M points of 360 projections of 89 x 721
// are one range), so its sort's memory and 32-bit indexes bound no sinogram
int64_t range_of(const Geom3D &g) {
    return std::min<int64_t>(g.nproj, std::max<int64_t>(1, ((int64_t)1 << 27) / ((int64_t)g.nrows * g.ncols)));
}

// nsort: projections sorted at a time
Work3 work3(Ctx &c, const Geom3D &g, int64_t nsort) {
    const Nufft3D &u = g.nu;
    const int64_t npts = nsort * g.nrows * g.ncols;
    LC_REQUIRE(npts < (int64_t)UINT32_MAX, "3-D projector: more than 2^32 detector points");
    const size_t bC = align256(sizeof(float2) * (size_t)g.nproj * g.nrows * g.ncols);
    const size_t bF = align256(sizeof(float2) * (size_t)u.nf[0] * u.nf[1] * u.nf[2]);
    const size_t bV1 = align256(sizeof(float2) * (size_t)u.nf[0] * u.nf[1] * g.n3);
    const size_t bV2 = align256(sizeof(float2) * (size_t)u.nf[0] * g.n2 * g.n3);
    const size_t base = bC + bF + bV1 + bV2;
    const unsigned nbins = count_of(bins_of(u.nf));
    const size_t bK = align256(sizeof(unsigned) * (size_t)npts);
    const size_t bB = align256(sizeof(unsigned) * (size_t)nbins);
    Work3 w{};
    char *ws = reinterpret_cast<char *>(c.scratch(4, base + spread_bytes(npts, u.nf)));
    w.C = reinterpret_cast<float2 *>(ws);
    w.F = reinterpret_cast<float2 *>(ws + bC);
    w.V1 = reinterpret_cast<float2 *>(ws + bC + bF);
    w.V2 = reinterpret_cast<float2 *>(ws + bC + bF + bV1);
    char *q = ws + base;
    w.key_a = reinterpret_cast<unsigned *>(q);
    w.key_b = reinterpret_cast<unsigned *>(q + bK);
    w.val_a = reinterpret_cast<unsigned *>(q + 2 * bK);
    w.val_b = reinterpret_cast<unsigned *>(q + 3 * bK);
    q += 4 * bK;
    w.bstart = reinterpret_cast<unsigned *>(q);   // bstart and bend are adjacent
    w.bend = reinterpret_cast<unsigned *>(q + bB);
    w.okey_a = reinterpret_cast<unsigned *>(q + 2 * bB);
    w.okey_b = reinterpret_cast<unsigned *>(q + 3 * bB);
    w.oval_a = reinterpret_cast<unsigned *>(q + 4 * bB);
    w.order = reinterpret_cast<unsigned *>(q + 5 * bB);
    q += 6 * bB;
    w.sort_tmp = q;
    w.sort_bytes = sort_tmp_bytes(npts, nbins);
    return w;
}

// lines per block and grid of a line pass over (outer, L, inner): row mode
// (inner == 1) takes up to 64 whole rows; column mode up to 64 consecutive
// inner indices per block (a power of two for the compiled passes)
struct LineShape {
    int nl, lsh;
    dim3 grid;
};
LineShape line_shape(int64_t outer, int64_t inner, int L, int cap, bool pow2, const char *what) {
    LineShape sh;
    sh.lsh = 0;
    const int most = std::max(1, std::min(cap / L, 64));
    if (inner == 1) {
        sh.nl = most;
        sh.grid = dim3((unsigned)ceil_div(outer, sh.nl));
    } else {
        LC_REQUIRE(outer <= 65535, std::string(what) + ": too many planes");
        if (pow2) {
            while ((2 << sh.lsh) <= most && (1 << sh.lsh) < inner) ++sh.lsh;
            sh.nl = 1 << sh.lsh;
        } else {
            sh.nl = (int)std::max<int64_t>(1, std::min<int64_t>(most, inner));
        }
        sh.grid = dim3((unsigned)ceil_div(inner, sh.nl), (unsigned)outer);
    }
    return sh;
}

// one axis pass of the fine-grid transform
template <int DIR, bool RIN, bool ROUT>
void nu_axis(Ctx &c, const void *in, void *out, int64_t outer, int64_t inner, int nf, int nm,
             const float *corr, float scale, const FftPlan &plan) {
    const float2 *tw = c.twiddles<float>(nf);
    const bool ct = with_line_len(nf, [](auto) {});
    // runtime plans: the smaller block (fewer registers) while a line fits it
    const bool small = nf <= LN_NT * LN_ME_CT;
    const int cap = LN_NT * (small ? LN_ME_CT : LN_ME);
    LC_REQUIRE(nf <= cap, "3-D NUFFT: line too long");
    const LineShape ls = line_shape(outer, inner, nf, cap, ct, "3-D NUFFT");
    const size_t sh = sizeof(float2) * lds_round(ls.nl * nf);
    if (!with_line_len(nf, [&](auto len) {
            hipLaunchKernelGGL((k_nu_axis<DIR, RIN, ROUT, LN_NT, LN_ME_CT, decltype(len)::value>), ls.grid,
                               dim3(LN_NT), sh, c.stream(), in, out, outer, inner, nf, nm, ls.nl, ls.lsh, corr,
                               scale, plan, tw);
        })) {
        if (small)
            hipLaunchKernelGGL((k_nu_axis<DIR, RIN, ROUT, LN_NT, LN_ME_CT, 0>), ls.grid, dim3(LN_NT), sh,
                               c.stream(), in, out, outer, inner, nf, nm, ls.nl, ls.lsh, corr, scale, plan, tw);
        else
            hipLaunchKernelGGL((k_nu_axis<DIR, RIN, ROUT, LN_NT, LN_ME, 0>), ls.grid, dim3(LN_NT), sh,
                               c.stream(), in, out, outer, inner, nf, nm, ls.nl, ls.lsh, corr, scale, plan, tw);
    }
    LC_HIP(hipGetLastError());
}

// detector transform along one axis
template <bool RIN, bool ROUT>
void det_axis(Ctx &c, const DetLine &d, const void *in, void *out, int64_t outer, int64_t inner,
              int din, int dout, int sign, float scale) {
    const int L = d.blue ? d.plan.L : d.n;
    const float2 *tw = c.twiddles<float>(d.plan.L);
    const bool ct = with_line_len(L, [](auto) {});
    const bool small = L <= LN_NT * LN_ME_CT;
    const int cap = LN_NT * (small ? LN_ME_CT : LN_ME);
    LC_REQUIRE(L <= cap, "detector transform: line too long");
    const LineShape ls = line_shape(outer, inner, L, cap, ct, "detector transform");
    const size_t sh = sizeof(float2) * lds_round(ls.nl * L);
    const float2 *ch = d.blue ? d.chirp.as<float2>() : nullptr, *bh = d.blue ? d.bhat.as<float2>() : nullptr;
    if (!with_line_len(L, [&](auto len) {
            hipLaunchKernelGGL((k_det_axis<RIN, ROUT, LN_NT, LN_ME_CT, decltype(len)::value>), ls.grid,
                               dim3(LN_NT), sh, c.stream(), in, out, outer, inner, d.n, ls.nl, ls.lsh, din,
                               dout, sign, scale, d.blue ? 1 : 0, d.plan, tw, ch, bh);
        })) {
        if (small)
            hipLaunchKernelGGL((k_det_axis<RIN, ROUT, LN_NT, LN_ME_CT, 0>), ls.grid, dim3(LN_NT), sh, c.stream(),
                               in, out, outer, inner, d.n, ls.nl, ls.lsh, din, dout, sign, scale, d.blue ? 1 : 0,
                               d.plan, tw, ch, bh);
        else
            hipLaunchKernelGGL((k_det_axis<RIN, ROUT, LN_NT, LN_ME, 0>), ls.grid, dim3(LN_NT), sh, c.stream(), in,
                               out, outer, inner, d.n, ls.nl, ls.lsh, din, dout, sign, scale, d.blue ? 1 : 0,
                               d.plan, tw, ch, bh);
    }
    LC_HIP(hipGetLastError());
}

// orders the points of np projections from p0 on by their bins
// (w.key_b, w.val_b, w.bstart, w.bend); drop: the values of masked points among
// them are cleared there
Bins3 sort_points(Ctx &c, const Geom3D &g, const Work3 &w, const Grid3 &gg, float2 *drop, int64_t p0, int64_t np) {
    const Bins3 bn = bins_of(g.nu.nf);
    const unsigned nbins = count_of(bn);
    const int64_t npts = np * g.nrows * g.ncols;
    const int bits = key_bits(nbins);
    hipLaunchKernelGGL(k_bin_keys, dim3((unsigned)ceil_div(npts, 256)), dim3(256), 0, c.stream(),
                       g.d_rot.as<double>() + 6 * p0, gg, bn, w.key_a, w.val_a, npts, nbins, drop);
    LC_HIP(hipGetLastError());
    size_t tb = w.sort_bytes;
    LC_HIP(rocprim::radix_sort_pairs(w.sort_tmp, tb, w.key_a, w.key_b, w.val_a, w.val_b, (size_t)npts, 0, bits,
                                     c.stream()));
    hipLaunchKernelGGL(k_zero_u32, dim3(1024), dim3(256), 0, c.stream(), w.bstart,
                       (int64_t)(w.bend - w.bstart) + nbins);
    hipLaunchKernelGGL(k_bin_ranges, dim3((unsigned)ceil_div(npts, 256)), dim3(256), 0, c.stream(), w.key_b,
                       npts, w.bstart, w.bend, nbins);
    LC_HIP(hipGetLastError());
    return bn;
}

// Whether the forward projector interpolates npts points unsorted: what that
// takes, by the plane of the fine grid that a point's neighbours in a row walk
// over, against the sort's launches and a region read for every bin, both fitted
// to 14 volumes from 8 x 64^2 to 29 x 721^2 of 3e4 to 2e6 points (the measured
// crossings lie within a tenth of the time).  Forward projection (us, unsorted /
// sorted): 8 x 64^2 0.5 M points 266 / 285, 0.8 M 376 / 349; 16 x 256^2 0.3 M 319 /
// 354, 0.5 M 448 / 422; 5 x 200^2 0.2 M 252 / 301, 0.4 M 405 / 361; 32 x 511^2 0.5 M
// 1090 / 1165, 0.8 M 1396 / 1294; 29 x 721^2 0.6 M 2241 / 2365, 1.5 M 3168 / 2808.
bool interp_direct(int64_t npts, const int nf[3]) {
    const double plane = (double)nf[1] * nf[2];
    const double ns = std::min(0.8, std::max(0.26, 0.42 + 0.13 * std::log2(plane / 65536.0)));   // per point
    return (double)npts * ns * 1e-3 < 175.0 + 0.003 * count_of(bins_of(nf));                     // us
}

// vol -> w.C, nsort projections at a time; sort: leaves the last ones' points
// sorted, for a type 1 to follow
void type2_3d(Ctx &c, const Geom3D &g, const Work3 &w, const float *vol, bool mask, int64_t nsort, bool sort) {
    const Nufft3D &u = g.nu;
    const int n1 = (int)g.n1, n2 = (int)g.n2, n3 = (int)g.n3;
    const float *corr = g.nu.corr.as<float>();
    // z: (n1, n2*n3) real -> (nf0, n2*n3)
    nu_axis<2, true, false>(c, vol, w.V2, 1, (int64_t)n2 * n3, u.nf[0], n1, corr + u.coff[0], 1.0f, u.plan[0]);
    // y: (nf0, n2, n3) -> (nf0, nf1, n3)
    nu_axis<2, false, false>(c, w.V2, w.V1, u.nf[0], n3, u.nf[1], n2, corr + u.coff[1], 1.0f, u.plan[1]);
    // x: rows (nf0*nf1, n3) -> (nf0*nf1, nf2)
    nu_axis<2, false, false>(c, w.V1, w.F, (int64_t)u.nf[0] * u.nf[1], 1, u.nf[2], n3,
                             corr + u.coff[2], 1.0f, u.plan[2]);
    const Grid3 gg = grid3(g, mask);
    const int64_t all = g.nproj * g.nrows * g.ncols;
    if (!sort && interp_direct(all, u.nf)) {
        hipLaunchKernelGGL(k_interp3d_direct, dim3((unsigned)ceil_div(all, 256)), dim3(256), 0, c.stream(), w.F, w.C,
                           g.d_rot.as<double>(), (unsigned)all, gg);
        LC_HIP(hipGetLastError());
        return;
    }
    for (int64_t p0 = 0; p0 < g.nproj; p0 += nsort) {
        const int64_t np = std::min<int64_t>(nsort, g.nproj - p0), npts = np * g.nrows * g.ncols;
        float2 *C = w.C + p0 * g.nrows * g.ncols;
        const Bins3 bn = sort_points(c, g, w, gg, C, p0, np);
        // long runs read a bin's region once; short ones keep a small grid's blocks many
        const unsigned chunk =
            (unsigned)std::min<int64_t>(1024, std::max<int64_t>(1, npts / (4096 * BATCH)) * BATCH);
        hipLaunchKernelGGL(k_interp3d, dim3((unsigned)ceil_div(npts, chunk)), dim3(256), 0, c.stream(), w.F, C,
                           g.d_rot.as<double>() + 6 * p0, w.key_b, w.val_b, w.bend, (unsigned)npts, count_of(bn),
                           chunk, gg, bn);
        LC_HIP(hipGetLastError());
    }
}

// the sorted-bin spread: w.C -> w.F (sorted: the points are already
// in the order of the bins)
template <unsigned HEAVY> void spread3d(Ctx &c, const Geom3D &g, const Work3 &w, const Grid3 &gg, bool sorted) {
    const Nufft3D &u = g.nu;
    const Bins3 bn = sorted ? bins_of(u.nf) : sort_points(c, g, w, gg, nullptr, 0, g.nproj);
    const unsigned nbins = count_of(bn);
    hipLaunchKernelGGL(k_bin_order_keys, dim3(ceil_div(nbins, 256)), dim3(256), 0, c.stream(), w.bstart,
                       w.bend, bn, w.okey_a, w.oval_a, nbins);
    LC_HIP(hipGetLastError());
    size_t tb = w.sort_bytes;
    LC_HIP(rocprim::radix_sort_pairs(w.sort_tmp, tb, w.okey_a, w.okey_b, w.oval_a, w.order, (size_t)nbins, 0,
                                     ORDER_BITS, c.stream()));
    hipLaunchKernelGGL(k_zero2, dim3(2048), dim3(256), 0, c.stream(), w.F,
                       (int64_t)u.nf[0] * u.nf[1] * u.nf[2]);
    LC_HIP(hipGetLastError());
    int64_t first = 0;   // the phase's first entry in the launch order
    int per[3];
    for (int a = 0; a < 3; ++a) per[a] = phases_along(bn.nb[a]);
    for (int ph = 0; ph < per[0] * per[1] * per[2]; ++ph) {
        // phase (rz, ry, rx): the bins whose index along each axis is r mod its phases
        const int r[3] = {ph / (per[1] * per[2]), (ph / per[2]) % per[1], ph % per[2]};
        int nblk = 1;
        for (int a = 0; a < 3; ++a) nblk *= (bn.nb[a] - r[a] + per[a] - 1) / per[a];
        hipLaunchKernelGGL(k_spread3d_bin_heavy<HEAVY>, dim3(std::min(nblk, 256)), dim3(256 * TEAMS),
                           sizeof(SpreadLds) * TEAMS, c.stream(), w.C, w.F, g.d_rot.as<double>(), w.val_b,
                           w.bstart, w.bend, w.order + first, (unsigned)nblk, gg, bn);
        hipLaunchKernelGGL(k_spread3d_bin<HEAVY>, dim3(nblk), dim3(256), sizeof(SpreadLds), c.stream(), w.C, w.F,
                           g.d_rot.as<double>(), w.val_b, w.bstart, w.bend, w.order + first, gg, bn);
        LC_HIP(hipGetLastError());
        first += nblk;
    }
}

// sorted: type2_3d has just run on the same points
void type1_3d(Ctx &c, const Geom3D &g, const Work3 &w, float *vol, bool mask, const double *shifts,
              float scale, bool sorted) {
    const Nufft3D &u = g.nu;
    const int n1 = (int)g.n1, n2 = (int)g.n2, n3 = (int)g.n3;
    const Grid3 gg = grid3(g, mask);
    if (shifts) {
        const int64_t np = (int64_t)g.nproj * g.nrows * g.ncols;
        hipLaunchKernelGGL(k_phase_shift3d, dim3(ceil_div(np, 256)), dim3(256), 0, c.stream(), w.C,
                           shifts, gg, np);
        LC_HIP(hipGetLastError());
    }
    with_heavy3(c.nu3_shape(u.nf), [&](auto heavy) { spread3d<decltype(heavy)::value>(c, g, w, gg, sorted); });
    const float *corr = g.nu.corr.as<float>();
    // x: rows (nf0*nf1, nf2) -> (nf0*nf1, n3)
    nu_axis<1, false, false>(c, w.F, w.V1, (int64_t)u.nf[0] * u.nf[1], 1, u.nf[2], n3,
                             corr + u.coff[2], 1.0f, u.plan[2]);
    // y: (nf0, nf1, n3) -> (nf0, n2, n3)
    nu_axis<1, false, false>(c, w.V1, w.V2, u.nf[0], n3, u.nf[1], n2, corr + u.coff[1], 1.0f, u.plan[1]);
    // z: (nf0, n2*n3) -> (n1, n2*n3) real, scaled
    nu_axis<1, false, true>(c, w.V2, vol, 1, (int64_t)n2 * n3, u.nf[0], n1, corr + u.coff[0], scale,
                            u.plan[0]);
}

void nu3_check(Ctx &c, Geom3D &g) {
    if (!g.nu.ready) nufft3d_init(c, g);
}

} // namespace

// forward (src/projection.cpp:42-64): vol {n1, N, N} -> proj {nproj, nrows, ncols}
void forward3d_dev(Ctx &c, Geom3D &g, const float *vol, float *proj) {
    nu3_check(c, g);
    const int64_t nsort = range_of(g);
    const Work3 w = work3(c, g, nsort);
    type2_3d(c, g, w, vol, true, nsort, false);
    const int nr = (int)g.nrows, nc = (int)g.ncols;
    // fftshift2 -> ifft2 -> ifftshift2 along x then y; real part / (nrows ncols)
    det_axis<false, false>(c, g.nu.det_x, w.C, w.C, g.nproj * nr, 1, nc / 2, nc / 2 + (nc & 1), 1, 1.0f);
    det_axis<false, true>(c, g.nu.det_y, w.C, proj, g.nproj, nc, nr / 2, nr / 2 + (nr & 1), 1,
                          1.0f / ((float)nr * (float)nc));
}

// backproj (src/projection.cpp:71-131): proj -> vol; shifts (dx, dy) per
// projection or nullptr
void backproj3d_dev(Ctx &c, Geom3D &g, const float *proj, float *vol, const double *shifts) {
    nu3_check(c, g);
    const Work3 w = work3(c, g, g.nproj);
    const int nr = (int)g.nrows, nc = (int)g.ncols;
    // fftshift2 -> fft2 -> ifftshift2 along x then y
    det_axis<true, false>(c, g.nu.det_x, proj, w.C, g.nproj * nr, 1, nc / 2, nc / 2 + (nc & 1), -1, 1.0f);
    det_axis<false, false>(c, g.nu.det_y, w.C, w.C, g.nproj, nc, nr / 2, nr / 2 + (nr & 1), -1, 1.0f);
    type1_3d(c, g, w, vol, true, shifts, 1.0f / ((float)nr * (float)nc), false);
}

// sysmat(x, grid) (src/gradient.cpp:32-41): Re(T1(T2 x)) / (nrows ncols), no mask
void sysmat3d_nufft_dev(Ctx &c, Geom3D &g, const float *x, float *y) {
    nu3_check(c, g);
    const Work3 w = work3(c, g, g.nproj);
    type2_3d(c, g, w, x, false, g.nproj, true);
    type1_3d(c, g, w, y, false, nullptr, 1.0f / ((float)g.nrows * (float)g.ncols), true);
}

// device bytes of a 3-D back-projection's spread beyond the fine grid (the sort
// of the points by bin and its scratch)
size_t nufft3d_spread_bytes(int64_t npts, const int nf[3]) { return spread_bytes(npts, nf); }

int nufft3d_num_shapes() { return N_SHAPES3; }

// Times the back-projection of g's grid with every compiled choice of the
// spread (zero projections: the spread's work depends on where the points
// fall, not on their values), installs the fastest in c.nu3_tuning for g's
// fine-grid shape and returns its index (best_ms: one back-projection).
int nufft3d_autotune(Ctx &c, Geom3D &g, double *best_ms) {
    nu3_check(c, g);
    const int64_t np = g.nproj * g.nrows * g.ncols, nv = g.n1 * g.n2 * g.n3;
    DBuf proj(sizeof(float) * (size_t)np), vol(sizeof(float) * (size_t)nv);
    LC_HIP(hipMemsetAsync(proj.as(), 0, sizeof(float) * (size_t)np, c.stream()));
    const std::array<int, 3> key{g.nu.nf[0], g.nu.nf[1], g.nu.nf[2]};
    const auto saved = c.nu3_tuning;
    hipEvent_t e0, e1;
    LC_HIP(hipEventCreate(&e0));
    LC_HIP(hipEventCreate(&e1));
    int best = 0;
    float tbest = 1e30f;
    try {
        for (int i : {0, 2}) {
            c.nu3_tuning[key] = i;
            backproj3d_dev(c, g, proj.as<float>(), vol.as<float>(), nullptr);   // warm-up
            LC_HIP(hipEventRecord(e0, c.stream()));
            for (int r = 0; r < 2; ++r) backproj3d_dev(c, g, proj.as<float>(), vol.as<float>(), nullptr);
            LC_HIP(hipEventRecord(e1, c.stream()));
            LC_HIP(hipEventSynchronize(e1));
            float ms = 0.f;
            LC_HIP(hipEventElapsedTime(&ms, e0, e1));
            if (ms / 2 < tbest) {
                tbest = ms / 2;
                best = i;
            }
        }
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        c.nu3_tuning = saved;
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    c.nu3_tuning = saved;
    c.nu3_tuning[key] = best;
    if (best_ms) *best_ms = tbest;
    return best;
}

} // namespace lc
