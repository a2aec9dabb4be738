// 2-D polar-grid NUFFT projectors on gfx950 (forward2d / backproj2d,
// src/projection.cpp:146-182).
//
// Type 1 (backproj2d):  f_m = sum_j c_j exp(+i m.w_j),   w_j = r_k (cos th_i, sin th_i)
// Type 2 (forward2d):   c_j = sum_m f_m exp(-i m.w_j)
// with modes m in [-N/2, N/2) (CMCL order; include/nufft.h:64-95).  The
// method is the exponential-of-semicircle NUFFT (Barnett, Magland and
// af Klinteberg, SIAM J. Sci. Comput. 41(5), 2019): spread / interpolate
// with psi(u) = exp(beta (sqrt(1 - (2u/w)^2) - 1)) on a fine grid of nf = 2N
// (rounded to 2^p 3^q) cells, FFT the fine grid, divide by the kernel's
// Fourier transform.  The fine grid is indexed with its centre at nf/2 so a
// radial line of points is a straight segment of cells; the resulting
// (-1)^m phase is folded into the correction factors.
//
// Spreading is deterministic: every tile of the fine grid gathers the points
// that reach it, in a fixed order.
#include <algorithm>
#include <cmath>
#include <complex>

#include <rocprim/device/device_radix_sort.hpp>

#include "lc_engine.hpp"


namespace lc {

extern __shared__ __align__(16) char lc_smem[];

constexpr int NU_W = 8;        // kernel width (cells)
using f32x4 = __attribute__((ext_vector_type(4))) float;

// exp(beta (sqrt(1 - z^2) - 1)) for |z| < 1, else 0.  The hardware square
// root (within 1 ulp; s lies in (0, 1]) instead of the correctly rounded
// sequence: one instruction instead of about fifteen, a relative weight
// error near 1e-6, inside the kernel's own approximation error
__device__ __forceinline__ float es_kernel(float z, float beta) {
    const float s = 1.0f - z * z;
    return s > 0.0f ? __expf(beta * (__builtin_amdgcn_sqrtf(s) - 1.0f)) : 0.0f;
}

// ---------------------------------------------------------------------------
// detector transforms along each sinogram row (length n = nrad)
// backproj: G = ifftshift1(fft1(fftshift1(y)))      (complex out)
// forward:  y = Re(fftshift1(ifft1(ifftshift1(C)))) / n
// fftshift: out[k] = in[(k + n/2) % n]; ifftshift: d = n/2 + (n odd)
// ---------------------------------------------------------------------------
// LC > 0 (every kernel of this file): line length LC compiled, with unrolled
// stages (fft_lds_ct); 0: the runtime plan
template <int SIGN, int NT, int MAXE, bool LFAST, int LC>
__device__ __forceinline__ void nu_fft(float2 *buf, int nl, int L, int lsh, const FftPlan &plan,
                                       const float2 *__restrict__ tw) {
    if constexpr (LC > 0) fft_lds_ct<float, LC, SIGN, NT, MAXE, LFAST>(buf, nl, lsh, tw);
    else fft_lds<float, SIGN, NT, MAXE, LFAST>(buf, nl, LFAST ? 0 : L, plan, tw);
}

template <int SIGN, int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_det_fft(const float *__restrict__ real_in, const float2 *__restrict__ cplx_in,
          float2 *__restrict__ cplx_out, float *__restrict__ real_out, int nrows, int n, int nl,
          FftPlan plan, const float2 *__restrict__ tw, float scale) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) n = LC;
    // blocks never straddle slices (blockIdx.y = slice, nrows rows each): a
    // row's place in its block, which its rounding depends on, is then the
    // same whether the slice is transformed alone or inside a stack
    const int lrow0 = blockIdx.x * nl;
    const int nloc = min(nl, nrows - lrow0);
    const int64_t row0 = (int64_t)blockIdx.y * nrows + lrow0;
    const int dfw = n / 2, dinv = n / 2 + (n & 1);
    // input shift: fftshift for backproj (SIGN -1), ifftshift for forward (+1)
    const int din = SIGN < 0 ? dfw : dinv;
    const int dout = SIGN < 0 ? dinv : dfw;
    for (int idx = threadIdx.x; idx < nl * n; idx += NT) {
        const int l = idx / n, k = idx - l * n;
        float2 v = make_float2(0.f, 0.f);
        if (l < nloc) {
            int src = k + din;
            if (src >= n) src -= n;
            const int64_t q = (row0 + l) * n + src;
            v = SIGN < 0 ? make_float2(real_in[q], 0.f) : cplx_in[q];
        }
        buf[lds_row(l, k, n)] = v;
    }
    __syncthreads();
    nu_fft<SIGN, NT, MAXE, false, LC>(buf, nl, n, 0, plan, tw);
    for (int idx = threadIdx.x; idx < nloc * n; idx += NT) {
        const int l = idx / n, k = idx - l * n;
        int src = k + dout;
        if (src >= n) src -= n;
        const float2 v = buf[lds_row(l, src, n)];
        const int64_t q = (row0 + l) * n + k;
        if (SIGN < 0) cplx_out[q] = v;
        else real_out[q] = v.x * scale;
    }
}

// The same for widths that are not 2^p 3^q (65 to 2048): Bluestein's algorithm
// with a power-of-two length L >= 2 n - 1, in FP64 (as the direct sum below
// accumulates; the FP64 rate equals that of unpacked FP32 and the rows are few):
//   X_m = a_m sum_k (x_k a_k) b_{m-k},  a_k = e^{SIGN i pi k^2 / n},  b_k = conj(a_k)
// chirp: e^{i pi k^2 / n}; bhat: FFT-(b) / L for SIGN -1 (b is even, so the
// SIGN +1 spectrum is its conjugate).  Rows per block and slices as above.
// 1440 rows of 511: 25 us against 516 us for the direct sum.
template <int SIGN, int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_det_blue(const float *__restrict__ real_in, const float2 *__restrict__ cplx_in,
           float2 *__restrict__ cplx_out, float *__restrict__ real_out, int nrows, int n, int nl,
           FftPlan plan, const double2 *__restrict__ tw, const double2 *__restrict__ chirp,
           const double2 *__restrict__ bhat, float scale) {
    double2 *buf = reinterpret_cast<double2 *>(lc_smem);
    const int L = LC > 0 ? LC : plan.L;
    const int lrow0 = blockIdx.x * nl;
    const int nloc = min(nl, nrows - lrow0);
    const int64_t row0 = (int64_t)blockIdx.y * nrows + lrow0;
    const int dfw = n / 2, dinv = n / 2 + (n & 1);
    const int din = SIGN < 0 ? dfw : dinv, dout = SIGN < 0 ? dinv : dfw;
    auto phase = [&](int k) { return SIGN < 0 ? cconj(chirp[k]) : chirp[k]; };
    for (int idx = threadIdx.x; idx < nl * L; idx += NT) {
        const int l = idx / L, k = idx - l * L;
        double2 v = make_double2(0.0, 0.0);
        if (l < nloc && k < n) {
            int src = k + din;
            if (src >= n) src -= n;
            const int64_t q = (row0 + l) * n + src;
            if constexpr (SIGN < 0) v = cscale(phase(k), (double)real_in[q]);
            else v = cmul(phase(k), make_double2(cplx_in[q].x, cplx_in[q].y));
        }
        buf[lds_row(l, k, L)] = v;
    }
    __syncthreads();
    auto fft = [&](auto sign) {
        constexpr int SG = decltype(sign)::value;
        if constexpr (LC > 0) fft_lds_ct<double, LC, SG, NT, MAXE, false>(buf, nl, 0, tw);
        else fft_lds<double, SG, NT, MAXE, false>(buf, nl, L, plan, tw);
    };
    fft(std::integral_constant<int, -1>{});
    for (int idx = threadIdx.x; idx < nl * L; idx += NT) {
        const int l = idx / L, k = idx - l * L;
        double2 *p = buf + lds_row(l, k, L);
        *p = cmul(*p, SIGN < 0 ? bhat[k] : cconj(bhat[k]));
    }
    __syncthreads();
    fft(std::integral_constant<int, 1>{});
    for (int idx = threadIdx.x; idx < nloc * n; idx += NT) {
        const int l = idx / n, k = idx - l * n;
        int src = k + dout;
        if (src >= n) src -= n;
        const double2 v = cmul(buf[lds_row(l, src, L)], phase(src));
        const int64_t q = (row0 + l) * n + k;
        if constexpr (SIGN < 0) cplx_out[q] = make_float2((float)v.x, (float)v.y);
        else real_out[q] = (float)v.x * scale;
    }
}

// direct DFT for widths that are not 2^p 3^q, up to 64 or above 2048, and for
// all above 4096
template <int SIGN>
__global__ void k_det_dft(const float *__restrict__ real_in, const float2 *__restrict__ cplx_in,
                          float2 *__restrict__ cplx_out, float *__restrict__ real_out, int nrows,
                          int n, const float2 *__restrict__ tw, float scale) {
    const int row = blockIdx.x;   // grid: one block per row
    const int dfw = n / 2, dinv = n / 2 + (n & 1);
    const int din = SIGN < 0 ? dfw : dinv, dout = SIGN < 0 ? dinv : dfw;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        // output index k reads transform bin kk
        int kk = k + dout;
        if (kk >= n) kk -= n;
        double re = 0.0, im = 0.0;
        for (int j = 0; j < n; ++j) {
            int src = j + din;
            if (src >= n) src -= n;
            const int64_t q = (int64_t)row * n + src;
            const float2 v = SIGN < 0 ? make_float2(real_in[q], 0.f) : cplx_in[q];
            float2 w = tw[(int)(((int64_t)j * kk) % n)];
            if (SIGN > 0) w.y = -w.y;
            re += (double)v.x * w.x - (double)v.y * w.y;
            im += (double)v.x * w.y + (double)v.y * w.x;
        }
        const int64_t q = (int64_t)row * n + k;
        if (SIGN < 0) cplx_out[q] = make_float2((float)re, (float)im);
        else real_out[q] = (float)re * scale;
    }
}

// ---------------------------------------------------------------------------
// Type-1 spreading by output tiles.  A point's corner is its first footprint
// cell, ceil(g - 4) per axis, taken modulo nf.  The geometry holds the points
// sorted by 8 x 8 bins of corners (row major; the points do not depend on the
// data, so nufft2d_order sorts them once), so a tile of 16 x 16 cells of
// the fine grid finds the points that reach it (corners from 7 cells before it
// to its end) in one or two runs per row of bins.  It takes them in that order
// and writes its cells once: no clearing, no adding into the grid, no order
// between tiles, any fine-grid size, and a slice's sums do not depend on the
// rest of the stack.
//
// A tile is a matrix product: with wy, wx a point's 8 weights per axis placed
// in 16 slots, zero elsewhere,
//   tile[y][x] = sum_p wy_p[y] (c_p wx_p[x])
// which runs on FP32 MFMA tiles (v_mfma_f32_16x16x4_f32: lane l holds
// A[l & 15][l >> 4], B[l >> 4][l & 15] and, in register q,
// D[4 (l >> 4) + q][l & 15]), real and imaginary part apart, four points per
// instruction.  A wave computes the weights of 64 points into LDS tables and
// uses them for up to SC slices of the stack.  A block's four waves take a tile
// each; a tile of more than HEAVY points (near the k-space origin every angle
// passes) gets the whole block, each wave taking a part of the points.  The
// tiles by their number of points, fullest first, are part of the geometry too.
// 8 slices of 1024^2 from 720 angles: 310 us, against 763 us (and a 270 us sort
// and a 40 us clearing per call) for a wave per bin adding each point's cells
// to an LDS region that is then added to the grid in four phases.  The slices
// of a wave are a compile-time number: with a run-time bound inside the product
// loop the sums moved between register files and the spread took 423 us.
// ---------------------------------------------------------------------------
constexpr int CB = 8;                       // corner bin edge
constexpr int TE = 16;                      // tile edge, that of an MFMA tile (tiles of 32 rows took 1.1 to
                                            // 1.5 times as long at each of 14 sizes)
constexpr int TAB = 64;                     // points per table
constexpr int TS = 17;                      // row stride of a 16-slot table
constexpr int SW = 4;                       // waves per block
constexpr int HEAVY = 512;                  // points of the fullest light tile (1024: 253 us in place of 231
                                            // for 16 slices of 256^2 from 360 angles, 2048: 310 us)

struct Grid2 {
    int nang, nrad, nf;
    int nb;                    // corner bins per edge, ceil(nf / CB)
    double dr;                 // 2 pi / nrad
    double sc;                 // nf / (2 pi): radians -> cells
    double inrad;              // 1 / nrad
    float beta;
};

// a / b for inv = 1.0 / b: the FP64 product is within one of the quotient
__device__ __forceinline__ int div_by(int a, int b, double inv) {
    const int q = (int)((double)a * inv), r = a - q * b;
    return r < 0 ? q - 1 : r >= b ? q + 1 : q;
}

// fine-grid corner of point p of a slice, taken modulo nf, and the offset of
// its cell 4 from the point, in [0, 1), per axis
struct Foot2 {
    int ly, lx;
    double dy, dx;
    float fy, fx;   // rounded
};
__device__ __forceinline__ Foot2 foot2(double2 t, int k, const Grid2 &g) {   // t: (cos, sin), k: radial index
    // the fused multiply-adds are explicit, so the kernel that sorts the points
    // and the one that spreads them take the same corner: positions that are
    // whole numbers up to rounding are common (angles 0 and pi / 2 with nrad = N),
    // and one on the two sides of the periodic edge would be lost
    const double r = __builtin_fma((double)k + 0.5, g.dr, -M_PI);
    const double gx = __builtin_fma(g.sc * r, t.x, 0.5 * g.nf), gy = __builtin_fma(g.sc * r, t.y, 0.5 * g.nf);
    const double hw = 0.5 * NU_W;
    Foot2 f;
    f.lx = (int)ceil(gx - hw);
    f.ly = (int)ceil(gy - hw);
    f.dx = (double)(f.lx + NU_W / 2) - gx;
    f.dy = (double)(f.ly + NU_W / 2) - gy;
    f.fx = (float)f.dx;
    f.fy = (float)f.dy;
    f.lx += f.lx < 0 ? g.nf : 0;     // |r| <= pi: a corner lies in [-4, nf - 3]
    f.ly += f.ly < 0 ? g.nf : 0;
    f.lx -= f.lx >= g.nf ? g.nf : 0;
    f.ly -= f.ly >= g.nf ? g.nf : 0;
    return f;
}

__device__ __forceinline__ Foot2 foot2(const double2 *__restrict__ cs, const Grid2 &g, int p) {
    const int ang = div_by(p, g.nrad, g.inrad);
    return foot2(cs[ang], p - ang * g.nrad, g);
}

// key[p] = corner bin of point p, val[p] = p
__global__ void k_bin2_keys(const double2 *__restrict__ cs, Grid2 g, unsigned *__restrict__ key,
                            unsigned *__restrict__ val, int npts) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npts) return;
    const Foot2 f = foot2(cs, g, p);
    key[p] = (unsigned)((f.ly / CB) * g.nb + f.lx / CB);
    val[p] = (unsigned)p;
}

__global__ void k_zero_i32(int *p) { p[threadIdx.x] = 0; }

// start[b] = first sorted point of bin b or a later one, b = 0 .. nbins
__global__ void k_bin2_starts(const unsigned *__restrict__ skey, int npts, int *__restrict__ start, int nbins) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nbins) return;
    int lo = 0, hi = npts;
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (skey[mid] < (unsigned)b) lo = mid + 1;
        else hi = mid;
    }
    start[b] = lo;
}

// The corner bins that reach cells [c0, c0 + n) of an axis (n <= 16, 7 corners
// before them): the bins lo .. hi of the grid itself (image 0, corners as they
// are) and, for the first tile, the last bins (image 1, corners less nf).
__device__ __forceinline__ void tile_bins(int c0, int n, int nf, int image, int &lo, int &hi) {
    if (image == 0) {
        lo = (c0 >= NU_W - 1 ? c0 - (NU_W - 1) : 0) / CB;
        hi = (c0 + n - 1) / CB;
    } else {
        lo = (nf + c0 - (NU_W - 1)) / CB;
        hi = c0 < NU_W - 1 ? (nf - 1) / CB : -1;
    }
}

// the runs of sorted points of a tile, walked in a fixed order
template <typename F> __device__ __forceinline__ void tile_runs(int y0, int x0, int nf, int nb, F &&run) {
    for (int iy = 1; iy >= 0; --iy) {
        int yl, yh;
        tile_bins(y0, min(nf - y0, TE), nf, iy, yl, yh);
        for (int by = yl; by <= yh; ++by)
            for (int ix = 1; ix >= 0; --ix) {
                int xl, xh;
                tile_bins(x0, min(nf - x0, TE), nf, ix, xl, xh);
                if (xl <= xh) run(by * nb + xl, by * nb + xh + 1, iy ? nf : 0, ix ? nf : 0);
            }
    }
}
// key[t] = 2^31 - 1 - points of tile t, val[t] = t; heavy counts the tiles of more than HEAVY
__global__ void k_tile_keys(const int *__restrict__ start, unsigned *__restrict__ key, int *__restrict__ val,
                            int *__restrict__ heavy, int ntiles, int ntx, int nf, int nb) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    int n = 0;
    tile_runs(t / ntx * TE, t % ntx * TE, nf, nb, [&](int b0, int b1, int, int) { n += start[b1] - start[b0]; });
    key[t] = 0x7fffffffu - (unsigned)n;
    val[t] = t;
    if (n > HEAVY) atomicAdd(heavy, 1);
}
// most runs of a tile: its own rows of bins and the wrapped ones, in two pieces
constexpr int MAX_RUNS = 2 * ((TE + NU_W - 2) / CB + 2 + 2);

// (a multiple of 16 bytes: every wave's tables start where 16-byte accesses may)
template <int SC> struct alignas(16) SpreadLds2 {
    float x[TAB * TS], y[TAB * TS];
    float2 c[SC][TAB];
    int rbeg[MAX_RUNS], rpos[MAX_RUNS + 1], roff[MAX_RUNS];
};

// spreads tile `tile` of slices s0 .. s0 + SC - 1 with one wave, or with the
// block's SW waves (TEAM)
template <int SC, bool TEAM>
__device__ __forceinline__ void spread2_tile(const float2 *__restrict__ C, float2 *__restrict__ fine,
                                             const double2 *__restrict__ cs, const unsigned *__restrict__ sval,
                                             const int *__restrict__ start, int tile, int s0, int ntx,
                                             const Grid2 &g, SpreadLds2<SC> *lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ty = tile / ntx, y0 = ty * TE, x0 = (tile - ty * ntx) * TE;
    const int npts = g.nang * g.nrad;
    SpreadLds2<SC> &L = lds[wave];
    // the runs: first sorted point, position of it in the tile's sequence, image
    int nr = 0, total = 0;
    tile_runs(y0, x0, g.nf, g.nb, [&](int b0, int b1, int oy, int ox) {
        const int a = start[b0], n = start[b1] - a;
        if (lane == 0) {
            L.rbeg[nr] = a;
            L.rpos[nr] = total;
            L.roff[nr] = (oy ? 1 : 0) | (ox ? 2 : 0);
        }
        total += n;
        ++nr;
    });
    wave_lds_fence();
    f32x4 tr[SC], ti[SC];
#pragma unroll
    for (int s = 0; s < SC; ++s) tr[s] = ti[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    // wave w of a team takes the w-th part of the sequence, in order
    constexpr int NW = TEAM ? SW : 1;
    const int per = ((total + NW - 1) / NW + TAB - 1) / TAB * TAB;
    const int ws = TEAM ? min(total, wave * per) : 0, we = min(total, ws + per);
    const int n = lane & 15, k4 = lane >> 4;
    const float ihw = 1.0f / (0.5f * NU_W);
    // the sequence's points, their angles and values are fetched a table ahead
    auto index = [&](int base, int &im) -> int {
        const int i = min(base + lane, we - 1);
        int r = 0;
        while (r + 1 < nr && i >= L.rpos[r + 1]) ++r;   // an empty run starts where the next one does
        im = L.roff[r];
        return (int)sval[L.rbeg[r] + (i - L.rpos[r])];
    };
    int im = 0, k = 0;
    double2 t = make_double2(0.0, 0.0);
    float2 cv[SC];
    auto fetch = [&](int p) {
        const int ang = div_by(p, g.nrad, g.inrad);
        k = p - ang * g.nrad;
        t = cs[ang];
#pragma unroll
        for (int s = 0; s < SC; ++s)
            cv[s] = C[(int64_t)(s0 + s) * npts + p];
    };
    if (ws < we) fetch(index(ws, im));
    for (int base = ws; base < we; base += TAB) {
        const bool ok = base + lane < we, more = base + TAB < we;
        int imn = 0, pn = 0;
        if (more) pn = index(base + TAB, imn);
        const Foot2 f = foot2(t, k, g);
        const int oy = f.ly - ((im & 1) ? g.nf : 0) - y0, ox = f.lx - ((im & 2) ? g.nf : 0) - x0;
        wave_lds_fence();   // the previous table is read
#pragma unroll
        for (int s = 0; s < SC; ++s)
            L.c[s][lane] = ok ? cv[s] : make_float2(0.f, 0.f);
        // the 8 weights per axis fall on distinct slots modulo 8
#pragma unroll
        for (int q = 0; q < NU_W; ++q) {
            const int dx = (q - ox) & (NU_W - 1), dy = (q - oy) & (NU_W - 1);
            const float wx = es_kernel(((float)(dx - NU_W / 2) + f.fx) * ihw, g.beta);
            const float wy = es_kernel(((float)(dy - NU_W / 2) + f.fy) * ihw, g.beta);
#pragma unroll
            for (int sl = q; sl < TE; sl += NU_W) {
                L.x[lane * TS + sl] = (ok && sl == ox + dx) ? wx : 0.f;
                L.y[lane * TS + sl] = sl == oy + dy ? wy : 0.f;
            }
        }
        wave_lds_fence();
        if (more) fetch(pn);
        im = imn;
        f32x4 ar[SC], ai[SC];   // this table's sums (short rounding chains)
#pragma unroll
        for (int s = 0; s < SC; ++s) ar[s] = ai[s] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int ng = (min(TAB, we - base) + 3) >> 2;
        for (int gr = 0; gr < ng; ++gr) {
            const int pt = 4 * gr + k4;
            const float wx = L.x[pt * TS + n], wy = L.y[pt * TS + n];
#pragma unroll
            for (int s = 0; s < SC; ++s) {
                const float2 c = L.c[s][pt];
                ar[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wy, wx * c.x, ar[s], 0, 0, 0);
                ai[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wy, wx * c.y, ai[s], 0, 0, 0);
            }
        }
#pragma unroll
        for (int s = 0; s < SC; ++s) {
            tr[s] += ar[s];
            ti[s] += ai[s];
        }
    }
    auto put = [&](int s, const f32x4 &vr, const f32x4 &vi) {
        float2 *fs = fine + (int64_t)(s0 + s) * g.nf * g.nf;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int y = y0 + 4 * k4 + q, x = x0 + n;
            if (y < g.nf && x < g.nf) fs[(int64_t)y * g.nf + x] = make_float2(vr[q], vi[q]);
        }
    };
    if constexpr (!TEAM) {
#pragma unroll
        for (int s = 0; s < SC; ++s) put(s, tr[s], ti[s]);
    } else {
        // summed in wave order, through the tables' space
        static_assert(sizeof(L.x) >= sizeof(f32x4) * 2 * 64, "the exchange fits the tables");
        static_assert(alignof(SpreadLds2<SC>) >= alignof(f32x4), "and starts where f32x4 may, in every wave");
#pragma unroll
        for (int s = 0; s < SC; ++s) {
            __syncthreads();
            f32x4 *ex = reinterpret_cast<f32x4 *>(L.x);   // [re, im][lane]
            ex[lane] = tr[s];
            ex[64 + lane] = ti[s];
            __syncthreads();
            if (wave == s % SW) {
                const f32x4 *e0 = reinterpret_cast<const f32x4 *>(lds[0].x);
                f32x4 vr = e0[lane], vi = e0[64 + lane];
                for (int v = 1; v < SW; ++v) {
                    const f32x4 *ev = reinterpret_cast<const f32x4 *>(lds[v].x);
                    vr += ev[lane];
                    vi += ev[64 + lane];
                }
                put(s, vr, vi);
            }
        }
    }
}

// order: the tiles, fullest first; the first nheavy take a block each, the
// others a wave each.  grid.y: SC slices each, from slice `first`
template <int SC>
__global__ void __launch_bounds__(64 * SW)
k_spread2d(const float2 *__restrict__ C, float2 *__restrict__ fine, const double2 *__restrict__ cs,
           const unsigned *__restrict__ sval, const int *__restrict__ start, const int *__restrict__ order,
           int ntiles, int nheavy, int first, int ntx, Grid2 g) {
    __shared__ SpreadLds2<SC> lds[SW];
    const int s0 = first + blockIdx.y * SC, b = blockIdx.x;
    if (b < nheavy) {
        spread2_tile<SC, true>(C, fine, cs, sval, start, __builtin_amdgcn_readfirstlane(order[b]), s0, ntx, g, lds);
        return;
    }
    const int t = nheavy + (b - nheavy) * SW + (int)(threadIdx.x >> 6);
    if (t >= ntiles) return;   // whole wave (no barrier below)
    spread2_tile<SC, false>(C, fine, cs, sval, start, __builtin_amdgcn_readfirstlane(order[t]), s0, ntx, g, lds);
}

// ---------------------------------------------------------------------------
// Type-2 interpolation.  A wave takes PW consecutive points of a slice: lane l
// first finds the footprint and the weights of point l, then the wave takes
// the points two at a time, 32 lanes each: 8 rows x 4 lanes of two adjacent
// cells, so a footprint row is one 64-byte piece read by 16-byte loads.  (One
// lane per point reads the same cells as 64 8-byte loads whose lanes all fall
// on different cache lines.)  The 32 lanes are summed in a fixed order.
// 4 slices of 511^2, 360 x 511 points: 38 us against 201 us with a lane per point.
// PW is 64, or 16 where that leaves too few waves (type2; the same sums): a
// forward projection of 64^2 from 60 angles 52.6 -> 43.9 us (50.6 with a lane
// per point), 512^2 from 360 66.1 -> 58.8 us (2880 waves of 64), but two such
// slices 68.4 -> 72.1 us (5760).
// ---------------------------------------------------------------------------
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));   // two cells

// v summed over 32 lanes; valid in the last 16 of them
__device__ __forceinline__ float sum32(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, true));   // row_ror:1
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, true));
    // rows 1 and 3 add the row before them (row_bcast:15)
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xa, 0xf, false));
}

constexpr int IW = 4;                       // waves per interpolation block
template <int PW>                           // points of a wave
__global__ void __launch_bounds__(64 * IW)
k_interp2d(const float2 *__restrict__ fine, float2 *__restrict__ C, const double2 *__restrict__ cs, Grid2 g,
           int npts) {
    constexpr int XW = 10, YW = 9;          // row strides of the weight tables
    __shared__ __align__(16) float tx[IW][64 * XW], ty[IW][64 * YW];
    __shared__ int2 tpos[IW][64];
    __shared__ float2 res[IW][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int base = (blockIdx.x * IW + wave) * PW;
    if (base >= npts) return;   // whole wave (no barrier below)
    float *X = tx[wave], *Y = ty[wave];
    const int p = base + lane;
    const Foot2 f = foot2(cs, g, min(p, npts - 1));
    const float ihw = 1.0f / (0.5f * NU_W);
#pragma unroll
    for (int d = 0; d < NU_W; ++d) {
        X[lane * XW + d] = es_kernel((float)((double)(d - NU_W / 2) + f.dx) * ihw, g.beta);
        Y[lane * YW + d] = es_kernel((float)((double)(d - NU_W / 2) + f.dy) * ihw, g.beta);
    }
    tpos[wave][lane] = make_int2(f.lx, f.ly);
    const bool wrap = __ballot(lane < PW && f.lx + NU_W > g.nf) != 0;   // a footprint row crosses the edge
    wave_lds_fence();
    const float2 *fs = fine + (int64_t)blockIdx.y * g.nf * g.nf;
    const int half = lane >> 5, r = (lane >> 2) & 7, c2 = 2 * (lane & 3);
    auto point = [&](int q, auto edge) {
        const int2 l = tpos[wave][q];
        const float2 wx = *reinterpret_cast<const float2 *>(X + q * XW + c2);
        const float wy = Y[q * YW + r];
        int yy = l.y + r, xx = l.x + c2;
        yy -= yy >= g.nf ? g.nf : 0;
        const float2 *row = fs + (int64_t)yy * g.nf;
        f32x4u v;
        if constexpr (decltype(edge)::value) {
            int x1 = xx + 1;
            xx -= xx >= g.nf ? g.nf : 0;
            x1 -= x1 >= g.nf ? g.nf : 0;
            const float2 a = row[xx], b = row[x1];
            v = f32x4u{a.x, a.y, b.x, b.y};
        } else {
            v = *reinterpret_cast<const f32x4u *>(row + xx);
        }
        const float re = sum32(wy * (wx.x * v.x + wx.y * v.z)), im = sum32(wy * (wx.x * v.y + wx.y * v.w));
        if ((lane & 31) == 31) res[wave][q] = make_float2(re, im);
    };
    if (wrap) {
        for (int i = 0; i < PW / 2; ++i) point(2 * i + half, std::true_type{});
    } else {
#pragma unroll 4
        for (int i = 0; i < PW / 2; ++i) point(2 * i + half, std::false_type{});
    }
    wave_lds_fence();
    if (lane < PW && p < npts) C[(int64_t)blockIdx.y * npts + p] = res[wave][lane];
}

// ---------------------------------------------------------------------------
// fine-grid transforms (pruned to the N x N modes)
// fine row r, column l <-> cell (x = l, y = r); mode m <-> fine index m mod nf
// V: nf rows x N mode columns (row major), per slice
// ---------------------------------------------------------------------------
__device__ __forceinline__ int mode_to_fine(int a, int N, int nf) {
    const int m = a - N / 2;
    return m < 0 ? m + nf : m;
}

// type 1, pass A: FFT+ of every fine row, keep the N mode columns -> V
template <int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_fine_rows_t1(const float2 *__restrict__ fine, float2 *__restrict__ V, int nf, int N, int nl,
               FftPlan plan, const float2 *__restrict__ tw) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) nf = LC;
    const int slice = blockIdx.y;
    const int row0 = blockIdx.x * nl;
    const int nloc = min(nl, nf - row0);
    const float2 *fs = fine + (int64_t)slice * nf * nf;
    for (int idx = threadIdx.x; idx < nl * nf; idx += NT) {
        const int l = idx / nf, e = idx - l * nf;
        buf[lds_row(l, e, nf)] = l < nloc ? fs[(int64_t)(row0 + l) * nf + e] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    nu_fft<1, NT, MAXE, false, LC>(buf, nl, nf, 0, plan, tw);
    float2 *vs = V + (int64_t)slice * nf * N;
    for (int idx = threadIdx.x; idx < nloc * N; idx += NT) {
        const int l = idx / N, b = idx - l * N;
        vs[(int64_t)(row0 + l) * N + b] = buf[lds_row(l, mode_to_fine(b, N, nf), nf)];
    }
}

// type 1, pass B: FFT+ down each mode column, keep the N mode rows,
// deconvolve, real part / nrad -> image (N x N real)
// LC > 0: B = 1 << lsh
template <int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_fine_cols_t1(const float2 *__restrict__ V, float *__restrict__ img, const float *__restrict__ corr,
               int nf, int N, int B, int lsh, float scale, FftPlan plan, const float2 *__restrict__ tw) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) nf = LC;
    const int slice = blockIdx.y;
    const int col0 = blockIdx.x * B;
    const float2 *vs = V + (int64_t)slice * nf * N;
    for (int idx = threadIdx.x; idx < nf * B; idx += NT) {
        const int i = idx / B, c = idx - i * B;
        buf[lds_col(c, i, B)] = col0 + c < N ? vs[(int64_t)i * N + col0 + c] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    nu_fft<1, NT, MAXE, true, LC>(buf, B, nf, lsh, plan, tw);
    float *is = img + (int64_t)slice * N * N;
    for (int idx = threadIdx.x; idx < N * B; idx += NT) {
        const int a = idx / B, c = idx - a * B;
        const int b = col0 + c;
        if (b < N) is[(int64_t)a * N + b] = buf[lds_col(c, mode_to_fine(a, N, nf), B)].x * corr[a] * corr[b] * scale;
    }
}

// type 2, pass B: deconvolve the image, place the N mode rows on the fine
// column, FFT- -> V (nf x N)
template <int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_fine_cols_t2(const float *__restrict__ img, float2 *__restrict__ V, const float *__restrict__ corr,
               int nf, int N, int B, int lsh, FftPlan plan, const float2 *__restrict__ tw) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) nf = LC;
    const int slice = blockIdx.y;
    const int col0 = blockIdx.x * B;
    const float *is = img + (int64_t)slice * N * N;
    for (int idx = threadIdx.x; idx < nf * B; idx += NT) buf[swz(idx)] = make_float2(0.f, 0.f);
    __syncthreads();
    for (int idx = threadIdx.x; idx < N * B; idx += NT) {
        const int a = idx / B, c = idx - a * B;
        const int b = col0 + c;
        if (b < N) buf[lds_col(c, mode_to_fine(a, N, nf), B)] = make_float2(is[(int64_t)a * N + b] * corr[a] * corr[b], 0.f);
    }
    __syncthreads();
    nu_fft<-1, NT, MAXE, true, LC>(buf, B, nf, lsh, plan, tw);
    float2 *vs = V + (int64_t)slice * nf * N;
    for (int idx = threadIdx.x; idx < nf * B; idx += NT) {
        const int i = idx / B, c = idx - i * B;
        if (col0 + c < N) vs[(int64_t)i * N + col0 + c] = buf[lds_col(c, i, B)];
    }
}

// type 2, pass A: place the N mode columns of each V row on the fine row,
// FFT- -> fine grid
template <int NT, int MAXE, int LC>
__global__ void __launch_bounds__(NT)
k_fine_rows_t2(const float2 *__restrict__ V, float2 *__restrict__ fine, int nf, int N, int nl,
               FftPlan plan, const float2 *__restrict__ tw) {
    float2 *buf = reinterpret_cast<float2 *>(lc_smem);
    if constexpr (LC > 0) nf = LC;
    const int slice = blockIdx.y;
    const int row0 = blockIdx.x * nl;
    const int nloc = min(nl, nf - row0);
    for (int idx = threadIdx.x; idx < nl * nf; idx += NT) buf[swz(idx)] = make_float2(0.f, 0.f);
    __syncthreads();
    const float2 *vs = V + (int64_t)slice * nf * N;
    for (int idx = threadIdx.x; idx < nloc * N; idx += NT) {
        const int l = idx / N, b = idx - l * N;
        buf[lds_row(l, mode_to_fine(b, N, nf), nf)] = vs[(int64_t)(row0 + l) * N + b];
    }
    __syncthreads();
    nu_fft<-1, NT, MAXE, false, LC>(buf, nl, nf, 0, plan, tw);
    float2 *fs = fine + (int64_t)slice * nf * nf;
    for (int idx = threadIdx.x; idx < nloc * nf; idx += NT) {
        const int l = idx / nf, e = idx - l * nf;
        fs[(int64_t)(row0 + l) * nf + e] = buf[lds_row(l, e, nf)];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// the kernel's Fourier transform by 96-point Gauss-Legendre quadrature (FP64):
// Psi(xi) = (w/2) int_{-pi/2}^{pi/2} e^{beta (cos t - 1)} cos(xi (w/2) sin t) cos t dt
// The integrand is even, so 48 nodes; what does not depend on xi is tabulated.
namespace {
struct EsNodes {
    static constexpr int N = 96;
    double x[N / 2], w[N / 2];   // nodes in (0, 1) and weights
    EsNodes() {
        for (int i = 0; i < N / 2; ++i) {
            double v = std::cos(M_PI * (i + 0.75) / (N + 0.5)), dp = 0.0;
            for (int it = 0; it < 100; ++it) {
                double p0 = 1.0, p1 = v;
                for (int k = 2; k <= N; ++k) {
                    const double p2 = ((2.0 * k - 1.0) * v * p1 - (k - 1.0) * p0) / k;
                    p0 = p1;
                    p1 = p2;
                }
                dp = N * (v * p1 - p0) / (v * v - 1.0);
                const double dx = p1 / dp;
                v -= dx;
                if (std::fabs(dx) < 1e-16) break;
            }
            double p0 = 1.0, p1 = v;
            for (int k = 2; k <= N; ++k) {
                const double p2 = ((2.0 * k - 1.0) * v * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = N * (v * p1 - p0) / (v * v - 1.0);
            x[i] = v;
            w[i] = 2.0 / ((1.0 - v * v) * dp * dp);
        }
    }
};
} // namespace

void es_correction(int n, int nf, int w, double beta, float *corr) {
    static const EsNodes q;
    constexpr int NQ = EsNodes::N / 2;
    const double hw = 0.5 * w;
    double arg[NQ], amp[NQ];
    for (int i = 0; i < NQ; ++i) {
        const double t = 0.5 * M_PI * q.x[i], ct = std::cos(t);
        arg[i] = hw * std::sin(t) * 2.0 * M_PI / (double)nf;
        amp[i] = 2.0 * q.w[i] * std::exp(beta * (ct - 1.0)) * ct;
    }
    for (int m = 0; m <= n / 2; ++m) {
        double s = 0.0;
        for (int i = 0; i < NQ; ++i) s += amp[i] * std::cos((double)m * arg[i]);
        const float c = (float)(((m & 1) ? -1.0 : 1.0) / (hw * 0.5 * M_PI * s));
        corr[n / 2 - m] = c;
        if (n / 2 + m < n) corr[n / 2 + m] = c;
    }
}

// y[0 .. n) = DFT_- of x[0], x[step], ... (n = 2^p 3^q), recursively by radix 2 and 3
static void host_dft(const std::complex<double> *x, int n, int step, std::complex<double> *y) {
    if (n == 1) {
        y[0] = x[0];
        return;
    }
    const int r = n % 2 == 0 ? 2 : 3, m = n / r;
    for (int j = 0; j < r; ++j) host_dft(x + j * step, m, step * r, y + j * m);
    for (int k = 0; k < m; ++k) {
        const std::complex<double> a = y[k], b = y[m + k] * std::polar(1.0, -2.0 * M_PI * k / n);
        if (r == 2) {
            y[k] = a + b;
            y[m + k] = a - b;
        } else {
            const std::complex<double> c = y[2 * m + k] * std::polar(1.0, -4.0 * M_PI * k / n);
            const std::complex<double> s = b + c, d = std::complex<double>(0.0, -std::sqrt(0.75)) * (b - c);
            y[k] = a + s;
            y[m + k] = a - 0.5 * s + d;
            y[2 * m + k] = a - 0.5 * s - d;
        }
    }
}

void bluestein_tables(int n, int L, std::vector<std::complex<double>> &chirp, std::vector<std::complex<double>> &bhat) {
    chirp.resize(n);
    std::vector<std::complex<double>> b(L, 0.0);
    for (int k = 0; k < n; ++k) {
        const double ang = M_PI * (double)(((int64_t)k * k) % (2 * (int64_t)n)) / (double)n;
        b[k] = chirp[k] = std::complex<double>(std::cos(ang), std::sin(ang));
        if (k) b[L - k] = b[k];
    }
    bhat.resize(L);
    host_dft(b.data(), L, 1, bhat.data());
    for (auto &v : bhat) v /= (double)L;
}

// (cos, sin) of every projection angle, FP64, once per geometry: the sort, the
// spread and the interpolation read the point's angle's
__global__ void k_angle_table(const double *__restrict__ theta, double2 *__restrict__ cs, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        double s, c;
        sincos(theta[i], &s, &c);
        cs[i] = make_double2(c, s);
    }
}

int nufft2d_fine_n(int64_t N) {
    int64_t nf = 2 * N;
    while (!is_2_3_smooth(nf) || nf < 2 * NU_W) ++nf;
    return (int)nf;
}

// longest detector line in LDS: NU_NT * NU_ME values
constexpr int DET_FFT_MAX = 4096;

// Bluestein tables of a detector of n columns: chirp and chirp spectrum in FP64
static void det_blue_init(Ctx &c, Nufft2D &u, int n) {
    int L = 16;
    while (L < 2 * n - 1) L *= 2;
    LC_REQUIRE(fft_make_plan(L, u.plan_det), "detector transform: no Bluestein length");
    std::vector<std::complex<double>> ch, bh;
    bluestein_tables(n, L, ch, bh);
    std::vector<double2> t;
    for (const auto &v : ch) t.push_back(make_double2(v.real(), v.imag()));
    for (const auto &v : bh) t.push_back(make_double2(v.real(), v.imag()));
    u.chirp.alloc(sizeof(double2) * t.size());
    LC_HIP(hipMemcpyAsync(u.chirp.as(), t.data(), sizeof(double2) * t.size(), hipMemcpyHostToDevice, c.stream()));
    c.sync();
}

namespace {
size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

Grid2 grid2(const Geom2D &g) {
    Grid2 s;
    s.nang = (int)g.nang;
    s.nrad = (int)g.nrad;
    s.nf = g.nu.nf;
    s.nb = ceil_div(g.nu.nf, CB);
    s.dr = 2.0 * M_PI / (double)g.nrad;
    s.sc = (double)g.nu.nf / (2.0 * M_PI);
    s.inrad = 1.0 / (double)g.nrad;
    s.beta = (float)g.nu.beta;
    return s;
}

int tiles_of(int nf) { return ceil_div(nf, TE) * ceil_div(nf, TE); }
} // namespace

// the points sorted by corner bin, the bins' starts, and the tiles, fullest
// first: what type 1 needs beside nufft2d_init's tables.  The sort's working space, about 20 bytes per point, is
// the projections' scratch, which the caller's own call is about to use, or
// (own_work) freed again: a server's main context never projects
void nufft2d_order(Ctx &c, Geom2D &g, bool own_work) {
    Nufft2D &u = g.nu;
    const Grid2 s = grid2(g);
    LC_REQUIRE(g.nang * g.nrad < (int64_t)1 << 31, "2-D projector: 2^31 or more points per slice");
    const int npts = (int)(g.nang * g.nrad), nbins = s.nb * s.nb;
    int bits = 1;
    while ((1 << bits) < nbins) ++bits;
    const int tiles = u.ntiles = tiles_of(s.nf);
    const size_t bK = al256(sizeof(unsigned) * (size_t)std::max(npts, tiles));
    size_t tb = 0, tt = 0;
    LC_HIP(rocprim::radix_sort_pairs(nullptr, tb, (unsigned *)nullptr, (unsigned *)nullptr, (unsigned *)nullptr,
                                     (unsigned *)nullptr, (size_t)npts, 0, bits, c.stream()));
    LC_HIP(rocprim::radix_sort_pairs(nullptr, tt, (unsigned *)nullptr, (unsigned *)nullptr, (int *)nullptr,
                                     (int *)nullptr, (size_t)tiles, 0, 31, c.stream()));
    const size_t need = 3 * bK + al256(std::max(tb, tt)) + sizeof(int);
    DBuf own;
    if (own_work) own.alloc(need);
    char *ws = own_work ? own.as<char>() : reinterpret_cast<char *>(c.scratch(3, need));
    unsigned *ka = reinterpret_cast<unsigned *>(ws), *kb = reinterpret_cast<unsigned *>(ws + bK),
             *va = reinterpret_cast<unsigned *>(ws + 2 * bK);
    void *tmp = ws + 3 * bK;
    int *heavy = reinterpret_cast<int *>(ws + 3 * bK + al256(std::max(tb, tt)));
    const size_t bP = al256(sizeof(unsigned) * (size_t)npts);
    u.points.alloc(bP + sizeof(int) * (nbins + 1));
    unsigned *vb = u.points.as<unsigned>();
    int *st = reinterpret_cast<int *>(u.points.as<char>() + bP);
    hipLaunchKernelGGL(k_bin2_keys, dim3(ceil_div(npts, 256)), dim3(256), 0, c.stream(), u.cs.as<double2>(), s, ka,
                       va, npts);
    LC_HIP(hipGetLastError());
    LC_HIP(rocprim::radix_sort_pairs(tmp, tb, ka, kb, va, vb, (size_t)npts, 0, bits, c.stream()));
    hipLaunchKernelGGL(k_bin2_starts, dim3(ceil_div(nbins + 1, 256)), dim3(256), 0, c.stream(), kb, npts, st, nbins);
    LC_HIP(hipGetLastError());
    u.tiles.alloc(sizeof(int) * tiles);
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(1), 0, c.stream(), heavy);
    hipLaunchKernelGGL(k_tile_keys, dim3(ceil_div(tiles, 256)), dim3(256), 0, c.stream(), st, ka, (int *)va, heavy,
                       tiles, ceil_div(s.nf, TE), s.nf, s.nb);
    LC_HIP(hipGetLastError());
    LC_HIP(rocprim::radix_sort_pairs(tmp, tt, ka, kb, (int *)va, u.tiles.as<int>(), (size_t)tiles, 0, 31, c.stream()));
    LC_HIP(hipMemcpyAsync(&u.nheavy, heavy, sizeof(int), hipMemcpyDeviceToHost, c.stream()));
    c.sync();
    u.ordered = true;
}

// device bytes of the points' order and the tiles that a geometry keeps
size_t nufft2d_order_bytes(int64_t nang, int64_t nrad, int nf) {
    const size_t nb = ceil_div(nf, CB);
    return al256(sizeof(unsigned) * (size_t)(nang * nrad)) + sizeof(int) * (nb * nb + 1 + (size_t)tiles_of(nf));
}

void nufft2d_init(Ctx &c, Geom2D &g) {
    Nufft2D &u = g.nu;
    u.cs.alloc(sizeof(double2) * g.nang);
    hipLaunchKernelGGL(k_angle_table, dim3(ceil_div(g.nang, 256)), dim3(256), 0, c.stream(),
                       g.d_theta.as<double>(), u.cs.as<double2>(), (int)g.nang);
    LC_HIP(hipGetLastError());
    const int N = (int)g.N;
    const int64_t nf = nufft2d_fine_n(N);
    u.nf = (int)nf;
    u.w = NU_W;
    u.beta = 2.30 * NU_W;
    std::vector<float> corr(N);
    es_correction(N, (int)nf, NU_W, u.beta, corr.data());   // (-1)^m from the centred fine grid
    u.corr.alloc(sizeof(float) * N);
    // stream-ordered copy: a legacy-stream copy would have to wait on other
    // threads' streams, some of which may be capturing graphs
    LC_HIP(hipMemcpyAsync(u.corr.as(), corr.data(), sizeof(float) * N, hipMemcpyHostToDevice, c.stream()));
    c.sync();
    LC_REQUIRE(fft_make_plan(u.nf, u.plan_nf), "nufft: fine grid size not 2^p 3^q");
    u.det_fast = g.nrad <= DET_FFT_MAX && fft_make_plan((int)g.nrad, u.plan_det);
    // (back-projection of 360 rows, us, directly / by Bluestein: 37 columns 80 / 96,
    // 53 105 / 118, 67 126 / 124, 127 212 / 198, 511 1084 / 677)
    u.det_blue = !u.det_fast && g.nrad > 64 && 2 * g.nrad - 1 <= DET_FFT_MAX;
    if (u.det_blue) det_blue_init(c, u, (int)g.nrad);
    u.ready = true;
}

namespace {
constexpr int NU_NT = 256, NU_ME = 16, NU_MEC = 32;   // rows / columns: NT*ME elements in LDS
// compiled column passes: 512 threads x NU_ME, B = a power of two columns
constexpr int NU_NT_CT = 512;
struct ColShape {
    int B, lsh;
};
ColShape col_shape(int nf, int N) {
    ColShape cs{1, 0};
    while (2 * cs.B * nf <= NU_NT_CT * NU_ME && cs.B < N) {
        cs.B *= 2;
        ++cs.lsh;
    }
    return cs;
}

// ns slices of g.nang sinogram rows each
void det_transform(Ctx &c, const Geom2D &g, int sign, const float *real_in, const float2 *cplx_in,
                   float2 *cplx_out, float *real_out, int ns) {
    const int n = (int)g.nrad, nang = (int)g.nang, nrows = ns * nang;
    const float scale = 1.0f / (float)n;
    static_assert(DET_FFT_MAX == NU_NT * NU_ME, "a detector line fits a block");
    if (g.nu.det_blue) {
        const int L = g.nu.plan_det.L, nl = std::max(1, std::min(DET_FFT_MAX / L, 64));
        const double2 *tw = c.twiddles<double>(L), *chirp = g.nu.chirp.as<double2>();
        const size_t sh = sizeof(double2) * lds_round(nl * L);
        const dim3 grid(ceil_div(nang, nl), ns);
        auto launch = [&](auto len) {
            constexpr int LC = decltype(len)::value;
            if (sign < 0)
                hipLaunchKernelGGL((k_det_blue<-1, NU_NT, NU_ME, LC>), grid, dim3(NU_NT), sh, c.stream(), real_in,
                                   cplx_in, cplx_out, real_out, nang, n, nl, g.nu.plan_det, tw, chirp, chirp + n,
                                   scale);
            else
                hipLaunchKernelGGL((k_det_blue<1, NU_NT, NU_ME, LC>), grid, dim3(NU_NT), sh, c.stream(), real_in,
                                   cplx_in, cplx_out, real_out, nang, n, nl, g.nu.plan_det, tw, chirp, chirp + n,
                                   scale);
        };
        switch (L) {   // the lengths of common widths compiled, the rest by their plan
        case 256: launch(std::integral_constant<int, 256>{}); break;
        case 512: launch(std::integral_constant<int, 512>{}); break;
        case 1024: launch(std::integral_constant<int, 1024>{}); break;
        case 2048: launch(std::integral_constant<int, 2048>{}); break;
        default: launch(std::integral_constant<int, 0>{});
        }
    } else if (g.nu.det_fast) {
        const float2 *tw = c.twiddles<float>(n);
        const int nl = std::max(1, std::min(NU_NT * NU_ME / n, 64));
        const size_t sh = sizeof(float2) * lds_round(nl * n);
        const dim3 grid(ceil_div(nang, nl), ns);
        auto launch = [&](auto len) {
            constexpr int LC = decltype(len)::value;
            if (sign < 0)
                hipLaunchKernelGGL((k_det_fft<-1, NU_NT, NU_ME, LC>), grid, dim3(NU_NT), sh, c.stream(),
                                   real_in, cplx_in, cplx_out, real_out, nang, n, nl, g.nu.plan_det, tw, scale);
            else
                hipLaunchKernelGGL((k_det_fft<1, NU_NT, NU_ME, LC>), grid, dim3(NU_NT), sh, c.stream(),
                                   real_in, cplx_in, cplx_out, real_out, nang, n, nl, g.nu.plan_det, tw, scale);
        };
        if (!with_ct_len(n, launch)) launch(std::integral_constant<int, 0>{});
    } else {
        const float2 *tw = c.twiddles<float>(n);
        dim3 grid(nrows);
        if (sign < 0)
            hipLaunchKernelGGL(k_det_dft<-1>, grid, dim3(128), 0, c.stream(), real_in, cplx_in,
                               cplx_out, real_out, nrows, n, tw, scale);
        else
            hipLaunchKernelGGL(k_det_dft<1>, grid, dim3(128), 0, c.stream(), real_in, cplx_in,
                               cplx_out, real_out, nrows, n, tw, scale);
    }
    LC_HIP(hipGetLastError());
}
} // namespace

namespace {
struct NuWork {
    float2 *C, *F, *V;
};

NuWork nu_work(Ctx &c, const Geom2D &g, int ns) {
    const int N = (int)g.N, nf = g.nu.nf;
    const int64_t npts = g.nang * g.nrad;
    const size_t bC = al256(sizeof(float2) * (size_t)ns * npts);
    const size_t bF = al256(sizeof(float2) * (size_t)ns * nf * nf);
    const size_t bV = al256(sizeof(float2) * (size_t)ns * nf * N);
    char *ws = reinterpret_cast<char *>(c.scratch(3, bC + bF + bV));
    NuWork w;
    w.C = reinterpret_cast<float2 *>(ws);
    w.F = reinterpret_cast<float2 *>(ws + bC);
    w.V = reinterpret_cast<float2 *>(ws + bC + bF);
    return w;
}

// type-1 spread of nch runs of SC slices from slice `first`: C -> F
template <int SC> void spread2(Ctx &c, const Geom2D &g, const NuWork &w, int first, int nch) {
    if (nch == 0) return;
    const Nufft2D &u = g.nu;
    const Grid2 s = grid2(g);
    const unsigned *sval = u.points.as<unsigned>();
    const int *start = reinterpret_cast<const int *>(u.points.as<char>() +
                                                     al256(sizeof(unsigned) * (size_t)(g.nang * g.nrad)));
    hipLaunchKernelGGL(k_spread2d<SC>, dim3(u.nheavy + ceil_div(u.ntiles - u.nheavy, SW), nch), dim3(64 * SW), 0,
                       c.stream(), w.C, w.F, u.cs.as<double2>(), sval, start, u.tiles.as<int>(), u.ntiles, u.nheavy,
                       first, ceil_div(s.nf, TE), s);
    LC_HIP(hipGetLastError());
}

// type 1: C (ns x nang x nrad complex) -> vol = Re(T1 C) / nrad
void type1(Ctx &c, const Geom2D &g, const NuWork &w, float *vol, int ns) {
    const Nufft2D &u = g.nu;
    const int N = (int)g.N, nf = u.nf;
    // slices share a wave's weights by fours, the last ones by two and one
    spread2<4>(c, g, w, 0, ns / 4);
    spread2<2>(c, g, w, ns & ~3, (ns & 2) >> 1);
    spread2<1>(c, g, w, ns & ~1, ns & 1);
    const float2 *tw = c.twiddles<float>(nf);
    const int nl = std::min(NU_NT * NU_ME / nf, nf);
    const size_t shr = sizeof(float2) * lds_round(nl * nf);
    if (!with_ct_len(nf, [&](auto len) {
            hipLaunchKernelGGL((k_fine_rows_t1<NU_NT, NU_ME, decltype(len)::value>), dim3(ceil_div(nf, nl), ns),
                               dim3(NU_NT), shr, c.stream(), w.F, w.V, nf, N, nl, u.plan_nf, tw);
        }))
        hipLaunchKernelGGL((k_fine_rows_t1<NU_NT, NU_ME, 0>), dim3(ceil_div(nf, nl), ns), dim3(NU_NT), shr,
                           c.stream(), w.F, w.V, nf, N, nl, u.plan_nf, tw);
    LC_HIP(hipGetLastError());
    if (!with_ct_len(nf, [&](auto len) {
            const ColShape cs = col_shape(nf, N);
            hipLaunchKernelGGL((k_fine_cols_t1<NU_NT_CT, NU_ME, decltype(len)::value>), dim3(ceil_div(N, cs.B), ns),
                               dim3(NU_NT_CT), sizeof(float2) * lds_round(cs.B * nf), c.stream(), w.V, vol,
                               u.corr.as<float>(), nf, N, cs.B, cs.lsh, 1.0f / (float)g.nrad, u.plan_nf, tw);
        })) {
        const int B = std::min(NU_NT * NU_MEC / nf, N);
        hipLaunchKernelGGL((k_fine_cols_t1<NU_NT, NU_MEC, 0>), dim3(ceil_div(N, B), ns), dim3(NU_NT),
                           sizeof(float2) * lds_round(B * nf), c.stream(), w.V, vol, u.corr.as<float>(), nf, N,
                           B, 0, 1.0f / (float)g.nrad, u.plan_nf, tw);
    }
    LC_HIP(hipGetLastError());
}

// type 2: vol (ns x N x N real) -> C = T2 vol
void type2(Ctx &c, const Geom2D &g, const NuWork &w, const float *vol, int ns) {
    const Nufft2D &u = g.nu;
    const int N = (int)g.N, nf = u.nf;
    const int64_t npts = g.nang * g.nrad;
    const float2 *tw = c.twiddles<float>(nf);
    if (!with_ct_len(nf, [&](auto len) {
            const ColShape cs = col_shape(nf, N);
            hipLaunchKernelGGL((k_fine_cols_t2<NU_NT_CT, NU_ME, decltype(len)::value>), dim3(ceil_div(N, cs.B), ns),
                               dim3(NU_NT_CT), sizeof(float2) * lds_round(cs.B * nf), c.stream(), vol, w.V,
                               u.corr.as<float>(), nf, N, cs.B, cs.lsh, u.plan_nf, tw);
        })) {
        const int B = std::min(NU_NT * NU_MEC / nf, N);
        hipLaunchKernelGGL((k_fine_cols_t2<NU_NT, NU_MEC, 0>), dim3(ceil_div(N, B), ns), dim3(NU_NT),
                           sizeof(float2) * lds_round(B * nf), c.stream(), vol, w.V, u.corr.as<float>(), nf,
                           N, B, 0, u.plan_nf, tw);
    }
    LC_HIP(hipGetLastError());
    const int nl = std::min(NU_NT * NU_ME / nf, nf);
    const size_t shr = sizeof(float2) * lds_round(nl * nf);
    if (!with_ct_len(nf, [&](auto len) {
            hipLaunchKernelGGL((k_fine_rows_t2<NU_NT, NU_ME, decltype(len)::value>), dim3(ceil_div(nf, nl), ns),
                               dim3(NU_NT), shr, c.stream(), w.V, w.F, nf, N, nl, u.plan_nf, tw);
        }))
        hipLaunchKernelGGL((k_fine_rows_t2<NU_NT, NU_ME, 0>), dim3(ceil_div(nf, nl), ns), dim3(NU_NT), shr,
                           c.stream(), w.V, w.F, nf, N, nl, u.plan_nf, tw);
    LC_HIP(hipGetLastError());
    auto interp = [&](auto pw) {
        constexpr int PW = decltype(pw)::value;
        hipLaunchKernelGGL(k_interp2d<PW>, dim3(ceil_div(npts, PW * IW), ns), dim3(64 * IW), 0, c.stream(), w.F, w.C,
                           g.nu.cs.as<double2>(), grid2(g), (int)npts);
    };
    // below four waves per SIMD the time is that of a wave's loop over its points
    if ((int64_t)ceil_div(npts, 64) * ns < 4096) interp(std::integral_constant<int, 16>{});
    else interp(std::integral_constant<int, 64>{});
    LC_HIP(hipGetLastError());
}

void nu_check(Ctx &c, Geom2D &g, int ns, bool type1) {
    if (!g.nu.ready) nufft2d_init(c, g);
    LC_REQUIRE(g.nu.nf <= NU_NT * NU_ME, "nufft: fine grid too large (image size above 2048)");
    LC_REQUIRE(ns >= 1 && ns <= 65535, "nufft: 1 to 65535 slices per call");
    if (type1 && !g.nu.ordered) nufft2d_order(c, g);
}
} // namespace

// backproj2d: sino (ns x nang x nrad real, device) -> vol (ns x N x N real, device)
void backproj2d_dev(Ctx &c, Geom2D &g, const float *sino, float *vol, int ns) {
    nu_check(c, g, ns, true);
    const NuWork w = nu_work(c, g, ns);
    det_transform(c, g, -1, sino, nullptr, w.C, nullptr, ns);
    type1(c, g, w, vol, ns);
}

// forward2d: vol (ns x N x N real, device) -> sino (ns x nang x nrad real, device)
void forward2d_dev(Ctx &c, Geom2D &g, const float *vol, float *sino, int ns) {
    nu_check(c, g, ns, false);
    const NuWork w = nu_work(c, g, ns);
    type2(c, g, w, vol, ns);
    det_transform(c, g, 1, nullptr, w.C, nullptr, sino, ns);
}

// sysmat2d(x, grid) = Re(T1(T2 x)) / nrad (src/gradient.cpp:59-69)
void sysmat2d_nufft_dev(Ctx &c, Geom2D &g, const float *x, float *y, int ns) {
    nu_check(c, g, ns, true);
    const NuWork w = nu_work(c, g, ns);
    type2(c, g, w, x, ns);
    type1(c, g, w, y, ns);
}

// Times the back-projection of nslices zero sinograms on g's grid (best_ms) and
// installs choice 0: both numbers name the one compiled spread.
int nufft2d_autotune(Ctx &c, Geom2D &g, int nslices, double *best_ms) {
    nu_check(c, g, nslices, true);
    const int64_t npts = g.nang * g.nrad;
    DBuf sino(sizeof(float) * (size_t)(nslices * npts)), vol(sizeof(float) * (size_t)nslices * g.N * g.N);
    LC_HIP(hipMemsetAsync(sino.as(), 0, sizeof(float) * (size_t)(nslices * npts), c.stream()));
    hipEvent_t e0, e1;
    LC_HIP(hipEventCreate(&e0));
    LC_HIP(hipEventCreate(&e1));
    float ms = 0.f;
    try {
        backproj2d_dev(c, g, sino.as<float>(), vol.as<float>(), nslices);   // warm-up
        LC_HIP(hipEventRecord(e0, c.stream()));
        for (int r = 0; r < 3; ++r) backproj2d_dev(c, g, sino.as<float>(), vol.as<float>(), nslices);
        LC_HIP(hipEventRecord(e1, c.stream()));
        LC_HIP(hipEventSynchronize(e1));
        LC_HIP(hipEventElapsedTime(&ms, e0, e1));
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    c.nu2_tuning[g.nu.nf] = 0;
    if (best_ms) *best_ms = ms / 3;
    return 0;
}

int nufft2d_num_shapes() { return 2; }

} // namespace lc
