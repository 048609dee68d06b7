// HIP kernels of the MI355X DNS time step (gfx950, FP64 throughout).
//
// Nonlinear term pipeline for one field (reference: NSE::nonlinear,
// channelflow/nse.cpp:383-391 -> diffops.cpp rotationalNL/convectionNL/
// divergenceNL/skewsymmetricNL):
//   k_yinv_t Chebyshev coefficients -> values at the Chebyshev points y_n,
//            with d/dy folded into the operator (T, T*D) and the base flow
//            U(y), W(y), -Vsuck added to the kx=kz=0 mode;
//   k_xwinv  inverse x-FFT per (field, y, kz) line, optional d/dx (k_xinv:
//            LDS FFTs for the lengths the wavefront FFT does not cover);
//   k_zsplit per (y, x) line: c2r z-FFTs, pointwise products, r2c z-FFTs,
//            three wavefronts per group of lines (k_zwave: one; k_zpass: LDS
//            FFTs, block-wide, for the lengths the wavefront FFT does not cover);
//   k_xwfwd  forward x-FFT, live kx kept, 1/(Nx Nz) scaling (k_xfwd; k_xwfold: the
//            skew-symmetric form's, with the x part of its divergence);
//   k_yfwd_t values -> Chebyshev coefficients, with the spectral divergence
//            of u_i u_j folded in for the divergence/skew-symmetric forms.
// Only non-aliased modes |kx| <= kxd, kz <= kzd are ever stored, so the
// reference's zeroPaddedModes() (flowfield.cpp:2235) is implicit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "cfg_fft.hpp"
#include "cfg_wave.hpp"
#include "cfg_z.hpp"

namespace cfg {

// ===========================================================================
// Elementwise combination (dnsalgo.cpp:218-224, 668-673)
// ===========================================================================
struct CombineArgs {
    double coef[8];
    const double* in[8];
};

__global__ void k_combine(long n, int nterms, CombineArgs a, double* out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc = 0.0;
    for (int j = 0; j < nterms; ++j) acc += a.coef[j] * a.in[j][i];
    out[i] = acc;
}

void launch_combine(long n, int nterms, const double* coef, const double* const* in, double* out, hipStream_t st) {
    CombineArgs a;
    for (int j = 0; j < 8; ++j) {
        a.coef[j] = j < nterms ? coef[j] : 0.0;
        a.in[j] = j < nterms ? in[j] : nullptr;
    }
    const int blk = 256;
    k_combine<<<(int)((n + blk - 1) / blk), blk, 0, st>>>(n, nterms, a, out);
}

// ===========================================================================
// Finiteness of member states (the isfinite(L2Norm(u)) checks of
// cfdsi.cpp:707-710, 769-774): flags[m] = 1 if field m holds a NaN or an
// infinity. Blocks stride over the field; a wave with a non-finite value
// stores the flag (every such store writes the same 1).
// ===========================================================================
__global__ void __launch_bounds__(256) k_nonfinite(const double* const* __restrict__ fields, long n,
                                                   double* __restrict__ flags) {
    const double* __restrict__ f = fields[blockIdx.y];
    bool bad = false;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        bad = bad || !isfinite(f[i]);
    if (__any(bad) && bad) flags[blockIdx.y] = 1.0;
}

void launch_nonfinite(int nfields, const double* const* fields, long n, double* flags, hipStream_t st) {
    if (nfields <= 0) return;
    const int blk = 256;
    const long want = (n + blk * 8L - 1) / (blk * 8L);  // about 8 values per thread
    const unsigned gx = (unsigned)std::max(1L, std::min(want, 1024L));
    k_nonfinite<<<dim3(gx, (unsigned)nfields), blk, 0, st>>>(fields, n, flags);
}

// ===========================================================================
// Nonlinear term
// ===========================================================================
// inverse x-FFT: yp [F][Ny][nkz][nkx] -> xp [Fo][Ny][Nx][nkz]; output f >= nsrc is
// d/dx of source field f - nsrc. XL kz-lines per block.
__global__ void __launch_bounds__(256) k_xinv(Geom g, FFTPlan px, int XL, int nsrc, const double2* __restrict__ yp0,
                                              long sy, double2* __restrict__ xp0, long sx) {
    extern __shared__ double2 lds[];
    const double2* __restrict__ yp = yp0 + blockIdx.z * sy;
    double2* __restrict__ xp = xp0 + blockIdx.z * sx;
    const int Nx = g.Nx, nkz = g.nkz, nkx = g.nkx, Ny = g.Ny;
    const int nchunk = (nkz + XL - 1) / XL;
    const int y = blockIdx.x / nchunk, ikz0 = (blockIdx.x % nchunk) * XL;
    const int fo = blockIdx.y;
    const bool deriv = fo >= nsrc;
    const int fs = deriv ? fo - nsrc : fo;
    const int nl = min(XL, nkz - ikz0);
    const int P = lpitch(Nx);
    double2* tw = lds;
    double2* a = lds + Nx;
    double2* b = a + XL * P;
    stage_tw(tw, px);
    const double dk = 2 * PI / g.Lx;
    for (int w = threadIdx.x; w < nl * Nx; w += blockDim.x) {
        const int l = w / Nx, j = w - l * Nx;
        int ikx = -1;
        if (j <= g.kxd) ikx = j;
        else if (j >= Nx - g.kxd) ikx = j - Nx + nkx;
        double2 v = make_double2(0.0, 0.0);
        if (ikx >= 0) {
            v = yp[(((long)fs * Ny + y) * nkz + ikz0 + l) * nkx + ikx];
            if (deriv) v = imul(dk * kx_of(g, ikx), v);
        }
        a[l * P + pidx(j)] = v;
    }
    __syncthreads();
    double2* r = fft_lds<+1>(a, b, px, tw, nl);
    double2* out = xp + (((long)fo * Ny + y) * Nx) * nkz + ikz0;
    for (int w = threadIdx.x; w < nl * Nx; w += blockDim.x) {
        const int x = w / nl, l = w - x * nl;
        out[(long)x * nkz + l] = r[l * P + pidx(x)];
    }
}

// forward x-FFT: zo [G][Ny][Nx][nkz] -> fo [G][Ny][nkz][nkx], scaled by 1/(Nx Nz)
__global__ void __launch_bounds__(256) k_xfwd(Geom g, FFTPlan px, int XL, const double2* __restrict__ zo0, long sx,
                                              double2* __restrict__ fo0, long sy) {
    extern __shared__ double2 lds[];
    const double2* __restrict__ zo = zo0 + blockIdx.z * sx;
    double2* __restrict__ fo = fo0 + blockIdx.z * sy;
    const int Nx = g.Nx, nkz = g.nkz, nkx = g.nkx, Ny = g.Ny;
    const int nchunk = (nkz + XL - 1) / XL;
    const int y = blockIdx.x / nchunk, ikz0 = (blockIdx.x % nchunk) * XL;
    const int f = blockIdx.y;
    const int nl = min(XL, nkz - ikz0);
    const int P = lpitch(Nx);
    double2* tw = lds;
    double2* a = lds + Nx;
    double2* b = a + XL * P;
    stage_tw(tw, px);
    const double2* in = zo + (((long)f * Ny + y) * Nx) * nkz + ikz0;
    for (int w = threadIdx.x; w < nl * Nx; w += blockDim.x) {
        const int x = w / nl, l = w - x * nl;
        a[l * P + pidx(x)] = in[(long)x * nkz + l];
    }
    __syncthreads();
    double2* r = fft_lds<-1>(a, b, px, tw, nl);
    const double scale = 1.0 / ((double)g.Nx * g.Nz);
    for (int w = threadIdx.x; w < nl * nkx; w += blockDim.x) {
        const int l = w / nkx, ikx = w - l * nkx;
        const int j = ikx <= g.kxd ? ikx : ikx - nkx + Nx;
        const double2 v = r[l * P + pidx(j)];
        fo[(((long)f * Ny + y) * nkz + ikz0 + l) * nkx + ikx] = make_double2(v.x * scale, v.y * scale);
    }
}

// ---- wave-local x FFTs ---------------------------------------------------------
// One wavefront per 64/G consecutive kz-lines of one (field, y); each line's
// FFT as in the wave-local z pass. Consecutive lanes of a group hold
// consecutive kx (contiguous reads of yp / writes of fo); the lines of a
// wavefront are consecutive kz (128-byte runs of xp / zo).
//
// Value r of lane j is bin n = j + N1 r, live as kx = n in the lower half of the r
// and as kx = n - NX in the upper half (kxd < NX/2); an odd N2 has a middle r that can
// be either. Every access is at a uniform base, one of two 32-bit lane offsets and a
// constant or uniform distance; with 64-bit addresses and the bin tests formed per
// access those were half of the instructions. us per launch, before -> after: inverse
// 24 of 32^3 14.6 -> 12.7, 128^3 rotational 24.5 -> 22.6, convection 32.5 -> 30.6 (118
// MB, 3.9 TB/s); forward 128^3 15.9 -> 13.0, 48x35x48 4.4 -> 4.1, 54x57x72 6.2 -> 5.8;
// at 192x129x192, at the copy rate, 52.5 -> 53.8 and 36.4 -> 35.4.
struct XBins {
    int lo, hi;            // kx = j + N1 r is live if N1 r < lo, kx = j - N1 q if N1 q < hi
    unsigned at, at_hi;    // byte offsets of kx = j and of the slot N1 N2 past the line's upper half
};
__device__ __forceinline__ XBins x_bins(const Geom& g, int ikz, int j, bool act) {
    const unsigned row = (unsigned)ikz * (unsigned)g.nkx;
    return XBins{act ? g.kxd + 1 - j : 0, act ? g.kxd + 1 + j : 0, (row + (unsigned)j) * 16u,
                 (row + (unsigned)(j + g.nkx)) * 16u};
}
// the wavefront's place: its (y, kz chunk) and the lane's line and position in it
struct XPlace {
    int y, L, j, ikz;
    bool line_ok;
};
template <class S>
__device__ __forceinline__ XPlace x_place(const Geom& g, int wg) {
    const int lane = threadIdx.x % 64, nzc = (g.nkz + S::LPW - 1) / S::LPW;
    const int y = wg / nzc, L = lane / S::G;
    const int ikz = (wg - y * nzc) * S::LPW + L;
    return XPlace{y, L, lane % S::G, ikz, ikz < g.nkz};
}

// inverse x-FFT: yp [F][Ny][nkz][nkx] -> xp [Fo][Ny][Nx][nkz]; output f >= nsrc
// is d/dx of source field f - nsrc
template <int NX>
__global__ void __launch_bounds__(256) k_xwinv(Geom g, const double2* __restrict__ twg, int nsrc,
                                               const double2* __restrict__ yp0, long sy, double2* __restrict__ xp0,
                                               long sx) {
    const BlockId bid = xcd_grid();  // neighbouring blocks on one XCD
    using S = ZW<NX>;
    constexpr int N1 = S::N1, N2 = S::N2;
    extern __shared__ double2 lds[];
    for (int i = threadIdx.x; i < NX; i += blockDim.x) lds[i] = twg[i];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const XPlace w = x_place<S>(g, bid.x * (blockDim.x / 64) + wave);
    if (w.y >= g.Ny) return;
    const int j = w.j, fo = bid.y;
    const bool deriv = fo >= nsrc;
    const int fs = deriv ? fo - nsrc : fo;
    const gbytes src = reinterpret_cast<gbytes>(gmem(yp0) + bid.z * sy + ((long)fs * g.Ny + w.y) * g.M);
    const XBins bins = x_bins(g, w.ikz, j, w.line_ok && j < N1);
    double2 v[N2];
#pragma unroll
    for (int r = 0; r < N2; ++r) {
        v[r] = make_double2(0.0, 0.0);
        if (2 * r < N2 && N1 * r < bins.lo) v[r] = gload(src + 16 * N1 * r, bins.at);
        if (2 * r + 1 >= N2 && N1 * (N2 - r) < bins.hi) v[r] = gload(src - 16 * N1 * (N2 - r), bins.at_hi);
    }
    if (deriv) {
        const double dk = 2 * PI / g.Lx, sj = j;
#pragma unroll
        for (int r = 0; r < N2; ++r) {
            const bool up = 2 * r + 1 > N2 || (2 * r + 1 == N2 && N1 * r >= bins.lo);
            v[r] = imul(dk * (up ? sj - (double)(N1 * (N2 - r)) : sj + (double)(N1 * r)), v[r]);
        }
    }
    double2 u[N1];
    zw_a2b<NX, +1>(v, u, j, lds + NX + (wave * S::LPW + w.L) * S::LBUF, lds);
    if (w.line_ok && j < N2) {
        const gbytes_w out = reinterpret_cast<gbytes_w>(gmem_w(xp0) + bid.z * sx + ((long)fo * g.Ny + w.y) * NX * (long)g.nkz);
        const unsigned at = ((unsigned)j * (unsigned)g.nkz + (unsigned)w.ikz) * 16u;
#pragma unroll
        for (int m = 0; m < N1; ++m) gstore(out + (long)m * (N2 * 16) * g.nkz, at, u[m]);
    }
}

// one line's forward transform: field f of zo at (y, kz) into v[p] = X[j + N1 p]
template <int NX>
__device__ __forceinline__ void x_forward(const Geom& g, const double2* __restrict__ zo, int f, const XPlace& w,
                                          double2* T, const double2* tw, double2 (&v)[ZW<NX>::N2]) {
    constexpr int N1 = ZW<NX>::N1, N2 = ZW<NX>::N2;
    const gbytes in = reinterpret_cast<gbytes>(gmem(zo) + ((long)f * g.Ny + w.y) * NX * (long)g.nkz);
    const bool act = w.line_ok && w.j < N2;
    const unsigned at = act ? ((unsigned)w.j * (unsigned)g.nkz + (unsigned)w.ikz) * 16u : 0u;
    double2 u[N1];
#pragma unroll
    for (int m = 0; m < N1; ++m) {
        u[m] = make_double2(0.0, 0.0);
        if (act) u[m] = gload(in + (long)m * (N2 * 16) * g.nkz, at);
    }
    zw_b2a<NX, -1>(u, v, w.j, T, tw);
}
// calls put(value p, distance, offset, kx) for the live values of a lane
template <int NX, class Put>
__device__ __forceinline__ void x_live(const XBins& b, int j, Put&& put) {
    constexpr int N1 = ZW<NX>::N1, N2 = ZW<NX>::N2;
#pragma unroll
    for (int p = 0; p < N2; ++p) {
        if (2 * p < N2 && N1 * p < b.lo) put(p, 16 * N1 * p, b.at, j + N1 * p);
        if (2 * p + 1 >= N2 && N1 * (N2 - p) < b.hi) put(p, -16 * N1 * (N2 - p), b.at_hi, j - N1 * (N2 - p));
    }
}

// forward x-FFT: zo [G][Ny][Nx][nkz] -> fo [G][Ny][nkz][nkx], scaled by 1/(Nx Nz).
// xcd: blocks in XCD order (xcd_grid), for grids whose rows of nkz bins are
// not a whole number of 128-byte lines, so that neighbouring kz chunks, which
// share the lines at their edges, read them through one L2; where the rows
// are whole lines the dispatch order is faster.
template <int NX>
__global__ void __launch_bounds__(256) k_xwfwd(Geom g, const double2* __restrict__ twg,
                                               const double2* __restrict__ zo0, long sx, double2* __restrict__ fo0,
                                               long sy, int xcd) {
    const BlockId bid = xcd ? xcd_grid() : BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
    using S = ZW<NX>;
    extern __shared__ double2 lds[];
    for (int i = threadIdx.x; i < NX; i += blockDim.x) lds[i] = twg[i];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const XPlace w = x_place<S>(g, bid.x * (blockDim.x / 64) + wave);
    if (w.y >= g.Ny) return;
    double2 v[S::N2];
    x_forward<NX>(g, zo0 + bid.z * sx, bid.y, w, lds + NX + (wave * S::LPW + w.L) * S::LBUF, lds, v);
    const double scale = 1.0 / ((double)g.Nx * g.Nz);
    const gbytes_w out = reinterpret_cast<gbytes_w>(gmem_w(fo0) + bid.z * sy + ((long)bid.y * g.Ny + w.y) * g.M);
    x_live<NX>(x_bins(g, w.ikz, w.j, w.line_ok && w.j < S::N1), w.j,
               [&](int p, int dist, unsigned at, int) { gstore(out + dist, at, make_double2(v[p].x * scale, v[p].y * scale)); });
}

// The same for the skew-symmetric form's 8 fields, with the x-derivative part of
// its divergence added here, in x-spectral space: task c < 3 writes field c as
// f_c + 1/2 i kx (u_c u_0) (u_c u_0 is z-pass field 3 + c), task 1 also u_0u_1 as
// field 3, task 3 writes u_1u_1 (z-pass field 6) and u_1u_2 (7) as fields 4 and 5.
// The y-forward transform then reads f_c and u_c u_1 only. A task is a pair of
// wavefronts with a field each; the second hands its spectrum to the first through
// its LDS rows. One wavefront with both fields in turn held twice the registers and
// ran twice the chain (us per launch, before -> after, with the accesses as above
// after: one 32^3 field 5.5 -> 4.2, 64^3 7.1 -> 6.2, 96^3 17.6 -> 16.1, 24 of 32^3
// 13.3 -> 11.5, 4 of 96^3 54.9 -> 52.6; 16 of 64^3, 254 MB, 63.3 -> 64.6).
template <int NX>
__global__ void __launch_bounds__(256) k_xwfold(Geom g, const double2* __restrict__ twg,
                                                const double2* __restrict__ zo0, long sx, double2* __restrict__ fo0,
                                                long sy, int xcd) {
    const BlockId bid = xcd ? xcd_grid() : BlockId{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
    using S = ZW<NX>;
    constexpr int N1 = S::N1, N2 = S::N2;
    extern __shared__ double2 lds[];
    for (int i = threadIdx.x; i < NX; i += blockDim.x) lds[i] = twg[i];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), half = wave & 1;
    const XPlace w = x_place<S>(g, bid.x * (blockDim.x / 128) + wave / 2);
    const bool have = w.y < g.Ny;  // of the whole wavefront
    const int t = bid.y, j = w.j;
    double2* const T = lds + NX + (wave * S::LPW + w.L) * S::LBUF;
    double2 v[N2];
    if (have) x_forward<NX>(g, zo0 + bid.z * sx, t < 3 ? t + 3 * half : 6 + half, w, T, lds, v);
    const double scale = 1.0 / ((double)g.Nx * g.Nz);
#pragma unroll
    for (int p = 0; p < N2; ++p) v[p] = make_double2(v[p].x * scale, v[p].y * scale);
    if (t < 3) {
        wave_lds_sync();
        if (half && j < N1) {
#pragma unroll
            for (int p = 0; p < N2; ++p) T[j + N1 * p] = v[p];
        }
        __syncthreads();
    }
    if (!have || (half && t != 1 && t != 3)) return;
    const XBins bins = x_bins(g, w.ikz, j, w.line_ok && j < N1);
    const int o = t == 3 ? 4 + half : half ? 3 : t;
    const gbytes_w out = reinterpret_cast<gbytes_w>(gmem_w(fo0) + bid.z * sy + ((long)o * g.Ny + w.y) * g.M);
    const double2* const Tb = T + S::LPW * S::LBUF;  // the second wavefront's rows
    if (t < 3 && !half) {
        const double dk = PI / g.Lx;
        x_live<NX>(bins, j, [&](int p, int dist, unsigned at, int kx) {
            const double2 b = Tb[j + N1 * p];
            const double hk = dk * kx;  // f_c + 1/2 i (2 pi kx / Lx) b
            gstore(out + dist, at, make_double2(fma(-hk, b.y, v[p].x), fma(hk, b.x, v[p].y)));
        });
    } else {
        x_live<NX>(bins, j, [&](int p, int dist, unsigned at, int) { gstore(out + dist, at, v[p]); });
    }
}

// ---- y transforms as LDS-tiled contractions ----------------------------------
// Both directions are dense Ny x Ny products over the Chebyshev index applied to
// every (component, mode) column. A block computes YB_M modes x YB_R output
// rows of one member; the contraction index runs through LDS in chunks of
// YB_K, and each thread accumulates a 2 x 2 (mode, row) micro-tile of every
// product it needs, so the epilogue that mixes components (vorticity, base
// flow, divergence terms) stays in registers. Row tiles of one mode tile are
// adjacent in launch order, so the input tile's re-reads come from L2.
constexpr int YB_M = 32, YB_R = 32, YB_K = 16;

// Chebyshev -> y values (same outputs as k_yinv). QM: which components need T*D.
template <int METHOD>
__global__ void __launch_bounds__(256) k_yinv_t(Geom g, YMats ym, const NLMember* __restrict__ tab,
                                                double2* __restrict__ yp0, long sy) {
    constexpr bool Q0 = (METHOD != NL_DIV), Q1 = (METHOD == NL_CONV || METHOD == NL_SKEW), Q2 = (METHOD != NL_DIV);
    constexpr bool QA = Q0 || Q1 || Q2;
    __shared__ double2 Xs[3][YB_K][YB_M];
    __shared__ double As[2][YB_R][YB_K + 1];
    const NLMember& me = tab[blockIdx.y];
    const double2* __restrict__ u = reinterpret_cast<const double2*>(me.u);
    double2* __restrict__ yp = yp0 + blockIdx.y * sy;
    const int Ny = g.Ny;
    const long M = g.M;
    const int nrt = (Ny + YB_R - 1) / YB_R;
    const int m0 = (blockIdx.x / nrt) * YB_M, y0 = (blockIdx.x % nrt) * YB_R;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    double2 P[3][2][2], Q[3][2][2];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) P[c][i][j] = Q[c][i][j] = make_double2(0.0, 0.0);
    for (int k0 = 0; k0 < Ny; k0 += YB_K) {
        for (int i = threadIdx.x; i < 3 * YB_K * YB_M; i += 256) {
            const int mm = i % YB_M, kk = (i / YB_M) % YB_K, c = i / (YB_M * YB_K);
            const int k = k0 + kk, m = m0 + mm;
            Xs[c][kk][mm] = (k < Ny && m < M) ? u[((long)c * Ny + k) * M + m] : make_double2(0.0, 0.0);
        }
        for (int i = threadIdx.x; i < (QA ? 2 : 1) * YB_R * YB_K; i += 256) {
            const int kk = i % YB_K, r = (i / YB_K) % YB_R, a = i / (YB_K * YB_R);
            const int k = k0 + kk, y = y0 + r;
            As[a][r][kk] = (k < Ny && y < Ny) ? (a == 0 ? ym.T : ym.TD)[(long)y * Ny + k] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < YB_K; ++kk) {
            double t[2], d[2];
            double2 x[3][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                t[j] = As[0][ty + 16 * j][kk];
                d[j] = QA ? As[1][ty + 16 * j][kk] : 0.0;
            }
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int i = 0; i < 2; ++i) x[c][i] = Xs[c][kk][tx + 16 * i];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        P[c][i][j].x += t[j] * x[c][i].x;
                        P[c][i][j].y += t[j] * x[c][i].y;
                    }
                    if (Q0) { Q[0][i][j].x += d[j] * x[0][i].x; Q[0][i][j].y += d[j] * x[0][i].y; }
                    if (Q1) { Q[1][i][j].x += d[j] * x[1][i].x; Q[1][i][j].y += d[j] * x[1][i].y; }
                    if (Q2) { Q[2][i][j].x += d[j] * x[2][i].x; Q[2][i][j].y += d[j] * x[2][i].y; }
                }
        }
        __syncthreads();
    }
    const double* __restrict__ base = me.base;
    const double Vsuck = me.Vsuck;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + tx + 16 * i;
        if (m >= M) continue;
        const int ikx = m % g.nkx, ikz = m / g.nkx;
        const double dx = 2 * PI * kx_of(g, ikx) / g.Lx, dz = 2 * PI * ikz / g.Lz;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int y = y0 + ty + 16 * j;
            if (y >= Ny) continue;
            double2 p0 = P[0][i][j], p1 = P[1][i][j], p2 = P[2][i][j];
            double2 q0 = Q[0][i][j], q1 = Q[1][i][j], q2 = Q[2][i][j];
            if (m == 0) {  // base flow on the kx = kz = 0 mode (nse.cpp:28-36)
                p0.x += base[0 * Ny + y];
                q0.x += base[1 * Ny + y];
                p2.x += base[2 * Ny + y];
                q2.x += base[3 * Ny + y];
                p1.x -= Vsuck;
            }
            double2 o[6];
            o[0] = p0;
            o[1] = p1;
            o[2] = p2;
            int nout = 3;
            if (METHOD == NL_ROT) {
                o[3] = csub(q2, imul(dz, p1));               // dw/dy - dv/dz
                o[4] = csub(imul(dz, p0), imul(dx, p2));     // du/dz - dw/dx
                o[5] = csub(imul(dx, p1), q0);               // dv/dx - du/dy
                nout = 6;
            } else if (METHOD == NL_CONV || METHOD == NL_SKEW) {
                o[3] = q0;
                o[4] = q1;
                o[5] = q2;
                nout = 6;
            }
            for (int f = 0; f < nout; ++f) yp[((long)f * Ny + y) * M + m] = o[f];
        }
    }
}

// y values -> Chebyshev coefficients (same outputs as k_yfwd): f_i = Ti G_i + DTi H_i.
template <int METHOD>
__global__ void __launch_bounds__(256) k_yfwd_t(Geom g, YMats ym, int have_g, const double2* __restrict__ fo0,
                                                long sy, const NLMember* __restrict__ tab, int xfold) {
    constexpr bool DIVF = (METHOD == NL_DIV || METHOD == NL_SKEW);
    constexpr int NX = DIVF ? 6 : 3;
    __shared__ double2 Xs[NX][YB_K][YB_M];
    __shared__ double As[2][YB_R][YB_K + 1];
    const double2* __restrict__ fo = fo0 + blockIdx.y * sy;
    double2* __restrict__ f = reinterpret_cast<double2*>(tab[blockIdx.y].f);
    const int Ny = g.Ny;
    const long M = g.M;
    const int nrt = (Ny + YB_R - 1) / YB_R;
    const int m0 = (blockIdx.x / nrt) * YB_M, k0o = (blockIdx.x % nrt) * YB_R;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    const double beta = (METHOD == NL_SKEW) ? 0.5 : 1.0;
    double2 Acc[3][2][2];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) Acc[c][i][j] = make_double2(0.0, 0.0);
    for (int y0 = 0; y0 < Ny; y0 += YB_K) {
        // G_i = g_i + beta (ikx uu_i0 + ikz uu_i2), H_i = beta uu_i1 (uu index -> fo field: 00:3 01:4 02:5 11:6
        // 12:7 22:8). The skew-symmetric z pass has already added beta ikz uu_i2 to g_i (and keeps no uu22).
        for (int i = threadIdx.x; i < 3 * YB_K * YB_M; i += 256) {
            const int mm = i % YB_M, kk = (i / YB_M) % YB_K, c = i / (YB_M * YB_K);
            const int y = y0 + kk, m = m0 + mm;
            double2 G = make_double2(0.0, 0.0), H = make_double2(0.0, 0.0);
            if (y < Ny && m < M) {
                if (have_g) G = fo[((long)c * Ny + y) * M + m];
                if (DIVF && METHOD == NL_SKEW && xfold) {  // x and z terms already in g_c; uu_c1 is field 3 + c
                    const double2 x1 = fo[((long)(3 + c) * Ny + y) * M + m];
                    H = make_double2(beta * x1.x, beta * x1.y);
                } else if (DIVF) {
                    const int ikx = m % g.nkx, ikz = m / g.nkx;
                    const double dx = 2 * PI * kx_of(g, ikx) / g.Lx, dz = 2 * PI * ikz / g.Lz;
                    const int uuf[3][3] = {{3, 4, 5}, {4, 6, 7}, {5, 7, 8}};
                    const double2 x0 = fo[((long)uuf[c][0] * Ny + y) * M + m];
                    const double2 x1 = fo[((long)uuf[c][1] * Ny + y) * M + m];
                    double2 d = imul(dx, x0);
                    if (METHOD == NL_DIV) d = cadd(d, imul(dz, fo[((long)uuf[c][2] * Ny + y) * M + m]));
                    G = make_double2(G.x + beta * d.x, G.y + beta * d.y);
                    H = make_double2(beta * x1.x, beta * x1.y);
                }
            }
            Xs[c][kk][mm] = G;
            if (DIVF) Xs[3 + c][kk][mm] = H;
        }
        for (int i = threadIdx.x; i < (DIVF ? 2 : 1) * YB_R * YB_K; i += 256) {
            const int kk = i % YB_K, r = (i / YB_K) % YB_R, a = i / (YB_K * YB_R);
            const int y = y0 + kk, k = k0o + r;
            As[a][r][kk] = (k < Ny && y < Ny) ? (a == 0 ? ym.Ti : ym.DTi)[(long)k * Ny + y] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int kk = 0; kk < YB_K; ++kk) {
            double t[2], d[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                t[j] = As[0][ty + 16 * j][kk];
                d[j] = DIVF ? As[1][ty + 16 * j][kk] : 0.0;
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double2 xg[2], xh[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    xg[i] = Xs[c][kk][tx + 16 * i];
                    xh[i] = DIVF ? Xs[3 * DIVF + c][kk][tx + 16 * i] : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        Acc[c][i][j].x += t[j] * xg[i].x;
                        Acc[c][i][j].y += t[j] * xg[i].y;
                        if (DIVF) {
                            Acc[c][i][j].x += d[j] * xh[i].x;
                            Acc[c][i][j].y += d[j] * xh[i].y;
                        }
                    }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = m0 + tx + 16 * i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int k = k0o + ty + 16 * j;
            if (k >= Ny) continue;
            for (int c = 0; c < 3; ++c) f[((long)c * Ny + k) * M + m] = Acc[c][i][j];
        }
    }
}

// ---- y transforms on the FP64 matrix cores ----------------------------------
// v_mfma_f64_16x16x4f64 (one wave: D = A B + C, A 16x4, B 4x16, D 16x16).
// Operand layout, lane l: A[l % 16][l / 16], B[l / 16][l % 16]; result
// register r of lane l is D[4 r + l / 16][l % 16].
//
// A block is three waves per transform matrix; wave c handles velocity
// component c of YW_MODES = 8 consecutive modes, i.e. 16 real columns (real,
// imaginary part of each mode), over all output rows of the block. Each lane's B
// operand streams from HBM straight into registers, one chunk ahead; the chunk of
// the transform matrices, shared by the waves, is staged in LDS. The matrices come
// in the order in which they are staged (y_tiles): a chunk is one contiguous copy in
// 16-byte pieces. Picked entry by entry out of the row-major matrices, with the row,
// column and bounds formed for each, the staging took half the kernels' VALU
// instructions; us per launch, before -> after (inverse, forward): one 32^3 field
// 5.4 -> 4.8, 6.0 -> 4.7; 64^3 10.8 -> 6.9 (with the row split), 11.6 -> 8.6; 96^3
// 17.0 -> 14.4, 19.1 -> 13.8; 128^3 convection 41 -> 35, 22 -> 19; 192x129x192 81 ->
// 63, 44 -> 35 (57.5 and 28.4 with the addressing below); 16 of 64^3 52 -> 46, 51 -> 44. The inverse at 192x129x192 then takes
// 24 us for its loads alone, 23 us of matrix products at their peak rate and writes
// 96 MB (20 us at the copy rate), one after the other in each block. Loading two or
// three chunks ahead is slower (67, 72), and so are two column tiles per wave (71: the
// registers leave half the blocks).
//
// Both transforms use the mirror symmetry of the Chebyshev points,
// y_{Ny-1-j} = -y_j: T[Ny-1-j][k] = (-1)^k T[j][k], and the derivative flips
// the parity. Only the upper half of the points (j < (Ny+1)/2) enters the
// products, split by the parity of k, which halves the matrix work.
typedef double mfma4d __attribute__((ext_vector_type(4)));
constexpr int YW_MODES = 8;

__device__ __forceinline__ mfma4d mfma16x16x4(double a, double b, mfma4d c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Waves per SIMD the register allocation of a wave-column kernel must allow:
// the accumulators take 16 NRT registers, the rest is operand staging (without
// a bound the scheduler hoists a whole chunk's LDS reads) and, in the inverse,
// the next matrix chunk in flight.
constexpr int yw_waves(int nrt) { return nrt <= 3 ? 4 : (nrt <= 4 ? 3 : 2); }
// The forward transform also holds sums and differences of mirrored values of
// the prefetched chunk, and the next matrix chunk in flight (two matrices in
// the divergence forms).
constexpr int yw_waves_fwd(bool divf, int nrt) { return nrt <= 1 ? 4 : (nrt <= (divf ? 2 : 3) ? 3 : 2); }

// Chebyshev -> y values (outputs as k_yinv_t): p = T u and, unless the form is
// the divergence one, q = T D u = du/dy values. Waves 0-2 compute p of
// components 0-2, waves 3-5 q; the two halves read the same coefficient
// columns (the second read is served by the caches). For an upper point
// j < Ny/2, E = sum over even k, O = sum over odd k: p_j = E + O,
// p_{Ny-1-j} = E - O, q_j = E + O, q_{Ny-1-j} = O - E. The middle point of an
// odd Ny is a dot product per lane, summed over the lane groups. NRT: row
// tiles of 16 upper points.
template <int METHOD, int NRT, int NSP>
__global__ void __launch_bounds__(METHOD == NL_DIV ? 192 : 384) __attribute__((amdgpu_waves_per_eu(yw_waves(NRT))))
    k_yinv_w(Geom g, YMats ym, const NLMember* __restrict__ tab, double2* __restrict__ yp0, long sy) {
    const BlockId bid = xcd_grid();  // neighbouring blocks on one XCD
    constexpr int NMAT = (METHOD == NL_DIV) ? 1 : 2, NT = 192 * NMAT;
    constexpr int KC = YINV_KC, AP = KC + 1, EP = 17;  // chunk columns: 8 even k, then 8 odd k
    constexpr int RS = NRT * 16 + 1;                   // LDS rows per matrix: tiles, middle point
    // two matrix chunk buffers: chunk i + 1 is loaded into registers while
    // chunk i is multiplied, and stored to the other buffer after it. A chunk is
    // one contiguous piece of ym.inv, laid out as it lies in LDS.
    constexpr int SM = yinv_tile(NRT), SA = NMAT * SM, SE = NMAT * 3 * 2 * 16 * EP;
    constexpr int NST = (SA / 2 + NT - 1) / NT;  // 16-byte pieces per thread
    static_assert(SM == RS * AP + 1 && SM % 2 == 0, "the staged chunk's layout");
    __shared__ __align__(16) double sm[2 * SA > SE ? 2 * SA : SE];
    const NLMember& me = tab[bid.y];
    double2* __restrict__ yp = yp0 + bid.y * sy;
    const int Ny = g.Ny, nm = Ny / 2, mid = (Ny & 1) ? nm : -1;
    const long M = g.M;
    const int nrt = (nm + 15) / 16;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = w % 3, am = w / 3, l = threadIdx.x & 63, lr = l & 15, lk = l >> 4;
    const int sp = bid.x % NSP, rt0 = sp * NRT;  // this block's row tiles
    const long m0 = (long)(bid.x / NSP) * YW_MODES;
    const long mcol = m0 + (lr >> 1);
    // Two and four row tiles load without conditions (modes past M read mode M - 1 and are
    // dropped, coefficients past Ny meet zeros of the staged matrix) at a uniform base
    // and a 32-bit lane offset: 80 registers, not 89, and so 6 wavefronts, four blocks
    // (128^3 31.4 -> 29.9 us, convection 33.2 -> 31.0, 192x129x192 62.6 -> 57.5). Where the
    // occupancy stays the same the condition saves the loads (one 32^3 field 4.7
    // against 4.9, 96^3 14.2 against 14.5).
    constexpr bool ALL = NRT % 2 == 0;
    const bool mok = mcol < M;
    const gbytes ub = reinterpret_cast<gbytes>(gmem(me.u) + 2 * (long)c * Ny * M);
    const unsigned uoff = (unsigned)(2 * min(mcol, M - 1) + (l & 1)) * 8u;
    auto coefficient = [&](int k) {
        if (ALL) return *reinterpret_cast<gcdouble>(ub + (16L * min(k, Ny - 1) * M + uoff));
        return (mok && k < Ny) ? *reinterpret_cast<gcdouble>(ub + (16L * k * M + uoff)) : 0.0;
    };
    const int nch = yinv_chunks(Ny), kend = nch * KC;
    mfma4d ae[NRT], ao[NRT];
    double dmid = 0.0;
    double bn[4];  // [parity * 2 + step]: k = k0 + 2 (4 step + lane / 16) + parity
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = k0 + 2 * (4 * (i & 1) + lk) + (i >> 1);
            bn[i] = coefficient(k);
        }
    };
    dvec2 mv[NST];
    auto load_mat = [&](int k0) {
        const auto src = gmem(reinterpret_cast<const dvec2*>(ym.inv + ((long)sp * nch + k0 / KC) * 2 * SM));
#pragma unroll
        for (int s = 0; s < NST; ++s) mv[s] = src[min((int)threadIdx.x + s * NT, SA / 2 - 1)];
    };
    // the remainder of the contraction, straight from the caches (zero without one)
    double ta[NRT][2], tm[2] = {0.0, 0.0}, tb[2] = {0.0, 0.0};
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) ta[rt][0] = ta[rt][1] = 0.0;
    if (kend < Ny) {
        const gcdouble tail = gmem(ym.inv) + (long)NSP * nch * 2 * SM + (sp * 2 + am) * yinv_tail(NRT);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int k = kend + 2 * lk + p;
            tb[p] = coefficient(k);
            tm[p] = tail[2 * 64 * NRT + 4 * p + lk];
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt) ta[rt][p] = tail[(rt * 2 + p) * 64 + l];
        }
    }
    fetch(0);
    load_mat(0);
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        ae[rt] = mfma16x16x4(ta[rt][0], tb[0], mfma4d{0.0, 0.0, 0.0, 0.0});
        ao[rt] = mfma16x16x4(ta[rt][1], tb[1], mfma4d{0.0, 0.0, 0.0, 0.0});
    }
    dmid = fma(tm[0], tb[0], tm[1] * tb[1]);
    for (int k0 = 0, buf = 0; k0 < kend; k0 += KC, buf ^= 1) {
        double b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = bn[i];
        // buffer buf was last read two chunks ago, before every thread passed
        // the previous chunk's barrier
        double* __restrict__ sb = sm + buf * SA;
#pragma unroll
        for (int s = 0; s < NST; ++s) {
            const int i = threadIdx.x + s * NT;
            if (i < SA / 2) reinterpret_cast<dvec2*>(sb)[i] = mv[s];
        }
        __syncthreads();
        if (k0 + KC < kend) {
            fetch(k0 + KC);
            load_mat(k0 + KC);
        }
        const double* __restrict__ arow = sb + am * SM + lr * AP + lk;
        const double* __restrict__ amid = sb + am * SM + NRT * 16 * AP + lk;
        if (METHOD == NL_ROT && w == 4) continue;  // dv/dy, which no vorticity component needs (uniform)
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            // unconditional: staged rows and columns past the grid are zero,
            // and a conditional update keeps the tiles from staying in place
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt) {
                ae[rt] = mfma16x16x4(arow[rt * 16 * AP + 4 * st], b[st], ae[rt]);
                ao[rt] = mfma16x16x4(arow[rt * 16 * AP + 8 + 4 * st], b[2 + st], ao[rt]);
            }
            dmid = fma(amid[4 * st], b[st], fma(amid[8 + 4 * st], b[2 + st], dmid));
            __builtin_amdgcn_sched_barrier(0);  // keep each step's operand reads next to its MFMAs
        }
    }
    const int pm = threadIdx.x & 7;
    const long m = m0 + pm;
    const int ikx = (int)(m % g.nkx), ikz = (int)(m / g.nkx);
    const double dx = 2 * PI * kx_of(g, ikx) / g.Lx, dz = 2 * PI * ikz / g.Lz;
    // outputs of one point from the exchange rows: p of component cc at e + cc * ps, q at e + (3 + cc) * ps
    auto emit = [&](int y, const double* e, int ps) {
        double2 p[3], q[3];
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            p[cc] = make_double2(e[cc * ps], e[cc * ps + 1]);
            q[cc] = NMAT == 2 ? make_double2(e[(3 + cc) * ps], e[(3 + cc) * ps + 1]) : make_double2(0.0, 0.0);
        }
        if (m == 0) {  // base flow on the kx = kz = 0 mode (nse.cpp:28-36)
            const gcdouble base = gmem(me.base);
            p[0].x += base[0 * Ny + y];
            q[0].x += base[1 * Ny + y];
            p[2].x += base[2 * Ny + y];
            q[2].x += base[3 * Ny + y];
            p[1].x -= me.Vsuck;
        }
        double2 o[6];
        o[0] = p[0];
        o[1] = p[1];
        o[2] = p[2];
        int nout = 3;
        if (METHOD == NL_ROT) {
            o[3] = csub(q[2], imul(dz, p[1]));            // dw/dy - dv/dz
            o[4] = csub(imul(dz, p[0]), imul(dx, p[2]));  // du/dz - dw/dx
            o[5] = csub(imul(dx, p[1]), q[0]);            // dv/dx - du/dy
            nout = 6;
        } else if (METHOD == NL_CONV || METHOD == NL_SKEW) {
            o[3] = q[0];
            o[4] = q[1];
            o[5] = q[2];
            nout = 6;
        }
        for (int f = 0; f < nout; ++f) yp[((long)f * Ny + y) * M + m] = o[f];
    };
    // row tiles: the components and both halves meet in LDS
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        if (rt0 + rt >= nrt) continue;  // uniform
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double e = ae[rt][r], o = ao[rt][r];
            sm[(((am * 3 + c) * 2 + 0) * 16 + 4 * r + lk) * EP + lr] = e + o;
            sm[(((am * 3 + c) * 2 + 1) * 16 + 4 * r + lk) * EP + lr] = am == 0 ? e - o : o - e;
        }
        __syncthreads();
        for (int pt = threadIdx.x; pt < 256; pt += NT) {
            const int half = pt >> 7, pr = (pt >> 3) & 15;
            const int yt = (rt0 + rt) * 16 + pr;
            if (yt >= nm || m >= M) continue;
            emit(half ? Ny - 1 - yt : yt, sm + (half * 16 + pr) * EP + 2 * pm, 2 * 16 * EP);
        }
    }
    if (mid < 0 || sp != NSP - 1) return;  // uniform
    dmid += __shfl_xor(dmid, 16);
    dmid += __shfl_xor(dmid, 32);
    __syncthreads();
    if (lk == 0) sm[(am * 3 + c) * EP + lr] = dmid;
    __syncthreads();
    if (threadIdx.x < YW_MODES && m < M) emit(mid, sm + 2 * pm, EP);
}

// y values -> Chebyshev coefficients (outputs as k_yfwd_t): f_c = Ti G_c +
// DTi H_c, with G_c = g_c + beta (i kx uu_c0 + i kz uu_c2) and H_c = beta uu_c1
// for the divergence forms (beta 1/2 in the skew-symmetric one), G_c = g_c
// otherwise. With S, D the sum and difference of the values at an upper point
// and its mirror (the middle point of an odd Ny counted once):
// f_{2i} = Ti S_G + DTi D_H, f_{2i+1} = Ti D_G + DTi S_H over the upper points.
// The MFMA tiles hold i < Ny/2; the last coefficient of an odd Ny (k = Ny-1)
// is a dot product per lane, summed over the lane groups. NRT: row tiles of 16
// coefficients of each parity.
template <int METHOD, int NRT>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(yw_waves_fwd(METHOD == NL_DIV || METHOD == NL_SKEW, NRT)))) k_yfwd_w(Geom g, YMats ym, int have_g, const double2* __restrict__ fo0,
                                                long sy, const NLMember* __restrict__ tab, int xfold) {
    const BlockId bid = xcd_grid();  // neighbouring blocks on one XCD
    constexpr bool DIVF = (METHOD == NL_DIV || METHOD == NL_SKEW);
    constexpr int NMAT = DIVF ? 2 : 1;
    constexpr int KC = YFWD_KC, AP = KC + 1, NS = KC / 4;
    // two matrix chunk buffers, as in k_yinv_w, unless the chunk in flight
    // would not fit the registers (two matrices of 6 or 8 row tiles): then one
    // buffer, loaded and stored between two barriers
    constexpr int SM = yfwd_tile(NRT), SA = NMAT * SM, NST = (SA / 2 + 191) / 192;
    static_assert(SM % 2 == 0, "16-byte pieces");
    constexpr bool DB = !(DIVF && NRT >= 6);
    __shared__ __align__(16) double sm[(DB ? 2 : 1) * SA];
    const double* __restrict__ fo = reinterpret_cast<const double*>(fo0 + bid.y * sy);
    __attribute__((address_space(1))) double* __restrict__ f = gmem_w(tab[bid.y].f);
    const int Ny = g.Ny, nh = (Ny + 1) / 2, nm = Ny / 2;
    const bool odd = Ny & 1;
    const long M = g.M;
    const int c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, lr = l & 15, lk = l >> 4, part = l & 1;
    const long mcol = (long)bid.x * YW_MODES + (lr >> 1);
    const bool mok = mcol < M;
    const double beta = (METHOD == NL_SKEW) ? 0.5 : 1.0;
    double sdx = 0, sdz = 0;  // i k multiplication of the other part, with its sign
    if (DIVF) {
        const int ikx = (int)(mcol % g.nkx), ikz = (int)(mcol / g.nkx);
        const double sg = part ? beta : -beta;
        sdx = sg * 2 * PI * kx_of(g, ikx) / g.Lx;
        sdz = sg * 2 * PI * ikz / g.Lz;
    }
    // field of uu_cj in fo: 00:3 01:4 02:5 11:6 12:7 22:8. The skew-symmetric
    // z pass has already added beta ikz uu_c2 to g_c (and keeps no uu22); with
    // xfold the forward x-FFT has added beta ikx uu_c0 too, and uu_c1 is field
    // 3 + c.
    constexpr bool ZTERM = (METHOD == NL_DIV);
    const bool XTERM = !(METHOD == NL_SKEW && xfold);
    const int f0 = c == 0 ? 3 : (c == 1 ? 4 : 5), f2 = c == 0 ? 5 : (c == 1 ? 7 : 8);
    const int f1 = XTERM ? (c == 0 ? 4 : (c == 1 ? 6 : 7)) : 3 + c;
    // Every access is at a component's uniform base and a 32-bit lane offset; with a
    // 64-bit pointer per field and lane two to four row tiles held 16 registers more,
    // a wavefront per SIMD less (us per launch, before -> after: 192x129x192 34.1 ->
    // 28.4, 128^3 18.2 -> 17.3, 16 of 64^3 45.0 -> 42.3, 4 of 96^3 40.1 -> 38.4, 54x57x72
    // 8.8 -> 8.1). Columns past M read mode M - 1 (every field of fo has Ny x M modes);
    // the values are masked where they are used.
    const unsigned rowb = (unsigned)M * 16u, mcl = (unsigned)(mok ? mcol : M - 1);
    const unsigned own = (2 * mcl + part) * 8u, other = (2 * mcl + 1 - part) * 8u;
    auto field = [&](int i) { return reinterpret_cast<gbytes>(gmem(fo) + 2 * (long)i * Ny * M); };
    const gbytes pg = field(c), p0 = field(f0), p1 = field(f1), p2 = field(f2);
    auto at = [](gbytes b, unsigned o) { return *reinterpret_cast<gcdouble>(b + o); };
    const int nch = yfwd_chunks(nh), yend = nch * KC;
    mfma4d ae[NRT], ao[NRT];
    double dlast = 0.0;
    // Raw values of a chunk, per step: g at the upper point and its mirror,
    // then (divergence forms) uu_c1, then the x and z terms of G. They are
    // loaded without branches, at clamped addresses, and combined only when
    // the chunk is multiplied: a load under a lane condition whose value is
    // used at once gets its own wait, and the chunk's loads were then
    // serialized instead of in flight behind the previous chunk's products.
    constexpr int NR = DIVF ? 8 : 2;
    double rv[NS][NR];
    auto fetch1 = [&](int y0, double (&r)[NR]) {
        const int y = min(y0 + lk, nh - 1), ymr = Ny - 1 - y;
        const unsigned u = y * rowb, d = ymr * rowb;
        r[0] = at(pg, u + own);
        r[1] = at(pg, d + own);
        if (DIVF) {
            r[2] = at(p1, u + own);
            r[3] = at(p1, d + own);
            if (XTERM) {
                r[4] = at(p0, u + other);
                r[5] = at(p0, d + other);
            }
            if (ZTERM) {
                r[6] = at(p2, u + other);
                r[7] = at(p2, d + other);
            }
        }
    };
    auto fetch = [&](int y0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) fetch1(y0 + 4 * s, rv[s]);
    };
    // G at a point from its raw values (i: 0 the upper point, 1 its mirror)
    auto gval = [&](const double* r, int i) {
        double G = have_g ? r[i] : 0.0;
        if (DIVF && XTERM) G += ZTERM ? sdx * r[4 + i] + sdz * r[6 + i] : sdx * r[4 + i];
        return G;
    };
    // sums and differences of G and H at an upper point and its mirror
    auto comb = [&](int y, const double (&r)[NR], double& sg, double& dg, double& sh, double& dh) {
        const int ymr = Ny - 1 - y;
        double G = 0, Gm = 0, H = 0, Hm = 0;
        if (mok && y < nh) {
            G = gval(r, 0);
            if (DIVF) H = beta * r[2];
            if (ymr != y) {
                Gm = gval(r, 1);
                if (DIVF) Hm = beta * r[3];
            }
        }
        sg = G + Gm;
        dg = G - Gm;
        sh = H + Hm;
        dh = H - Hm;
    };
    dvec2 mv[NST];
    auto mat = [&](int y0) { return gmem(reinterpret_cast<const dvec2*>(ym.fwd + (long)(y0 / KC) * 2 * SM)); };
    auto load_mat = [&](int y0) {
        const auto src = mat(y0);
#pragma unroll
        for (int s = 0; s < NST; ++s) mv[s] = src[min((int)threadIdx.x + s * 192, SA / 2 - 1)];
    };
    // the remainder of the contraction, straight from the caches (zero without one)
    double ta[NMAT][NRT][2], tl[NMAT], rt0[NR];
#pragma unroll
    for (int a = 0; a < NMAT; ++a) {
        tl[a] = 0.0;
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) ta[a][rt][0] = ta[a][rt][1] = 0.0;
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) rt0[i] = 0.0;
    if (yend < nh) {
        fetch1(yend, rt0);
#pragma unroll
        for (int a = 0; a < NMAT; ++a) {
            const gcdouble tail = gmem(ym.fwd) + (long)nch * 2 * SM + a * yfwd_tail(NRT);
            tl[a] = tail[2 * 64 * NRT + lk];
#pragma unroll
            for (int i = 0; i < 2 * NRT; ++i) ta[a][i >> 1][i & 1] = tail[i * 64 + l];
        }
    }
    fetch(0);
    if (DB) load_mat(0);
    {
        double sg, dg, sh, dh;
        comb(yend + lk, rt0, sg, dg, sh, dh);
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) {
            ae[rt] = mfma16x16x4(ta[0][rt][0], sg, mfma4d{0.0, 0.0, 0.0, 0.0});
            ao[rt] = mfma16x16x4(ta[0][rt][1], dg, mfma4d{0.0, 0.0, 0.0, 0.0});
            if (DIVF) {
                ae[rt] = mfma16x16x4(ta[NMAT - 1][rt][0], dh, ae[rt]);
                ao[rt] = mfma16x16x4(ta[NMAT - 1][rt][1], sh, ao[rt]);
            }
        }
        dlast = tl[0] * sg;
        if (DIVF) dlast = fma(tl[NMAT - 1], dh, dlast);
    }
    for (int y0 = 0, buf = 0; y0 < yend; y0 += KC, buf ^= DB) {
        double sg[NS], dg[NS], sh[NS], dh[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) comb(y0 + 4 * s + lk, rv[s], sg[s], dg[s], sh[s], dh[s]);
        // DB: buffer buf was last read two chunks ago, before every thread
        // passed the previous chunk's barrier
        double* __restrict__ sb = sm + buf * SA;
        if (DB) {
#pragma unroll
            for (int s = 0; s < NST; ++s) {
                const int i = threadIdx.x + s * 192;
                if (i < SA / 2) reinterpret_cast<dvec2*>(sb)[i] = mv[s];
            }
        } else {
            __syncthreads();  // the previous chunk's matrix reads are done
            const auto src = mat(y0);
            for (int i = threadIdx.x; i < SA / 2; i += 192) reinterpret_cast<dvec2*>(sb)[i] = src[i];
        }
        __syncthreads();
        if (y0 + KC < yend) {
            fetch(y0 + KC);
            if (DB) load_mat(y0 + KC);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            // unconditional: staged rows and columns past the grid are zero,
            // and a conditional update keeps the tiles from staying in place
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt) {
                const double* A = sb + (rt * 16 + lr) * AP + 4 * s + lk;
                ae[rt] = mfma16x16x4(A[0], sg[s], ae[rt]);
                ao[rt] = mfma16x16x4(A[NRT * 16 * AP], dg[s], ao[rt]);
                if (DIVF) {
                    ae[rt] = mfma16x16x4(A[SM], dh[s], ae[rt]);
                    ao[rt] = mfma16x16x4(A[SM + NRT * 16 * AP], sh[s], ao[rt]);
                }
            }
            const double* A = sb + 2 * NRT * 16 * AP + 4 * s + lk;
            dlast = fma(A[0], sg[s], dlast);
            if (DIVF) dlast = fma(A[SM], dh[s], dlast);
            __builtin_amdgcn_sched_barrier(0);  // keep each step's operand reads next to its MFMAs
        }
    }
    dlast += __shfl_xor(dlast, 16);
    dlast += __shfl_xor(dlast, 32);
    if (!mok) return;
    const gbytes_w fc = reinterpret_cast<gbytes_w>(f + 2 * (long)c * Ny * M);
    auto put = [&](int k, double v) { *reinterpret_cast<__attribute__((address_space(1))) double*>(fc + (k * rowb + own)) = v; };
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = rt * 16 + 4 * r + lk;
            if (i < nm) {
                put(2 * i, ae[rt][r]);
                put(2 * i + 1, ao[rt][r]);
            }
        }
    }
    if (odd && lk == 0) put(Ny - 1, dlast);
}

// Row-tile count classes with a wave-column kernel; above the last one the
// vector tiles run.
template <int METHOD>
static void launch_yinv(const Geom& g, const YMats& ym, int n, const NLMember* tab, double2* yp, long sy,
                        hipStream_t st) {
    const int cls = yw_class(g.Ny), nt = METHOD == NL_DIV ? 192 : 384;
    auto go = [&](auto c) {
        constexpr int C = decltype(c)::value, NSP = yinv_split(C);
        const dim3 grid((unsigned)((g.M + YW_MODES - 1) / YW_MODES * NSP), n);
        k_yinv_w<METHOD, yinv_rows(C), NSP><<<grid, nt, 0, st>>>(g, ym, tab, yp, sy);
    };
    if (cls == 1) go(std::integral_constant<int, 1>{});
    else if (cls == 2) go(std::integral_constant<int, 2>{});
    else if (cls == 3) go(std::integral_constant<int, 3>{});
    else if (cls == 4) go(std::integral_constant<int, 4>{});
    else if (cls == 6) go(std::integral_constant<int, 6>{});
    else if (cls == 8) go(std::integral_constant<int, 8>{});
    else {
        const dim3 tg((unsigned)(((g.M + YB_M - 1) / YB_M) * ((g.Ny + YB_R - 1) / YB_R)), n);
        k_yinv_t<METHOD><<<tg, 256, 0, st>>>(g, ym, tab, yp, sy);
    }
}

// xfold: the skew-symmetric fields come folded from k_xwfold (f_c with its
// x-derivative term in fields 0-2, u_cu_1 in 3 + c)
template <int METHOD>
static void launch_yfwd(const Geom& g, const YMats& ym, int n, int have_g, const double2* fo, long sy,
                        const NLMember* tab, hipStream_t st, bool xfold = false) {
    const int nrt = (g.Ny / 2 + 15) / 16, xf = xfold ? 1 : 0;
    const dim3 grid((unsigned)((g.M + YW_MODES - 1) / YW_MODES), n);
    if (nrt <= 1) k_yfwd_w<METHOD, 1><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else if (nrt <= 2) k_yfwd_w<METHOD, 2><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else if (nrt <= 3) k_yfwd_w<METHOD, 3><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else if (nrt <= 4) k_yfwd_w<METHOD, 4><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else if (nrt <= 6) k_yfwd_w<METHOD, 6><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else if (nrt <= 8) k_yfwd_w<METHOD, 8><<<grid, 192, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    else {
        const dim3 tg((unsigned)(((g.M + YB_M - 1) / YB_M) * ((g.Ny + YB_R - 1) / YB_R)), n);
        k_yfwd_t<METHOD><<<tg, 256, 0, st>>>(g, ym, have_g, fo, sy, tab, xf);
    }
}

// largest x-FFT lines per block that fit (power of two <= 16, at most the kz lines)
static int xfft_lines_max(const Geom& g) {
    const long per = 32L * lpitch(g.Nx);  // two complex work lines
    const long avail = (long)lds_budget() - 16L * g.Nx;
    int xl = 1;
    while (xl < 16 && xl * 2 <= g.nkz && (long)(xl * 2) * per <= avail) xl *= 2;
    return xl;
}

static int xfft_lines(const Geom& g, const NLTune& tn) {
    const int m = xfft_lines_max(g);
    return tn.xl > 0 ? std::min(tn.xl, m) : std::min(4, m);
}

// fold (forward only): the skew-symmetric layout of k_xwfold (8 z-pass fields in,
// 6 out, the x-derivative part of the divergence added); only the wavefront
// FFT lengths have it. Returns whether it folded.
template <int NX>
static bool launch_x(bool inverse, const Geom& g, const FFTPlan& px, int nsrc, int nf, int n, const double2* in,
                     long sin, double2* out, long sout, const NLTune& tn, hipStream_t st, bool fold) {
    if constexpr (zwave_size(NX)) {
        using S = ZW<NX>;
        const int wb = (!inverse && tn.xwbf > 0) ? tn.xwbf : (tn.xwb > 0 ? tn.xwb : 4);
        const long waves = (long)g.Ny * ((g.nkz + S::LPW - 1) / S::LPW);
        const size_t lds = (size_t)(NX + wb * S::LPW * S::LBUF) * sizeof(double2);
        if (inverse) {
            const dim3 grid((unsigned)((waves + wb - 1) / wb), nf, n);
            allow_lds(k_xwinv<NX>, lds);
            k_xwinv<NX><<<grid, 64 * wb, lds, st>>>(g, px.tw, nsrc, in, sin, out, sout);
        } else {
            if (fold && nf != 8) throw std::runtime_error("x-FFT fold: the skew-symmetric layout has 8 fields");
            const int xcd = (g.nkz * (int)sizeof(double2)) % 128 != 0;
            if (fold) {  // pairs of wavefronts
                const int np = wb > 2 ? 2 : 1;
                const size_t ldsp = (size_t)(NX + 2 * np * S::LPW * S::LBUF) * sizeof(double2);
                allow_lds(k_xwfold<NX>, ldsp);
                k_xwfold<NX><<<dim3((unsigned)((waves + np - 1) / np), 4, n), 128 * np, ldsp, st>>>(
                    g, px.tw, in, sin, out, sout, xcd);
            } else {
                allow_lds(k_xwfwd<NX>, lds);
                k_xwfwd<NX><<<dim3((unsigned)((waves + wb - 1) / wb), nf, n), 64 * wb, lds, st>>>(g, px.tw, in, sin,
                                                                                               out, sout, xcd);
            }
        }
        return fold && !inverse;
    } else {
        const int XL = xfft_lines(g, tn);
        const int nchunk = (g.nkz + XL - 1) / XL;
        const size_t lds = (size_t)(g.Nx + 2 * XL * lpitch(g.Nx)) * sizeof(double2);
        const dim3 grid(g.Ny * nchunk, nf, n);
        if (inverse) {
            allow_lds(k_xinv, lds);
            k_xinv<<<grid, 256, lds, st>>>(g, px, XL, nsrc, in, sin, out, sout);
        } else {
            allow_lds(k_xfwd, lds);
            k_xfwd<<<grid, 256, lds, st>>>(g, px, XL, in, sin, out, sout);
        }
        return false;
    }
}

// in/out strides are per member, in double2. Returns whether the forward
// transform folded the skew-symmetric layout (launch_x).
static bool launch_xfft(bool inverse, const Geom& g, const FFTPlan& px, int nsrc, int nf, int n, const double2* in,
                        long sin, double2* out, long sout, const NLTune& tn, hipStream_t st, bool fold = false) {
    switch (g.Nx) {
#define CASE_X(N) \
    case N: return launch_x<N>(inverse, g, px, nsrc, nf, n, in, sin, out, sout, tn, st, fold);
        CFG_FFT_SIZES(CASE_X)
#undef CASE_X
        default: return launch_x<0>(inverse, g, px, nsrc, nf, n, in, sin, out, sout, tn, st, fold);
    }
}

void launch_cfl(const Geom& g, const YMats& ym, const FFTPlan& px, const FFTPlan& pz, int n, const NLMember* tab,
                const NLWork& w, double* out, hipStream_t st) {
    const long sy = nlwork_y_doubles(g) / 2, sx = nlwork_x_doubles(g) / 2;
    double2* yp = reinterpret_cast<double2*>(w.yp);
    double2* xp = reinterpret_cast<double2*>(w.xp);
    double* part = w.zo;  // n x blocks partial maxima
    launch_yinv<NL_DIV>(g, ym, n, tab, yp, sy, st);
    launch_xfft(true, g, px, 3, 3, n, yp, sy, xp, sx, NLTune{}, st);
    const int nb = launch_zcfl(g, pz, n, tab, xp, sx, part, st);
    launch_cfl_reduce(n, nb, part, out, st);
}

// Nonlinear term of n members of one grid class. rotating: some member has a
// nonzero rotation (only then does the divergence form compute g).
void launch_nonlinear(const Geom& g, const YMats& ym, const FFTPlan& px, const FFTPlan& pz, int method, int n,
                      const NLMember* tab, bool rotating, const NLWork& w, const NLTune& tn, hipStream_t st,
                      KTimer* kt) {
    KTimer dummy;
    KTimer& T = kt ? *kt : dummy;
    const long sy = nlwork_y_doubles(g) / 2, sx = nlwork_x_doubles(g) / 2;  // per-member strides in double2
    double2* yp = reinterpret_cast<double2*>(w.yp);
    double2* xp = reinterpret_cast<double2*>(w.xp);
    double2* zo = reinterpret_cast<double2*>(w.zo);
    double2* fo = reinterpret_cast<double2*>(w.fo);
    int nsrc = 3, nxout = 3;
    hipEvent_t ev = T.begin();
    switch (method) {
        case NL_ROT:
            launch_yinv<NL_ROT>(g, ym, n, tab, yp, sy, st);
            nsrc = 6; nxout = 6;
            break;
        case NL_CONV:
            launch_yinv<NL_CONV>(g, ym, n, tab, yp, sy, st);
            nsrc = 6; nxout = 9;
            break;
        case NL_SKEW:
            launch_yinv<NL_SKEW>(g, ym, n, tab, yp, sy, st);
            nsrc = 6; nxout = 9;
            break;
        default:
            launch_yinv<NL_DIV>(g, ym, n, tab, yp, sy, st);
            nsrc = 3; nxout = 3;
    }
    T.end(K_YINV, ev);
    ev = T.begin();
    // d/dx outputs (fields nsrc..) derive from fields 0..2 only
    launch_xfft(true, g, px, nsrc == 6 && nxout == 9 ? 6 : nxout, nxout, n, yp, sy, xp, sx, tn, st);
    T.end(K_XINV, ev);
    const int want_g = (method != NL_DIV) || rotating;
    ev = T.begin();
    launch_z_any(method, g, pz, n, tab, want_g, xp, zo, sx, tn, st);
    T.end(K_ZPASS, ev);
    ev = T.begin();
    // forward x-FFT of the z-pass outputs that exist: fields 0-2 (g) when
    // want_g, fields 3-8 (u_i u_j) in the divergence form, 3-7 in the
    // skew-symmetric one; one launch when both exist (the fields are
    // contiguous)
    const bool uu = method == NL_DIV || method == NL_SKEW;
    bool xfold = false;  // the skew-symmetric x-derivative terms already in fields 0-2 (k_xwfold)
    if (want_g)
        xfold = launch_xfft(false, g, px, 0, method == NL_SKEW ? 8 : (uu ? 9 : 3), n, zo, sx, fo, sy, tn, st,
                            method == NL_SKEW);
    else if (uu) {
        const long off = 3L * g.Ny * g.Nx * g.nkz;
        const long offo = 3L * g.Ny * g.M;
        launch_xfft(false, g, px, 0, 6, n, zo + off, sx, fo + offo, sy, tn, st);
    }
    T.end(K_XFWD, ev);
    ev = T.begin();
    switch (method) {
        case NL_ROT: launch_yfwd<NL_ROT>(g, ym, n, 1, fo, sy, tab, st); break;
        case NL_CONV: launch_yfwd<NL_CONV>(g, ym, n, 1, fo, sy, tab, st); break;
        case NL_SKEW: launch_yfwd<NL_SKEW>(g, ym, n, 1, fo, sy, tab, st, xfold); break;
        default: launch_yfwd<NL_DIV>(g, ym, n, want_g, fo, sy, tab, st);
    }
    T.end(K_YFWD, ev);
}

// Autotuner of the nonlinear-term tilings: each candidate block shape of the
// z-pass and of the x-FFTs (wavefronts per block for the wavefront FFTs,
// lines per block for the LDS ones) is timed (HIP events, best of 3 after a
// warm launch) on the caller's work buffers and member table. The tiling only
// changes which threads and blocks do a line's butterflies, never the
// arithmetic, so every choice gives bit-identical results.
NLTune tune_nonlinear(const Geom& g, const YMats& ym, const FFTPlan& px, const FFTPlan& pz, int method, int n,
                      const NLMember* tab, bool rotating, const NLWork& w, hipStream_t st) {
    (void)ym;
    const long sy = nlwork_y_doubles(g) / 2, sx = nlwork_x_doubles(g) / 2;
    double2* yp = reinterpret_cast<double2*>(w.yp);
    double2* xp = reinterpret_cast<double2*>(w.xp);
    double2* zo = reinterpret_cast<double2*>(w.zo);
    const int want_g = (method != NL_DIV) || rotating;
    const int nphys = zpass_nphys(method);
    const int nxout = (method == NL_ROT) ? 6 : (method == NL_DIV ? 3 : 9);
    const int nsrc = (method == NL_DIV) ? 3 : 6;
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess) return NLTune{};
    if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return NLTune{};
    }
    // Every candidate runs once to warm up, then all are timed in 5 interleaved
    // rounds (so clock ramps and neighbours' load fall on all of them alike);
    // each keeps its best time.
    auto pick = [&](const std::vector<NLTune>& cands, auto&& launch, const char* what) {
        for (const NLTune& c : cands) launch(c);
        std::vector<float> best(cands.size(), 1e30f);
        for (int r = 0; r < 5; ++r)
            for (size_t i = 0; i < cands.size(); ++i) {
                (void)hipEventRecord(a, st);
                launch(cands[i]);
                (void)hipEventRecord(b, st);
                (void)hipEventSynchronize(b);
                float ms = 0.f;
                (void)hipEventElapsedTime(&ms, a, b);
                best[i] = std::min(best[i], ms);
            }
        size_t k = 0;
        for (size_t i = 1; i < cands.size(); ++i)
            if (best[i] < best[k]) k = i;
        if (std::getenv("CFGPU_TUNE_LOG")) {
            std::fprintf(stderr, "cfg tune %s %dx%dx%d form %d members %d:", what, g.Nx, g.Ny, g.Nz, method, n);
            for (size_t i = 0; i < cands.size(); ++i)
                std::fprintf(stderr, " [zwb %d zxb %d xwb %d xwbf %d xl %d] %.1f us%s", cands[i].zwb,
                             cands[i].zxb, cands[i].xwb, cands[i].xwbf, cands[i].xl, best[i] * 1e3f,
                             i == k ? " *" : "");
            std::fprintf(stderr, "\n");
        }
        return cands[k];
    };
    NLTune out;
    std::vector<NLTune> zc;
    if (zwave_size(g.Nz) && zsplit(method, g.Nz)) {  // three wavefronts per block
    } else if (zwave_size(g.Nz)) {                   // wavefront z pass: wavefronts per block
        // a block of one wavefront of three-step lines, with its own twiddles, leaves
        // the LDS to fewer wavefronts (192x129x192: 68 us against 57 and 57)
        for (int wb = zwave_three(g.Nz) ? 2 : 1; wb <= 4; wb *= 2) {
            NLTune c;
            c.zwb = wb;
            zc.push_back(c);
        }
    } else {  // LDS z pass: lines per block
        for (int xb = 1; xb <= zpass_xb_max(g, nphys); xb *= 2) {
            NLTune c;
            c.zxb = xb;
            zc.push_back(c);
        }
    }
    if (!zc.empty()) {
        const NLTune z = pick(zc, [&](const NLTune& c) { launch_z_any(method, g, pz, n, tab, want_g, xp, zo, sx, c, st); },
                              "z");
        out.zwb = z.zwb;
        out.zxb = z.zxb;
    }
    std::vector<NLTune> xc;  // x-FFTs, timed on the inverse
    if (zwave_size(g.Nx)) {  // wavefront x-FFTs: wavefronts per block
        for (int wb = 1; wb <= 4; wb *= 2) {
            NLTune c;
            c.xwb = wb;
            xc.push_back(c);
        }
    } else {  // LDS x-FFTs: lines per block
        for (int xl = 1; xl <= xfft_lines_max(g); xl *= 2) {
            NLTune c;
            c.xl = xl;
            xc.push_back(c);
        }
    }
    if (!xc.empty()) {
        const NLTune x = pick(xc, [&](const NLTune& c) {
            launch_xfft(true, g, px, nsrc == 6 && nxout == 9 ? 6 : nxout, nxout, n, yp, sy, xp, sx, c, st);
        }, "x");
        out.xwb = x.xwb;
        out.xl = x.xl;
    }
    if (zwave_size(g.Nx) && want_g) {  // the forward wavefront x-FFT on its own (it folds the skew form)
        const int nzf = method == NL_SKEW ? 8 : (method == NL_DIV ? 9 : 3);  // as launch_nonlinear
        std::vector<NLTune> fc;
        for (int wb = method == NL_SKEW ? 2 : 1; wb <= 4; wb *= 2) {  // the fold runs in pairs
            NLTune c;
            c.xwbf = wb;
            fc.push_back(c);
        }
        const NLTune f = pick(fc, [&](const NLTune& c) {
            launch_xfft(false, g, px, 0, nzf, n, zo, sx, yp, sy, c, st, method == NL_SKEW);
        }, "xfwd");
        out.xwbf = f.xwbf;
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return out;
}

}  // namespace cfg
