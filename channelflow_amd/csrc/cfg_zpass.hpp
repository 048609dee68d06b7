// Kernels of the z pass of the nonlinear term (gfx950, FP64): per (y, x) line the
// inverse z-FFTs, the pointwise products and the forward z-FFTs. Each nonlinear
// form is compiled in a file of its own (cfg_z_*.hip).
#pragma once

#include <algorithm>
#include <type_traits>

#include "cfg_fft.hpp"
#include "cfg_wave.hpp"
#include "cfg_z.hpp"

namespace cfg {

// ---- z pass --------------------------------------------------------------
struct ZCtx {
    Geom g;
    FFTPlan pz;
    int y, x0, nl;
    double2 *wa, *wb, *tw;
    double* phys;  // [NP][XB][Nz]
    int XB;
};

__device__ __forceinline__ double* physf(const ZCtx& c, int f) { return c.phys + (long)f * c.XB * c.g.Nz; }

// c2r of two real fields at once: field fa -> phys[da], fb -> phys[db]
// (fb < 0: none). dza/dzb apply d/dz. Imag parts of kz = 0 are ignored, as
// FFTW's c2r does. The unused middle bins are zeroed in the same sweep.
template <int NZ>
__device__ void zc2r_pair(const ZCtx& c, const double2* __restrict__ xp, int fa, bool dza, int da, int fb, bool dzb,
                          int db) {
    const Geom& g = c.g;
    const int Nz = g.Nz, nkz = g.nkz;
    const int nmid = Nz - 2 * nkz + 1;  // bins nkz .. Nz-nkz
    const int P = lpitch(Nz);
    for (int w = threadIdx.x; w < c.nl * nmid; w += blockDim.x) {
        const int l = w / nmid, j = w - l * nmid;
        c.wa[l * P + pidx(nkz + j)] = make_double2(0.0, 0.0);
    }
    const long fsz = (long)g.Ny * g.Nx * nkz;
    const double dk = 2 * PI / g.Lz;
    for (int w = threadIdx.x; w < c.nl * nkz; w += blockDim.x) {
        const int l = w / nkz, k = w - l * nkz;
        const long base = ((long)c.y * g.Nx + c.x0 + l) * nkz + k;
        double2 A = xp[(long)fa * fsz + base];
        if (dza) A = imul(dk * k, A);
        double2 B = make_double2(0.0, 0.0);
        if (fb >= 0) {
            B = xp[(long)fb * fsz + base];
            if (dzb) B = imul(dk * k, B);
        }
        double2* z = c.wa + l * P;
        if (k == 0) {
            z[0] = make_double2(A.x, B.x);
        } else {
            z[pidx(k)] = make_double2(A.x - B.y, A.y + B.x);       // A + iB
            z[pidx(Nz - k)] = make_double2(A.x + B.y, B.x - A.y);  // conj(A) + i conj(B)
        }
    }
    __syncthreads();
    double2* r = fft_any<NZ, +1, true>(c.wa, c.wb, c.pz, c.tw, c.nl);
    double* pa = physf(c, da);
    double* pb = db >= 0 ? physf(c, db) : nullptr;
    for (int w = threadIdx.x; w < c.nl * Nz; w += blockDim.x) {
        const int l = w / Nz, zz = w - l * Nz;
        const double2 v = r[l * P + pidx(zz)];
        pa[w] = v.x;
        if (pb) pb[w] = v.y;
    }
    __syncthreads();
}

// r2c of phys[sa] (and phys[sb]) -> zo fields ga, gb (kz <= kzd kept).
// fold != 0 (with sb >= 0): field ga receives A + fold i kz B instead of A,
// kz = 2 pi k / Lz, A and B the spectra of phys[sa] and phys[sb]; gb < 0 then
// drops B.
template <int NZ>
__device__ void zr2c_pair(const ZCtx& c, double2* __restrict__ zo, int sa, int ga, int sb, int gb,
                          double fold = 0.0) {
    const Geom& g = c.g;
    const int Nz = g.Nz, nkz = g.nkz;
    const double* pa = physf(c, sa);
    const double* pb = sb >= 0 ? physf(c, sb) : nullptr;
    const int P = lpitch(Nz);
    for (int w = threadIdx.x; w < c.nl * Nz; w += blockDim.x) {
        const int l = w / Nz, zz = w - l * Nz;
        c.wa[l * P + pidx(zz)] = make_double2(pa[w], pb ? pb[w] : 0.0);
    }
    __syncthreads();
    double2* r = fft_any<NZ, -1, true>(c.wa, c.wb, c.pz, c.tw, c.nl);
    const long fsz = (long)g.Ny * g.Nx * nkz;
    for (int w = threadIdx.x; w < c.nl * nkz; w += blockDim.x) {
        const int l = w / nkz, k = w - l * nkz;
        const double2 Zk = r[l * P + pidx(k)];
        const double2 Zn = r[l * P + pidx((Nz - k) % Nz)];
        const long base = ((long)c.y * g.Nx + c.x0 + l) * nkz + k;
        const double2 A = make_double2(0.5 * (Zk.x + Zn.x), 0.5 * (Zk.y - Zn.y));
        const double2 B = make_double2(0.5 * (Zk.y + Zn.y), -0.5 * (Zk.x - Zn.x));
        if (fold != 0.0 && pb) {
            const double fk = fold * ((2 * PI / g.Lz) * k);
            zo[(long)ga * fsz + base] = make_double2(A.x - fk * B.y, A.y + fk * B.x);
        } else {
            zo[(long)ga * fsz + base] = A;
        }
        if (gb >= 0) zo[(long)gb * fsz + base] = B;
    }
    __syncthreads();
}

// physical-space products. xp fields: ROT u v w wx wy wz; CONV/SKEW u v w
// du/dy dv/dy dw/dy du/dx dv/dx dw/dx; DIV u v w. zo outputs: g0..g2 (the
// u.grad u / omega x u part and the rotation term) then uu00 uu01 uu02 uu11
// uu12 uu22 for DIV; for SKEW g_i + i kz u_i u_2 / 2 then uu00 uu01 uu02 uu11
// uu12 (8 fields).
template <int METHOD, int NZ>
__global__ void __launch_bounds__(256) k_zpass(Geom g, FFTPlan pz, int XB, const NLMember* __restrict__ tab,
                                               int want_g, const double2* __restrict__ xp0, double2* __restrict__ zo0,
                                               long sx) {
    extern __shared__ double2 lds[];
    const double rotation = tab[blockIdx.y].rotation;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
    double2* __restrict__ zo = zo0 + blockIdx.y * sx;
    const int nxc = (g.Nx + XB - 1) / XB;
    ZCtx c;
    c.g = g;
    c.pz = pz;
    c.y = blockIdx.x / nxc;
    c.x0 = (blockIdx.x % nxc) * XB;
    c.nl = min(XB, g.Nx - c.x0);
    c.XB = XB;
    c.tw = lds;
    c.wa = lds + g.Nz;
    c.wb = c.wa + XB * lpitch(g.Nz);
    c.phys = reinterpret_cast<double*>(c.wb + XB * lpitch(g.Nz));
    stage_tw(c.tw, pz);
    const int Nz = g.Nz;
    const int npts = c.nl * Nz;
    if (METHOD == NL_ROT) {
        zc2r_pair<NZ>(c, xp, 0, false, 0, 1, false, 1);
        zc2r_pair<NZ>(c, xp, 2, false, 2, 3, false, 3);
        zc2r_pair<NZ>(c, xp, 4, false, 4, 5, false, 5);
        double *u0 = physf(c, 0), *u1 = physf(c, 1), *u2 = physf(c, 2);
        double *w0 = physf(c, 3), *w1 = physf(c, 4), *w2 = physf(c, 5);
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {  // cross(vort, u) (diffops.cpp:2598-2605)
            const double a0 = u0[w], a1 = u1[w], a2 = u2[w], b0 = w0[w], b1 = w1[w], b2 = w2[w];
            double f0 = b1 * a2 - b2 * a1;
            double f1 = b2 * a0 - b0 * a2;
            const double f2 = b0 * a1 - b1 * a0;
            if (rotation != 0.0) {  // nse.cpp:61-80
                f0 -= rotation * a1;
                f1 += rotation * a0;
            }
            w0[w] = f0;
            w1[w] = f1;
            w2[w] = f2;
        }
        __syncthreads();
        zr2c_pair<NZ>(c, zo, 3, 0, 4, 1);
        zr2c_pair<NZ>(c, zo, 5, 2, -1, -1);
        return;
    }
    double *u0 = physf(c, 0), *u1 = physf(c, 1), *u2 = physf(c, 2);
    double *pa = physf(c, 3), *pb = physf(c, 4);
    if constexpr (METHOD == NL_CONV || METHOD == NL_SKEW) {
        // f_i = sum_j (s u_j) du_i/dx_j with the terms of each f_i added in the
        // order j = x, y, z (diffops.cpp:3192-3199, 3626-3633). Component by
        // component through phys 3, 4 (inputs) and 5, 6 (f); the inputs are
        // paired so that every two-for-one c2r is full.
        constexpr bool SK = (METHOD == NL_SKEW);
        const double s = SK ? 0.5 : 1.0;
        double *fa = physf(c, 5), *fb = physf(c, 6);
        auto su = [&](const double* uj, int w) { return SK ? s * uj[w] : uj[w]; };
        zc2r_pair<NZ>(c, xp, 0, false, 0, 1, false, 1);  // u, v
        zc2r_pair<NZ>(c, xp, 2, false, 2, 6, false, 3);  // w, du/dx
        for (int w = threadIdx.x; w < npts; w += blockDim.x) fa[w] = 0.0 + su(u0, w) * pa[w];
        zc2r_pair<NZ>(c, xp, 3, false, 3, 0, true, 4);   // du/dy, du/dz
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] += su(u1, w) * pa[w];
            fa[w] += su(u2, w) * pb[w];
            if (rotation != 0.0) fa[w] -= rotation * u1[w];  // nse.cpp:61-80
            if (SK) pb[w] = u0[w] * u2[w];
        }
        __syncthreads();
        // skew-symmetric: f0 + i kz u0u2 / 2 and u0u2 (the layout of k_zwave)
        zr2c_pair<NZ>(c, zo, 5, 0, SK ? 4 : -1, SK ? 5 : -1, SK ? 0.5 : 0.0);
        zc2r_pair<NZ>(c, xp, 7, false, 3, 4, false, 4);  // dv/dx, dv/dy
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] = 0.0 + su(u0, w) * pa[w];
            fa[w] += su(u1, w) * pb[w];
        }
        zc2r_pair<NZ>(c, xp, 1, true, 3, 8, false, 4);   // dv/dz, dw/dx
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] += su(u2, w) * pa[w];
            if (rotation != 0.0) fa[w] += rotation * u0[w];
            fb[w] = 0.0 + su(u0, w) * pb[w];
        }
        zc2r_pair<NZ>(c, xp, 5, false, 3, 2, true, 4);   // dw/dy, dw/dz
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fb[w] += su(u1, w) * pa[w];
            fb[w] += su(u2, w) * pb[w];
        }
        __syncthreads();
        if (SK) {
            // f1 + i kz u1u2 / 2 and u1u2, f2 + i kz u2u2 / 2, then the rest of
            // outer(u, u) (diffops.cpp:2336-2388): u0u0, u0u1, u1u1
            for (int w = threadIdx.x; w < npts; w += blockDim.x) {
                pa[w] = u1[w] * u2[w];
                pb[w] = u2[w] * u2[w];
            }
            __syncthreads();
            zr2c_pair<NZ>(c, zo, 5, 1, 3, 7, 0.5);
            zr2c_pair<NZ>(c, zo, 6, 2, 4, -1, 0.5);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) {
                pa[w] = u0[w] * u0[w];
                pb[w] = u0[w] * u1[w];
            }
            __syncthreads();
            zr2c_pair<NZ>(c, zo, 3, 3, 4, 4);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) pa[w] = u1[w] * u1[w];
            __syncthreads();
            zr2c_pair<NZ>(c, zo, 3, 6, -1, -1);
        } else {
            zr2c_pair<NZ>(c, zo, 5, 1, 6, 2);  // f1, f2
        }
    } else {
        zc2r_pair<NZ>(c, xp, 0, false, 0, 1, false, 1);
        zc2r_pair<NZ>(c, xp, 2, false, 2, -1, false, -1);
        if (want_g) {  // DIV with rotation: g = rotation terms only
            for (int w = threadIdx.x; w < npts; w += blockDim.x) {
                pa[w] = -(rotation * u1[w]);
                pb[w] = rotation * u0[w];
            }
            __syncthreads();
            zr2c_pair<NZ>(c, zo, 3, 0, 4, 1);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) pa[w] = 0.0;
            __syncthreads();
            zr2c_pair<NZ>(c, zo, 3, 2, -1, -1);
        }
        // outer(u, u) (diffops.cpp:2336-2388), two entries per r2c
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u0[w] * u0[w];
            pb[w] = u0[w] * u1[w];
        }
        __syncthreads();
        zr2c_pair<NZ>(c, zo, 3, 3, 4, 4);
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u0[w] * u2[w];
            pb[w] = u1[w] * u1[w];
        }
        __syncthreads();
        zr2c_pair<NZ>(c, zo, 3, 5, 4, 6);
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u1[w] * u2[w];
            pb[w] = u2[w] * u2[w];
        }
        __syncthreads();
        zr2c_pair<NZ>(c, zo, 3, 7, 4, 8);
    }
}

// ---- wave-local z pass -------------------------------------------------------
// One line's view: its lane in the group, where its data sit, its LDS rows.
struct ZWCtx {
    int gi;            // lane within the line's group
    bool line_ok;      // the line exists (x < Nx)
    long base, fsz;    // line offset and field size in the [field][y][x][kz] arrays
    int nkz;
    double dk;         // 2 pi / Lz
    double2* T;        // the line's LDS rows
    const double2* tw; // exp(-2 pi i m / N), m < N, in LDS
    // input staging: the wavefront's lines are one contiguous run of the
    // [field][y][x][kz] arrays (wcount values from wbase); two fields of it sit
    // in LDS (slots 0 and 1 from S, slot stride sstride), this line's bins at
    // L * nkz within a slot
    long wbase;
    int wcount, lane, sline, sstride;
    double2* S;
};

// Starts the copy of field f of the wavefront's lines into staging slot
// `slot` (global_load_lds_dwordx4: lane i of a copy instruction moves 16 bytes
// to its base + 16 i; lanes past the run copy nothing). The data are in LDS
// once the wavefront's vector-memory count has drained; the compiler waits for
// it before the first LDS read of the staging array.
__device__ __forceinline__ void zw_stage(const ZWCtx& c, const double2* __restrict__ xp, int f, int slot) {
    const __attribute__((address_space(1))) double2* src = gmem(xp) + (long)f * c.fsz + c.wbase;
    double2* dst = c.S + slot * c.sstride;
    for (int t = 0; t < c.wcount; t += 64) {
        if (t + c.lane < c.wcount)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + t + c.lane),
                                             (__attribute__((address_space(3))) void*)(dst + t), 16, 0, 0);
    }
}

// c2r of two real fields at once (fa -> pa, fb -> pb; fb < 0: none), from the
// live bins kz < nkz of xp; dza / dzb apply d/dz. As in FFTW's c2r, the
// imaginary part of bin 0 is ignored. STAGED: the bins come from staging
// slots 0 (fa) and 1 (fb), and once these are read the copies of fields na and
// nb (< 0: none) into them start, to land while this transform and what
// follows it run.
template <class S, bool STAGED>
__device__ __forceinline__ void zw_c2r(const ZWCtx& c, const double2* __restrict__ xp, int fa, bool dza, int fb,
                                       bool dzb, double (&pa)[S::PV], double (&pb)[S::PV], int na = -1,
                                       int nb = -1) {
    constexpr int SL = S::SL, SV = S::SV, PV = S::PV, N = S::N;
    const int j = c.gi;
    const bool act = c.line_ok && j < SL;
    const double2* Sa = c.S + c.sline;
    const double2* Sb = Sa + c.sstride;
    double2 v[SV];
#pragma unroll
    for (int r = 0; r < SV; ++r) {
        const int n = j + SL * r;
        const bool lo = n < c.nkz, hi = n > N - c.nkz;
        const int k = lo ? n : N - n;
        double2 A = make_double2(0.0, 0.0), B = make_double2(0.0, 0.0);
        if (act && (lo || hi)) {
            if constexpr (STAGED) {
                A = Sa[k];
                if (fb >= 0) B = Sb[k];
            } else {
                A = xp[(long)fa * c.fsz + c.base + k];
                if (fb >= 0) B = xp[(long)fb * c.fsz + c.base + k];
            }
        }
        if (dza) A = imul(c.dk * k, A);
        if (dzb) B = imul(c.dk * k, B);
        if (n == 0) v[r] = make_double2(A.x, B.x);
        else if (lo) v[r] = make_double2(A.x - B.y, A.y + B.x);  // A + iB
        else v[r] = make_double2(A.x + B.y, B.x - A.y);          // conj(A) + i conj(B) (zero in the gap)
    }
    if (STAGED && na >= 0) {
        // every lane's reads of the slots have returned before the copies may overwrite them
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        zw_stage(c, xp, na, 0);
        if (nb >= 0) zw_stage(c, xp, nb, 1);
    }
    double2 u[PV];
    line_s2p<S, +1>(v, u, j, c.T, c.tw);
#pragma unroll
    for (int m = 0; m < PV; ++m) {
        pa[m] = u[m].x;
        pb[m] = u[m].y;
    }
}

// r2c of pa (and pb when TWO) -> zo fields ga (and gb), bins kz < nkz.
// fold != 0 (with TWO): field ga receives A + fold i kz B instead of A, with
// kz = 2 pi k / Lz, A and B the spectra of pa and pb; gb < 0 then drops B.
template <class S, bool TWO>
__device__ __forceinline__ void zw_r2c(const ZWCtx& c, double2* __restrict__ zo, const double (&pa)[S::PV],
                                       const double (&pb)[S::PV], int ga, int gb, double fold = 0.0) {
    constexpr int SL = S::SL, SV = S::SV, PV = S::PV, N = S::N;
    const int j = c.gi;
    double2 v[PV];
#pragma unroll
    for (int m = 0; m < PV; ++m) v[m] = make_double2(pa[m], TWO ? pb[m] : 0.0);
    double2 w[SV];
    line_p2s<S, -1>(v, w, j, c.T, c.tw);  // w[p] = X[j + SL p]
    wave_lds_sync();
    if (j < SL) {
#pragma unroll
        for (int p = 0; p < SV; ++p) c.T[j + SL * p] = w[p];
    }
    wave_lds_sync();
    if (c.line_ok && j < SL) {
#pragma unroll
        for (int p = 0; p < SV; ++p) {
            const int k = j + SL * p;
            if (k < c.nkz) {
                const double2 Zk = w[p];
                const double2 Zn = c.T[(N - k) % N];
                const double2 A = make_double2(0.5 * (Zk.x + Zn.x), 0.5 * (Zk.y - Zn.y));
                const double2 B = make_double2(0.5 * (Zk.y + Zn.y), -0.5 * (Zk.x - Zn.x));
                if (TWO && fold != 0.0) {
                    const double fk = fold * (c.dk * k);
                    zo[(long)ga * c.fsz + c.base + k] = make_double2(A.x - fk * B.y, A.y + fk * B.x);
                } else {
                    zo[(long)ga * c.fsz + c.base + k] = A;
                }
                if (TWO && gb >= 0) zo[(long)gb * c.fsz + c.base + k] = B;
            }
        }
    }
}

// The z pass stages its inputs at Nz = 64. The choice depends on the grid alone
// (never on the member count), so a member's result is the same alone and in a
// batch: the two forms contract multiply-adds differently (the compiler fuses
// either product of a*b + c*d depending on the code around it) and differ in the
// last bits. At Nz = 64 the staged form wins where it matters, in batches (16
// members of 64x65x64, skew-symmetric: 104 against 122 us per launch) and loses
// 2.6 us on a lone field; at 32 and 48 (24 members) and at the three-step
// lengths (one 128^3 field: rotational 39.2 us staged, 35.0 not, convection 73.2
// and 70.1) the unstaged one is faster.
constexpr bool zwave_staged(int nz) { return nz == 64; }

// Three steps per transform (ZW3) at Nz = 72 and from 96 on. What bounds the z
// pass there is how few wavefronts a SIMD holds: with 6 physical values per lane
// instead of 8 to 16 and transforms of at most 9 values, 2 or 3 of them fit the
// registers where 1 did (skew-symmetric 96: 341 -> 162 registers, rotational
// 192: 297 -> 131), at the price of a second transpose through LDS. us per
// launch, two steps -> three: one 96^3 skew-symmetric field 59 -> 44, 128^3
// convection 92 -> 70, rotational 49 -> 35, 192x129x192 rotational 95 -> 76,
// 256x33x256 52 -> 48, 64x49x162 skew-symmetric 61 -> 32, 8 members of 32x49x72
// 72 -> 53. At 48 and 64, where 2 wavefronts fit anyway, the second transpose
// costs more than it gives in a batch (16 of 64^3 113 -> 127, 24 of 48^3 82 -> 88).
constexpr bool zwave_three(int nz) { return nz == 72 || nz >= 96; }
template <int NZ>
using ZLine = std::conditional_t<zwave_three(NZ), ZW3<NZ>, ZW<NZ>>;

// lengths the staged form is compiled for
constexpr bool zwave_has_staged(int nz) { return nz == 16 || nz == 32 || nz == 48 || nz == 64; }
// The z pass of k_zpass with one wavefront per 64/G lines (same fields, same
// products in the same order). A block is independent wavefronts: any number
// up to 4 (LDS sized at launch), or, STAGED, ZWAVE_WB of them, each staging
// the next transform's two input fields in LDS while it works on the current
// one. Staging hides the loads' latency where many wavefronts share a CU;
// with few wavefronts per SIMD the extra LDS round trip costs more than it
// hides (zwave_staged picks the form per grid).
template <int METHOD, int NZ, bool STAGED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 8)))
k_zwave(Geom g, const double2* __restrict__ twg, const NLMember* __restrict__ tab,
                                               int want_g, const double2* __restrict__ xp0, double2* __restrict__ zo0,
                                               long sx) {
    using S = ZLine<NZ>;
    constexpr int N1 = S::PV, SLOT = S::LPW * (NZ / 2);
    double2 *tw_l, *T_l, *in_l = nullptr;
    if constexpr (STAGED) {
        // Separate LDS arrays (not one dynamic block) let the compiler tell the
        // staging copies apart from the transposes: an LDS read waits for the
        // copies in flight only when it reads the staging array.
        __shared__ double2 tw_s[NZ];
        __shared__ double2 T_s[ZWAVE_WB * S::LPW * S::LBUF];
        __shared__ double2 in_s[ZWAVE_WB * 2 * SLOT];
        tw_l = tw_s;
        T_l = T_s;
        in_l = in_s;
    } else {
        extern __shared__ double2 lds[];
        tw_l = lds;
        T_l = lds + NZ;
    }
    for (int i = threadIdx.x; i < NZ; i += blockDim.x) tw_l[i] = twg[i];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int nxc = (g.Nx + S::LPW - 1) / S::LPW;
    const int wg = blockIdx.x * (blockDim.x / 64) + wave;
    const int y = wg / nxc;
    if (y >= g.Ny) return;
    const int L = lane / S::G;
    const int x0 = (wg - y * nxc) * S::LPW, x = x0 + L;
    ZWCtx c;
    c.gi = lane % S::G;
    c.line_ok = x < g.Nx;
    c.base = ((long)y * g.Nx + (c.line_ok ? x : 0)) * g.nkz;
    c.fsz = (long)g.Ny * g.Nx * g.nkz;
    c.nkz = g.nkz;
    c.dk = 2 * PI / g.Lz;
    c.T = T_l + (wave * S::LPW + L) * S::LBUF;
    c.tw = tw_l;
    c.wbase = ((long)y * g.Nx + x0) * g.nkz;
    c.wcount = min(S::LPW, g.Nx - x0) * g.nkz;
    c.lane = lane;
    c.sline = L * g.nkz;
    c.sstride = SLOT;
    c.S = in_l + wave * 2 * SLOT;
    const double rotation = tab[blockIdx.y].rotation;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
    double2* __restrict__ zo = zo0 + blockIdx.y * sx;
    if constexpr (STAGED) {
        zw_stage(c, xp, 0, 0);  // u, v: the first transform's pair
        zw_stage(c, xp, 1, 1);
    }
    if constexpr (METHOD == NL_ROT) {
        double u0[N1], u1[N1], u2[N1], w0[N1], w1[N1], w2[N1];
        zw_c2r<S, STAGED>(c, xp, 0, false, 1, false, u0, u1, 2, 3);
        zw_c2r<S, STAGED>(c, xp, 2, false, 3, false, u2, w0, 4, 5);
        zw_c2r<S, STAGED>(c, xp, 4, false, 5, false, w1, w2);
        double f0[N1], f1[N1], f2[N1];
#pragma unroll
        for (int m = 0; m < N1; ++m) {  // cross(vort, u) (diffops.cpp:2598-2605)
            const double a0 = u0[m], a1 = u1[m], a2 = u2[m], b0 = w0[m], b1 = w1[m], b2 = w2[m];
            f0[m] = b1 * a2 - b2 * a1;
            f1[m] = b2 * a0 - b0 * a2;
            f2[m] = b0 * a1 - b1 * a0;
            if (rotation != 0.0) {  // nse.cpp:61-80
                f0[m] -= rotation * a1;
                f1[m] += rotation * a0;
            }
        }
        zw_r2c<S, true>(c, zo, f0, f1, 0, 1);
        zw_r2c<S, false>(c, zo, f2, f2, 2, -1);
    } else if constexpr (METHOD == NL_CONV || METHOD == NL_SKEW) {
        // f_i = sum_j (s u_j) du_i/dx_j, terms added in the order j = x, y, z
        // (diffops.cpp:3192-3199, 3626-3633). The skew-symmetric form keeps
        // h = u/2 only: halving is exact, so s u_j is h_j, u_j is 2 h_j and
        // u_i u_j is 4 (h_i h_j), all with the bits of the unscaled products.
        //
        // Skew-symmetric outputs: the z-derivative part of div(u u)/2
        // (diffops.cpp:3254-3279) is added here, in z-spectral space:
        // field i = f_i + 1/2 i kz (u_i u_z) (i = 0, 1, 2), then u_0u_0, u_0u_1,
        // u_0u_2, u_1u_1, u_1u_2 in fields 3-7; u_2u_2 is needed only for that
        // z-derivative and never leaves. The forward transforms add the x and y
        // parts of the divergence.
        constexpr bool SK = (METHOD == NL_SKEW);
        constexpr double s = SK ? 0.5 : 1.0, us = SK ? 2.0 : 1.0;
        double h0[N1], h1[N1], h2[N1], pa[N1], pb[N1], fa[N1], fb[N1];
        zw_c2r<S, STAGED>(c, xp, 0, false, 1, false, h0, h1, 2, 6);   // u, v
        zw_c2r<S, STAGED>(c, xp, 2, false, 6, false, h2, pa, 3, 0);   // w, du/dx
        if constexpr (SK) {
#pragma unroll
            for (int m = 0; m < N1; ++m) {
                h0[m] *= s;
                h1[m] *= s;
                h2[m] *= s;
            }
        }
#pragma unroll
        for (int m = 0; m < N1; ++m) fa[m] = 0.0 + h0[m] * pa[m];
        zw_c2r<S, STAGED>(c, xp, 3, false, 0, true, pa, pb, 7, 4);    // du/dy, du/dz
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            fa[m] += h1[m] * pa[m];
            fa[m] += h2[m] * pb[m];
            if (rotation != 0.0) fa[m] -= rotation * (us * h1[m]);  // nse.cpp:61-80
            if (SK) pb[m] = 4.0 * (h0[m] * h2[m]);
        }
        if constexpr (SK) zw_r2c<S, true>(c, zo, fa, pb, 0, 5, 0.5);  // f0 + i kz u0u2 / 2, and u0u2
        else zw_r2c<S, false>(c, zo, fa, pb, 0, -1);                  // f0
        zw_c2r<S, STAGED>(c, xp, 7, false, 4, false, pa, pb, 1, 8);   // dv/dx, dv/dy
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            fa[m] = 0.0 + h0[m] * pa[m];
            fa[m] += h1[m] * pb[m];
        }
        zw_c2r<S, STAGED>(c, xp, 1, true, 8, false, pa, pb, 5, 2);    // dv/dz, dw/dx
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            fa[m] += h2[m] * pa[m];
            if (rotation != 0.0) fa[m] += rotation * (us * h0[m]);
            fb[m] = 0.0 + h0[m] * pb[m];
        }
        zw_c2r<S, STAGED>(c, xp, 5, false, 2, true, pa, pb);    // dw/dy, dw/dz
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            fb[m] += h1[m] * pa[m];
            fb[m] += h2[m] * pb[m];
        }
        if constexpr (SK) {
#pragma unroll
            for (int m = 0; m < N1; ++m) pa[m] = 4.0 * (h1[m] * h2[m]);
            zw_r2c<S, true>(c, zo, fa, pa, 1, 7, 0.5);   // f1 + i kz u1u2 / 2, and u1u2
#pragma unroll
            for (int m = 0; m < N1; ++m) pa[m] = 4.0 * (h2[m] * h2[m]);
            zw_r2c<S, true>(c, zo, fb, pa, 2, -1, 0.5);  // f2 + i kz u2u2 / 2
            // remaining entries of outer(u, u) (diffops.cpp:2336-2388)
#pragma unroll
            for (int m = 0; m < N1; ++m) {
                pa[m] = 4.0 * (h0[m] * h0[m]);
                pb[m] = 4.0 * (h0[m] * h1[m]);
            }
            zw_r2c<S, true>(c, zo, pa, pb, 3, 4);
#pragma unroll
            for (int m = 0; m < N1; ++m) pa[m] = 4.0 * (h1[m] * h1[m]);
            zw_r2c<S, false>(c, zo, pa, pa, 6, -1);
        } else {
            zw_r2c<S, true>(c, zo, fa, fb, 1, 2);            // f1, f2
        }
    } else {
        double u0[N1], u1[N1], u2[N1], pa[N1], pb[N1];
        zw_c2r<S, STAGED>(c, xp, 0, false, 1, false, u0, u1, 2);
        zw_c2r<S, STAGED>(c, xp, 2, false, -1, false, u2, pa);
        if (want_g) {  // DIV with rotation: g = rotation terms only
#pragma unroll
            for (int m = 0; m < N1; ++m) {
                pa[m] = -(rotation * u1[m]);
                pb[m] = rotation * u0[m];
            }
            zw_r2c<S, true>(c, zo, pa, pb, 0, 1);
#pragma unroll
            for (int m = 0; m < N1; ++m) pa[m] = 0.0;
            zw_r2c<S, false>(c, zo, pa, pa, 2, -1);
        }
        // outer(u, u) (diffops.cpp:2336-2388), two entries per r2c
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            pa[m] = u0[m] * u0[m];
            pb[m] = u0[m] * u1[m];
        }
        zw_r2c<S, true>(c, zo, pa, pb, 3, 4);
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            pa[m] = u0[m] * u2[m];
            pb[m] = u1[m] * u1[m];
        }
        zw_r2c<S, true>(c, zo, pa, pb, 5, 6);
#pragma unroll
        for (int m = 0; m < N1; ++m) {
            pa[m] = u1[m] * u2[m];
            pb[m] = u2[m] * u2[m];
        }
        zw_r2c<S, true>(c, zo, pa, pb, 7, 8);
    }
}

int zpass_xb(const Geom& g, int nphys, const NLTune& tn);

template <int METHOD, int NZ>
void launch_z_t(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, int want_g, const double2* xp,
                       double2* zo, long sx, const NLTune& tn, hipStream_t st) {
    if constexpr (zwave_size(NZ)) {
        using S = ZLine<NZ>;
        const long waves = (long)g.Ny * ((g.Nx + S::LPW - 1) / S::LPW);
        if constexpr (zwave_has_staged(NZ)) {
            if (tn.zstage < 0 ? zwave_staged(NZ) : tn.zstage != 0) {
                if (g.nkz > NZ / 2) throw std::runtime_error("z pass: more live kz bins than Nz/2");
                const dim3 grid((unsigned)((waves + ZWAVE_WB - 1) / ZWAVE_WB), n);
                k_zwave<METHOD, NZ, true><<<grid, 64 * ZWAVE_WB, 0, st>>>(g, pz.tw, tab, want_g, xp, zo, sx);
                return;
            }
        }
        const int wb = tn.zwb > 0 ? tn.zwb : 4;
        const size_t lds = (size_t)(NZ + wb * S::LPW * S::LBUF) * sizeof(double2);
        const dim3 grid((unsigned)((waves + wb - 1) / wb), n);
        allow_lds(k_zwave<METHOD, NZ, false>, lds);
        k_zwave<METHOD, NZ, false><<<grid, 64 * wb, lds, st>>>(g, pz.tw, tab, want_g, xp, zo, sx);
    } else {
        const int nphys = zpass_nphys(METHOD);
        const int XB = zpass_xb(g, nphys, tn);
        const size_t lds = (size_t)g.Nz * sizeof(double2) +
                           (size_t)XB * (2 * lpitch(g.Nz) * sizeof(double2) + (size_t)g.Nz * nphys * sizeof(double));
        const dim3 grid(g.Ny * ((g.Nx + XB - 1) / XB), n);
        allow_lds(k_zpass<METHOD, NZ>, lds);
        k_zpass<METHOD, NZ><<<grid, 256, lds, st>>>(g, pz, XB, tab, want_g, xp, zo, sx);
    }
}

template <int METHOD>
void launch_z(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, int want_g, const double2* xp,
                     double2* zo, long sx, const NLTune& tn, hipStream_t st) {
    switch (g.Nz) {
#define CASE_Z(N) \
    case N: launch_z_t<METHOD, N>(g, pz, n, tab, want_g, xp, zo, sx, tn, st); return;
        CFG_FFT_SIZES(CASE_Z)
#undef CASE_Z
        default: launch_z_t<METHOD, 0>(g, pz, n, tab, want_g, xp, zo, sx, tn, st);
    }
}

}  // namespace cfg
