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
__device__ inline void zc2r_pair(const ZCtx& c, const double2* __restrict__ xp, int fa, bool dza, int da, int fb, bool dzb,
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
    double2* r = fft_lds<+1>(c.wa, c.wb, c.pz, c.tw, c.nl);
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
__device__ inline void zr2c_pair(const ZCtx& c, double2* __restrict__ zo, int sa, int ga, int sb, int gb,
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
    double2* r = fft_lds<-1>(c.wa, c.wb, c.pz, c.tw, c.nl);
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
template <int METHOD>
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
        zc2r_pair(c, xp, 0, false, 0, 1, false, 1);
        zc2r_pair(c, xp, 2, false, 2, 3, false, 3);
        zc2r_pair(c, xp, 4, false, 4, 5, false, 5);
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
        zr2c_pair(c, zo, 3, 0, 4, 1);
        zr2c_pair(c, zo, 5, 2, -1, -1);
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
        zc2r_pair(c, xp, 0, false, 0, 1, false, 1);  // u, v
        zc2r_pair(c, xp, 2, false, 2, 6, false, 3);  // w, du/dx
        for (int w = threadIdx.x; w < npts; w += blockDim.x) fa[w] = 0.0 + su(u0, w) * pa[w];
        zc2r_pair(c, xp, 3, false, 3, 0, true, 4);   // du/dy, du/dz
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] += su(u1, w) * pa[w];
            fa[w] += su(u2, w) * pb[w];
            if (rotation != 0.0) fa[w] -= rotation * u1[w];  // nse.cpp:61-80
            if (SK) pb[w] = u0[w] * u2[w];
        }
        __syncthreads();
        // skew-symmetric: f0 + i kz u0u2 / 2 and u0u2 (the layout of k_zsplit)
        zr2c_pair(c, zo, 5, 0, SK ? 4 : -1, SK ? 5 : -1, SK ? 0.5 : 0.0);
        zc2r_pair(c, xp, 7, false, 3, 4, false, 4);  // dv/dx, dv/dy
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] = 0.0 + su(u0, w) * pa[w];
            fa[w] += su(u1, w) * pb[w];
        }
        zc2r_pair(c, xp, 1, true, 3, 8, false, 4);   // dv/dz, dw/dx
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            fa[w] += su(u2, w) * pa[w];
            if (rotation != 0.0) fa[w] += rotation * u0[w];
            fb[w] = 0.0 + su(u0, w) * pb[w];
        }
        zc2r_pair(c, xp, 5, false, 3, 2, true, 4);   // dw/dy, dw/dz
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
            zr2c_pair(c, zo, 5, 1, 3, 7, 0.5);
            zr2c_pair(c, zo, 6, 2, 4, -1, 0.5);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) {
                pa[w] = u0[w] * u0[w];
                pb[w] = u0[w] * u1[w];
            }
            __syncthreads();
            zr2c_pair(c, zo, 3, 3, 4, 4);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) pa[w] = u1[w] * u1[w];
            __syncthreads();
            zr2c_pair(c, zo, 3, 6, -1, -1);
        } else {
            zr2c_pair(c, zo, 5, 1, 6, 2);  // f1, f2
        }
    } else {
        zc2r_pair(c, xp, 0, false, 0, 1, false, 1);
        zc2r_pair(c, xp, 2, false, 2, -1, false, -1);
        if (want_g) {  // DIV with rotation: g = rotation terms only
            for (int w = threadIdx.x; w < npts; w += blockDim.x) {
                pa[w] = -(rotation * u1[w]);
                pb[w] = rotation * u0[w];
            }
            __syncthreads();
            zr2c_pair(c, zo, 3, 0, 4, 1);
            for (int w = threadIdx.x; w < npts; w += blockDim.x) pa[w] = 0.0;
            __syncthreads();
            zr2c_pair(c, zo, 3, 2, -1, -1);
        }
        // outer(u, u) (diffops.cpp:2336-2388), two entries per r2c
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u0[w] * u0[w];
            pb[w] = u0[w] * u1[w];
        }
        __syncthreads();
        zr2c_pair(c, zo, 3, 3, 4, 4);
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u0[w] * u2[w];
            pb[w] = u1[w] * u1[w];
        }
        __syncthreads();
        zr2c_pair(c, zo, 3, 5, 4, 6);
        for (int w = threadIdx.x; w < npts; w += blockDim.x) {
            pa[w] = u1[w] * u2[w];
            pb[w] = u2[w] * u2[w];
        }
        __syncthreads();
        zr2c_pair(c, zo, 3, 7, 4, 8);
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
};

// A lane's live bins: those of the lower half (s + SL r with SL r < lo) and the
// mirrored ones (SL - s + SL q with SL q < hi), and the byte offsets of bins s and
// SL - s of its line within a field.
struct Bins {
    int lo, hi;
    unsigned at, at_hi;
};
template <class S>
__device__ __forceinline__ Bins zw_bins(const ZWCtx& c) {
    const bool act = c.line_ok && c.gi < S::SL;
    return Bins{act ? c.nkz - c.gi : 0, act ? c.nkz - S::SL + c.gi : 0, (unsigned)(c.base + c.gi) * 16u,
                (unsigned)(c.base + (S::SL - c.gi)) * 16u};
}

// c2r of two real fields at once (fa -> pa, fb -> pb; fb < 0: none), from the
// live bins kz < nkz of xp. DZ: pb is d/dz of field fa, from the same loads. SB: pb
// passes through the transform at 1/SB of its size, a power of two and so exact: both
// halves of a transform share its rounding, and a derivative is some times larger
// than its field (with u_c and du_c/dz, du_c/dx and du_c/dy paired at full size the
// convection form's w was off by 8.2e-16 of its norm, at 1/8 by 4.7e-16, as with
// every field paired as loaded). The scale enters as the multiplier of an fma: as a
// product of the loaded value the compiler moves it under the load's condition, where
// every load gets a wait of its own (16 of 64^3 90 -> 108 us). As in FFTW's c2r, the
// imaginary part of bin 0 is ignored. issued is called once the loads are under way.
template <class S, bool DZ, int SB, class Then>
__device__ __forceinline__ void zw_c2r(const ZWCtx& c, const double2* __restrict__ xp, int fa, int fb,
                                       double (&pa)[S::PV], double (&pb)[S::PV], Then&& issued) {
    constexpr double sb = 1.0 / SB;
    constexpr int SL = S::SL, SV = S::SV, PV = S::PV;
    const int s = c.gi;
    // Value r of lane s is bin n = s + SL r. In the lower half of the r it can
    // only be a live bin k = n, in the upper half only the mirror of k = N - n =
    // SL - s + SL (SV - 1 - r) (nkz <= N/2); an odd SV has a middle r that can be
    // either. So each load is at a fixed distance from one of two lane addresses.
    const Bins bins = zw_bins<S>(c);
    double2 A[SV], B[SV];
    auto fetch = [&](int f, double2 (&X)[SV]) {
        const gbytes fld = reinterpret_cast<gbytes>(gmem(xp) + (long)f * c.fsz);
#pragma unroll
        for (int r = 0; r < SV; ++r) {
            X[r] = make_double2(0.0, 0.0);
            if (2 * r < SV && SL * r < bins.lo) X[r] = gload(fld + 16 * SL * r, bins.at);
            if (2 * r + 1 >= SV && SL * (SV - 1 - r) < bins.hi)
                X[r] = gload(fld + 16 * SL * (SV - 1 - r), bins.at_hi);
        }
    };
    fetch(fa, A);
    if (!DZ && fb >= 0) fetch(fb, B);
    issued();
    double2 v[SV];
    const double sd = s;
#pragma unroll
    for (int r = 0; r < SV; ++r) {
        const bool up = 2 * r + 1 > SV || (2 * r + 1 == SV && SL * r >= bins.lo);  // the mirror of bin k
        const double2 a = A[r];
        double2 b = !DZ && fb >= 0 ? B[r] : make_double2(0.0, 0.0);
        if (DZ) b = imul(c.dk * (up ? (double)(SL * (SV - r)) - sd : sd + (double)(SL * r)), a);
        if (up) {
            v[r] = make_double2(fma(sb, b.y, a.x), fma(sb, b.x, -a.y));  // conj(A) + i conj(B) (zero in the gap)
        } else {
            v[r] = make_double2(fma(-sb, b.y, a.x), fma(sb, b.x, a.y));  // A + iB
            if (r == 0 && s == 0) v[r] = make_double2(a.x, sb * b.x);
        }
    }
    double2 u[PV];
    line_s2p<S, +1>(v, u, s, c.T, c.tw);
#pragma unroll
    for (int m = 0; m < PV; ++m) {
        pa[m] = u[m].x;
        pb[m] = SB * u[m].y;
    }
}
template <class S>
__device__ __forceinline__ void zw_c2r(const ZWCtx& c, const double2* __restrict__ xp, int fa, int fb,
                                       double (&pa)[S::PV], double (&pb)[S::PV]) {
    zw_c2r<S, false, 1>(c, xp, fa, fb, pa, pb, [] {});
}

// r2c of pa (and pb when TWO) -> zo fields ga (and gb), bins kz < nkz.
// fold != 0 (with TWO): field ga receives A + fold i kz B instead of A, with
// kz = 2 pi k / Lz, A and B the spectra of pa and pb; gb < 0 then drops B.
template <class S, bool TWO>
__device__ __forceinline__ void zw_r2c(const ZWCtx& c, double2* __restrict__ zo, const double (&pa)[S::PV],
                                       const double (&pb)[S::PV], int ga, int gb, double fold = 0.0) {
    constexpr int SL = S::SL, SV = S::SV, PV = S::PV;
    const int s = c.gi;
    double2 v[PV];
#pragma unroll
    for (int m = 0; m < PV; ++m) v[m] = make_double2(pa[m], TWO ? pb[m] : 0.0);
    double2 w[SV];
    line_p2s<S, -1>(v, w, s, c.T, c.tw);  // w[p] = X[s + SL p]
    const Bins bins = zw_bins<S>(c);
    // the mirrors of the live bins meet them through the line's LDS rows; bin 0 is its own
    wave_lds_sync();
    if (s < SL) {
#pragma unroll
        for (int p = SV / 2; p < SV; ++p) c.T[s + SL * p] = w[p];
    }
    wave_lds_sync();
    const double sd = s;
    const gbytes_w oa = reinterpret_cast<gbytes_w>(gmem_w(zo) + (long)ga * c.fsz);
    const gbytes_w ob = reinterpret_cast<gbytes_w>(gmem_w(zo) + (long)(TWO && gb >= 0 ? gb : ga) * c.fsz);
#pragma unroll
    for (int p = 0; 2 * p < SV; ++p) {
        if (SL * p < bins.lo) {
            const double2 Zk = w[p];
            double2 Zn = c.T[SL - s + SL * (SV - 1 - p) - (p == 0 && s == 0 ? 1 : 0)];
            if (p == 0 && s == 0) Zn = Zk;
            const double2 A = make_double2(0.5 * (Zk.x + Zn.x), 0.5 * (Zk.y - Zn.y));
            const double2 B = make_double2(0.5 * (Zk.y + Zn.y), -0.5 * (Zk.x - Zn.x));
            if (TWO && fold != 0.0) {
                const double fk = fold * (c.dk * (sd + (double)(SL * p)));
                gstore(oa + 16 * SL * p, bins.at, make_double2(A.x - fk * B.y, A.y + fk * B.x));
            } else {
                gstore(oa + 16 * SL * p, bins.at, A);
            }
            if (TWO && gb >= 0) gstore(ob + 16 * SL * p, bins.at, B);
        }
    }
}

template <int NZ>
using ZLine = std::conditional_t<zwave_three(NZ), ZW3<NZ>, ZW<NZ>>;

// The z pass of k_zpass for the rotational and the divergence form, one wavefront
// per 64/G lines (same fields, same products in the same order). A block is
// independent wavefronts, any number up to 4 (LDS sized at launch). Every access is
// at a field's uniform base, one of two 32-bit lane offsets and a constant distance:
// with 64-bit addresses and the bin tests formed per access the kernel was bound by
// those instructions. us per launch, before -> after: rotational 128^3 35 -> 32,
// 192x129x192 76 -> 64 (228 MB, 3.6 TB/s). A form that staged its inputs in LDS one
// transform ahead is slower than this one at every length (16 members of 64^3
// rotational 52 against 42).
template <int METHOD, int NZ>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 8)))
k_zwave(Geom g, const double2* __restrict__ twg, const NLMember* __restrict__ tab,
                                               int want_g, const double2* __restrict__ xp0, double2* __restrict__ zo0,
                                               long sx) {
    using S = ZLine<NZ>;
    constexpr int N1 = S::PV;
    extern __shared__ double2 lds[];
    double2 *const tw_l = lds, *const T_l = lds + S::TWN;
    for (int i = threadIdx.x; i < S::TWN; i += blockDim.x) tw_l[i] = twg[S::tw_power(i)];
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
    const double rotation = tab[blockIdx.y].rotation;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
    double2* __restrict__ zo = zo0 + blockIdx.y * sx;
    if constexpr (METHOD == NL_ROT) {
        double u0[N1], u1[N1], u2[N1], w0[N1], w1[N1], w2[N1];
        zw_c2r<S>(c, xp, 0, 1, u0, u1);
        zw_c2r<S>(c, xp, 2, 3, u2, w0);
        zw_c2r<S>(c, xp, 4, 5, w1, w2);
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
    } else {
        double u0[N1], u1[N1], u2[N1], pa[N1], pb[N1];
        zw_c2r<S>(c, xp, 0, 1, u0, u1);
        zw_c2r<S>(c, xp, 2, -1, u2, pa);
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

// The z pass of 64/G lines by three wavefronts, one per velocity component (zsplit:
// where, and what it measured). Wavefront c transforms u_c and what belongs to it (its
// gradient, or the vorticity component w_c), hands the velocity (and w) to the other
// two through LDS and forms its part of the products. Each wavefront's transforms are
// a serial chain through LDS, so what bounds the pass is how many wavefronts a SIMD
// holds: 32 bins take 122 registers here against 180 in one wavefront, 64 bins 162
// against 238, 192 bins 101 against 200. The shared values lie in the wavefronts'
// line rows, which are free between the inverse and the forward transforms; in space
// of their own they cost a third of the occupancy (rotational 192x129x192 93 against
// 76 us). The first bins are requested before the twiddles are waited for. Two such
// groups of lines per block, or blocks in XCD order, are slower (16 of 64^3 100 ->
// 115, 107; the chain of barriers couples six wavefronts).
// u_c and du_c/dz come from one load of u_c: 9 fields are read, not 12 (16 of 64^3
// 95.8 -> 89.8, 24 of 48^3 65.6 -> 63.7, 24 of 32^3 22.2 -> 21.7, 128^3 convection 43.3
// -> 42.7).
// LDS of a block: the twiddles, then the line rows of the three wavefronts, which also carry the shared values
template <int METHOD, int NZ>
constexpr size_t zsplit_lds() {
    using S = ZLine<NZ>;
    const size_t rows = (size_t)3 * S::LPW * S::LBUF * sizeof(double2);
    const size_t shared = (size_t)(METHOD == NL_ROT ? 6 : 3) * S::PV * 64 * sizeof(double);
    return S::TWN * sizeof(double2) + (rows > shared ? rows : shared);
}
template <int METHOD, int NZ>
__global__ void __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(1, 8)))
k_zsplit(Geom g, const double2* __restrict__ twg, const NLMember* __restrict__ tab, int want_g,
         const double2* __restrict__ xp0, double2* __restrict__ zo0, long sx) {
    using S = ZLine<NZ>;
    constexpr int PV = S::PV;
    extern __shared__ double2 lds[];
    double2* const T_l = lds + S::TWN;
    double* const ex = reinterpret_cast<double*>(T_l);  // [shared field][value][lane]
    constexpr int NTW = (S::TWN + 191) / 192;
    dvec2 twr[NTW];
#pragma unroll
    for (int i = 0; i < NTW; ++i) twr[i] = gmem(reinterpret_cast<const dvec2*>(twg))[S::tw_power(min((int)threadIdx.x + 192 * i, S::TWN - 1))];
    auto twiddles = [&] {  // behind the first loads of bins
#pragma unroll
        for (int i = 0; i < NTW; ++i)
            if ((int)threadIdx.x + 192 * i < S::TWN) reinterpret_cast<dvec2*>(lds)[threadIdx.x + 192 * i] = twr[i];
        __syncthreads();
    };
    const int cc = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int nxc = (g.Nx + S::LPW - 1) / S::LPW;
    const int y = blockIdx.x / nxc;
    const int L = lane / S::G;
    const int x = (blockIdx.x - y * nxc) * S::LPW + L;
    ZWCtx c;
    c.gi = lane % S::G;
    c.line_ok = x < g.Nx;
    c.base = ((long)y * g.Nx + (c.line_ok ? x : 0)) * g.nkz;
    c.fsz = (long)g.Ny * g.Nx * g.nkz;
    c.nkz = g.nkz;
    c.dk = 2 * PI / g.Lz;
    c.T = T_l + (cc * S::LPW + L) * S::LBUF;
    c.tw = lds;
    const double rotation = tab[blockIdx.y].rotation;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
    double2* __restrict__ zo = zo0 + blockIdx.y * sx;
    auto share = [&](int f, const double (&v)[PV]) {
#pragma unroll
        for (int m = 0; m < PV; ++m) ex[(f * PV + m) * 64 + lane] = v[m];
    };
    auto get = [&](int f, int m) { return ex[(f * PV + m) * 64 + lane]; };
    if constexpr (METHOD == NL_ROT) {
        double u[PV], w[PV];
        zw_c2r<S, false, 1>(c, xp, cc, 3 + cc, u, w, twiddles);
        __syncthreads();
        share(cc, u);
        share(3 + cc, w);
        __syncthreads();
        // cross(vort, u) (diffops.cpp:2598-2605): wavefront 0 takes f0 and f1, 2 takes f2
#pragma unroll
        for (int m = 0; m < PV; ++m) {
            if (cc == 0) {
                const double a0 = get(0, m), a1 = get(1, m), a2 = get(2, m);
                const double b0 = get(3, m), b1 = get(4, m), b2 = get(5, m);
                u[m] = b1 * a2 - b2 * a1;
                w[m] = b2 * a0 - b0 * a2;
                if (rotation != 0.0) {  // nse.cpp:61-80
                    u[m] -= rotation * a1;
                    w[m] += rotation * a0;
                }
            } else if (cc == 2) {
                u[m] = get(3, m) * get(1, m) - get(4, m) * get(0, m);
            }
        }
        __syncthreads();
        if (cc == 0) zw_r2c<S, true>(c, zo, u, w, 0, 1);
        else if (cc == 2) zw_r2c<S, false>(c, zo, u, u, 2, -1);
    } else if constexpr (METHOD == NL_CONV || METHOD == NL_SKEW) {
        // f_i = sum_j (s u_j) du_i/dx_j, terms added in the order j = x, y, z
        // (diffops.cpp:3192-3199, 3626-3633). The skew-symmetric form shares
        // h = u/2: halving is exact, so s u_j is h_j, u_j is 2 h_j and u_i u_j is
        // 4 (h_i h_j), all with the bits of the unscaled products.
        //
        // Skew-symmetric outputs: the z-derivative part of div(u u)/2
        // (diffops.cpp:3254-3279) is added here, in z-spectral space:
        // field i = f_i + 1/2 i kz (u_i u_z) (i = 0, 1, 2), then u_0u_0, u_0u_1,
        // u_0u_2, u_1u_1, u_1u_2 in fields 3-7; u_2u_2 is needed only for that
        // z-derivative and never leaves. The forward transforms add the x and y
        // parts of the divergence.
        constexpr bool SK = (METHOD == NL_SKEW);
        constexpr double s = SK ? 0.5 : 1.0, us = SK ? 2.0 : 1.0;
        double h[PV], dx[PV], dy[PV], dz[PV], f[PV];
        zw_c2r<S, true, 8>(c, xp, cc, -1, h, dz, twiddles);      // u_c, du_c/dz
        zw_c2r<S, false, 8>(c, xp, 6 + cc, 3 + cc, dx, dy, [] {});  // du_c/dx, du_c/dy
        if constexpr (SK) {
#pragma unroll
            for (int m = 0; m < PV; ++m) h[m] *= s;
        }
        __syncthreads();
        share(cc, h);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < PV; ++m) {
            const double h0 = get(0, m), h1 = get(1, m), h2 = get(2, m);
            f[m] = 0.0 + h0 * dx[m];
            f[m] += h1 * dy[m];
            f[m] += h2 * dz[m];
            if (rotation != 0.0) {  // nse.cpp:61-80
                if (cc == 0) f[m] -= rotation * (us * h1);
                if (cc == 1) f[m] += rotation * (us * h0);
            }
            if constexpr (SK) {  // u_i u_z; u_0u_0 and u_0u_1, or u_1u_1 (diffops.cpp:2336-2388)
                dx[m] = 4.0 * (h[m] * h2);
                dy[m] = 4.0 * (h[m] * h[m]);
                dz[m] = cc == 0 ? 4.0 * (h0 * h1) : 0.0;
            }
        }
        __syncthreads();
        if constexpr (SK) {
            zw_r2c<S, true>(c, zo, f, dx, cc, cc == 0 ? 5 : cc == 1 ? 7 : -1, 0.5);
            if (cc < 2) zw_r2c<S, true>(c, zo, dy, dz, cc == 0 ? 3 : 6, cc == 0 ? 4 : -1);
        } else {
            // f0 and f1 in one transform of wavefront 0, f2 in one of wavefront 2
            double* const hand = reinterpret_cast<double*>(T_l + S::LPW * S::LBUF) + lane;  // wavefront 1's rows
            if (cc == 1) {
#pragma unroll
                for (int m = 0; m < PV; ++m) hand[64 * m] = f[m];
            }
            __syncthreads();
            if (cc == 0) {
#pragma unroll
                for (int m = 0; m < PV; ++m) dx[m] = hand[64 * m];
                zw_r2c<S, true>(c, zo, f, dx, 0, 1);
            } else if (cc == 2) {
                zw_r2c<S, false>(c, zo, f, f, 2, -1);
            }
        }
    } else {
        double u[PV], pa[PV], pb[PV], ga[PV], gb[PV];
        zw_c2r<S, false, 1>(c, xp, cc, -1, u, pa, twiddles);
        __syncthreads();
        share(cc, u);
        __syncthreads();
        // outer(u, u) (diffops.cpp:2336-2388): 00 01, 02 11, 12 22; with rotation g, the rotation terms only
        const int i0 = cc == 2 ? 1 : 0, j0 = cc == 0 ? 0 : 2, i1 = cc == 0 ? 0 : cc, j1 = cc == 2 ? 2 : 1;
#pragma unroll
        for (int m = 0; m < PV; ++m) {
            pa[m] = get(i0, m) * get(j0, m);
            pb[m] = get(i1, m) * get(j1, m);
            ga[m] = cc == 0 ? -(rotation * get(1, m)) : 0.0;
            gb[m] = cc == 0 ? rotation * get(0, m) : 0.0;
        }
        __syncthreads();
        if (want_g && cc < 2) zw_r2c<S, true>(c, zo, ga, gb, cc == 0 ? 0 : 2, cc == 0 ? 1 : -1);
        zw_r2c<S, true>(c, zo, pa, pb, 3 + 2 * cc, 4 + 2 * cc);
    }
}

int zpass_xb(const Geom& g, int nphys, const NLTune& tn);

template <int METHOD, int NZ>
void launch_z_t(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, int want_g, const double2* xp,
                       double2* zo, long sx, const NLTune& tn, hipStream_t st) {
    if constexpr (zwave_size(NZ)) {
        using S = ZLine<NZ>;
        const long waves = (long)g.Ny * ((g.Nx + S::LPW - 1) / S::LPW);
        if constexpr (zsplit(METHOD, NZ)) {
            constexpr size_t lds = zsplit_lds<METHOD, NZ>();
            allow_lds(k_zsplit<METHOD, NZ>, lds);
            k_zsplit<METHOD, NZ><<<dim3((unsigned)waves, n), 192, lds, st>>>(g, pz.tw, tab, want_g, xp, zo, sx);
        } else {
            const int wb = tn.zwb > 0 ? tn.zwb : 4;
            const size_t lds = (size_t)(S::TWN + wb * S::LPW * S::LBUF) * sizeof(double2);
            const dim3 grid((unsigned)((waves + wb - 1) / wb), n);
            allow_lds(k_zwave<METHOD, NZ>, lds);
            k_zwave<METHOD, NZ><<<grid, 64 * wb, lds, st>>>(g, pz.tw, tab, want_g, xp, zo, sx);
        }
    } else {
        const int nphys = zpass_nphys(METHOD);
        const int XB = zpass_xb(g, nphys, tn);
        const size_t lds = (size_t)g.Nz * sizeof(double2) +
                           (size_t)XB * (2 * lpitch(g.Nz) * sizeof(double2) + (size_t)g.Nz * nphys * sizeof(double));
        const dim3 grid(g.Ny * ((g.Nx + XB - 1) / XB), n);
        allow_lds(k_zpass<METHOD>, lds);
        k_zpass<METHOD><<<grid, 256, lds, st>>>(g, pz, XB, tab, want_g, xp, zo, sx);
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
