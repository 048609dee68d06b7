// The z pass of the nonlinear term and of the CFL factor: dispatch over the
// forms, and the CFL kernels.
#include <hip/hip_runtime.h>

#include "cfg_zpass.hpp"

namespace cfg {

// ---- CFL factor -------------------------------------------------------------
// FlowField::CFLfactor(Ubase, Wbase) as DNSAlgorithm::CFL calls it
// (flowfield.cpp:4035-4068, dnsalgo.cpp:63-67): the largest of
// (u_i + U_i(y)) / dx_i over every grid point and component, signed as in the
// reference, floored at 0; dx_y is the local Chebyshev spacing. The physical
// velocity comes from the divergence form's inverse transforms, which add U, W
// and -Vsuck to the (0,0) mode; Vsuck is added back for v. One partial maximum
// per block, then one per member.
__global__ void __launch_bounds__(256) k_zcfl(Geom g, FFTPlan pz, int XB, const NLMember* __restrict__ tab,
                                              const double2* __restrict__ xp0, long sx, double* __restrict__ part) {
    extern __shared__ double2 lds[];
    __shared__ double red[4];
    const double vs = tab[blockIdx.y].Vsuck;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
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
    zc2r_pair(c, xp, 0, false, 0, 1, false, 1);
    zc2r_pair(c, xp, 2, false, 2, -1, false, -1);
    const int Ny = g.Ny, y = c.y;
    const double piN = PI / (Ny - 1), rad = (g.b - g.a) / 2, cen = (g.b + g.a) / 2;  // chebypoints (chebyshev.cpp:746-754)
    auto yc = [&](int j) { return cen + rad * cos(j * piN); };
    const double dy = (y == 0 || y == Ny - 1) ? yc(0) - yc(1) : (yc(y - 1) - yc(y + 1)) / 2.0;
    const double dx = g.Lx / g.Nx, dz = g.Lz / g.Nz;
    const double *u0 = physf(c, 0), *u1 = physf(c, 1), *u2 = physf(c, 2);
    double m = 0.0;
    for (int w = threadIdx.x; w < c.nl * g.Nz; w += blockDim.x) {
        m = fmax(m, u0[w] / dx);
        m = fmax(m, (u1[w] + vs) / dy);
        m = fmax(m, u2[w] / dz);
    }
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fmax(m, red[i]);
        part[(long)blockIdx.y * gridDim.x + blockIdx.x] = m;
    }
}

// The same with a wavefront per group of lines, for the wavefront FFT lengths: the
// transforms have no block barriers, and a line's largest value is divided instead of
// every value (division by a positive spacing is monotone, so the result is the same).
// us per launch, LDS lines -> wavefront lines: 48x35x48 12.6 -> 6.5 (and 5.7 -> 1.7 for
// the reduction of its fewer blocks), 32^3 9.0 -> 5.2, 64^3 12.5 -> 6.2, 96^3 31.3 -> 11.2,
// 128^3 63 -> 18, 192x129x192 128 -> 32.
template <int NZ>
__global__ void __launch_bounds__(256) k_zcfl_w(Geom g, const double2* __restrict__ twg,
                                                const NLMember* __restrict__ tab, const double2* __restrict__ xp0,
                                                long sx, double* __restrict__ part) {
    using S = ZLine<NZ>;
    constexpr int PV = S::PV;
    extern __shared__ double2 lds[];
    __shared__ double red[4];
    for (int i = threadIdx.x; i < S::TWN; i += 256) lds[i] = twg[S::tw_power(i)];
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int nxc = (g.Nx + S::LPW - 1) / S::LPW;
    const int wg = min((int)blockIdx.x * 4 + wave, g.Ny * nxc - 1);  // the last block may repeat a group
    const int y = wg / nxc, L = lane / S::G, x = (wg - y * nxc) * S::LPW + L;
    ZWCtx c;
    c.gi = lane % S::G;
    c.line_ok = x < g.Nx;
    c.base = ((long)y * g.Nx + (c.line_ok ? x : 0)) * g.nkz;
    c.fsz = (long)g.Ny * g.Nx * g.nkz;
    c.nkz = g.nkz;
    c.dk = 2 * PI / g.Lz;
    c.T = lds + S::TWN + (wave * S::LPW + L) * S::LBUF;
    c.tw = lds;
    const double2* __restrict__ xp = xp0 + blockIdx.y * sx;
    double u0[PV], u1[PV], u2[PV], none[PV];
    zw_c2r<S>(c, xp, 0, 1, u0, u1);
    zw_c2r<S>(c, xp, 2, -1, u2, none);
    const int Ny = g.Ny;
    const double piN = PI / (Ny - 1), rad = (g.b - g.a) / 2, cen = (g.b + g.a) / 2;
    auto yc = [&](int j) { return cen + rad * cos(j * piN); };
    const double dy = (y == 0 || y == Ny - 1) ? yc(0) - yc(1) : (yc(y - 1) - yc(y + 1)) / 2.0;
    double m = 0.0;
    if (c.line_ok && c.gi < S::PL) {
        const double vs = tab[blockIdx.y].Vsuck;
        double m0 = u0[0], m1 = u1[0] + vs, m2 = u2[0];
#pragma unroll
        for (int k = 1; k < PV; ++k) {
            m0 = fmax(m0, u0[k]);
            m1 = fmax(m1, u1[k] + vs);
            m2 = fmax(m2, u2[k]);
        }
        m = fmax(fmax(m, m0 / (g.Lx / g.Nx)), fmax(m1 / dy, m2 / (g.Lz / g.Nz)));
    }
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[(long)blockIdx.y * gridDim.x + blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

__global__ void __launch_bounds__(256) k_cfl_reduce(int nb, const double* __restrict__ part, double* __restrict__ out) {
    __shared__ double red[4];
    const double* p = part + (long)blockIdx.x * nb;
    double m = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) m = fmax(m, p[i]);
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fmax(m, red[i]);
        out[blockIdx.x] = m;
    }
}

// LDS budget per block (set from the device's opt-in limit at start-up)
static size_t g_lds_budget = 64 * 1024;
void set_lds_budget(size_t bytes) { g_lds_budget = bytes; }
size_t lds_budget() { return g_lds_budget; }

// real physical lines per (y, x) line the z-pass keeps in LDS
int zpass_nphys(int method) { return method == NL_ROT ? 6 : (method == NL_DIV ? 5 : 7); }

// largest z-pass lines per block that fit the LDS budget (power of two <= 32)
int zpass_xb_max(const Geom& g, int nphys) {
    const long per = 32L * lpitch(g.Nz) + 8L * g.Nz * nphys;  // two complex work lines + nphys real lines
    const long avail = (long)g_lds_budget - 16L * g.Nz;
    int xb = 1;
    while (xb < 32 && xb * 2 <= g.Nx && (long)(xb * 2) * per <= avail) xb *= 2;
    return xb;
}

int zpass_xb(const Geom& g, int nphys, const NLTune& tn) {
    const int m = zpass_xb_max(g, nphys);
    return tn.zxb > 0 ? std::min(tn.zxb, m) : m;
}

#define CFG_Z_EXTERN(F)                                                                                            \
    extern template void launch_z<F>(const Geom&, const FFTPlan&, int, const NLMember*, int, const double2*, double2*, \
                                     long, const NLTune&, hipStream_t);
CFG_Z_EXTERN(NL_ROT)
CFG_Z_EXTERN(NL_CONV)
CFG_Z_EXTERN(NL_DIV)
CFG_Z_EXTERN(NL_SKEW)
#undef CFG_Z_EXTERN

void launch_z_any(int method, const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, int want_g,
                         const double2* xp, double2* zo, long sx, const NLTune& tn, hipStream_t st) {
    switch (method) {
        case NL_ROT: launch_z<NL_ROT>(g, pz, n, tab, want_g, xp, zo, sx, tn, st); break;
        case NL_CONV: launch_z<NL_CONV>(g, pz, n, tab, want_g, xp, zo, sx, tn, st); break;
        case NL_SKEW: launch_z<NL_SKEW>(g, pz, n, tab, want_g, xp, zo, sx, tn, st); break;
        default: launch_z<NL_DIV>(g, pz, n, tab, want_g, xp, zo, sx, tn, st);
    }
}

// returns the partial maxima per member
template <int NZ>
static int launch_zcfl_t(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, const double2* xp, long sx,
                         double* part, hipStream_t st) {
    if constexpr (zwave_size(NZ)) {
        using S = ZLine<NZ>;
        const int nb = (g.Ny * ((g.Nx + S::LPW - 1) / S::LPW) + 3) / 4;
        constexpr size_t lds = (size_t)(S::TWN + 4 * S::LPW * S::LBUF) * sizeof(double2);
        allow_lds(k_zcfl_w<NZ>, lds);
        k_zcfl_w<NZ><<<dim3((unsigned)nb, n), 256, lds, st>>>(g, pz.tw, tab, xp, sx, part);
        return nb;
    } else {
        const int XB = zpass_xb_max(g, 3), nb = g.Ny * ((g.Nx + XB - 1) / XB);
        const size_t lds = (size_t)g.Nz * sizeof(double2) +
                           (size_t)XB * (2 * lpitch(g.Nz) * sizeof(double2) + (size_t)g.Nz * 3 * sizeof(double));
        allow_lds(k_zcfl, lds);
        k_zcfl<<<dim3((unsigned)nb, n), 256, lds, st>>>(g, pz, XB, tab, xp, sx, part);
        return nb;
    }
}

int launch_zcfl(const Geom& g, const FFTPlan& pz, int n, const NLMember* tab, const double2* xp, long sx, double* part,
                hipStream_t st) {
    switch (g.Nz) {
#define CASE_Z(N) \
    case N: return launch_zcfl_t<N>(g, pz, n, tab, xp, sx, part, st);
        CFG_FFT_SIZES(CASE_Z)
#undef CASE_Z
        default: return launch_zcfl_t<0>(g, pz, n, tab, xp, sx, part, st);
    }
}

void launch_cfl_reduce(int n, int nb, const double* part, double* out, hipStream_t st) {
    k_cfl_reduce<<<n, 256, 0, st>>>(nb, part, out);
}

}  // namespace cfg
