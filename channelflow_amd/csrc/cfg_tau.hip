// Tau-solver kernels of the MI355X DNS time step (gfx950, FP64): the per-mode
// set-up, NSE::solve, PressureSolver::solve and NSE::linear, one (kx, kz) mode
// (or one real part of it) per segment of a wavefront.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cfg_dev.hpp"
#include "cfg_math.hpp"
#include "cfg_wave.hpp"

namespace cfg {

// Block order of a launch over (mode block, member) pairs: the dispatcher
// hands consecutive workgroups to the 8 XCDs in turn, so the linear block
// index is renumbered to put a contiguous range of pairs on each XCD, members
// fastest. The members of a launch share their tau factors, which one XCD
// then reads from its own L2 for every member after the first.
__device__ __forceinline__ void xcd_block(int nmem, int& mode_block, int& member) {
    const int T = gridDim.x;  // mode blocks x members
    const int L = blockIdx.x;
    const int q = T / NXCD, r = T % NXCD, x = L % NXCD;
    const int p = x * q + (x < r ? x : r) + L / NXCD;
    mode_block = p / nmem;
    member = p - mode_block * nmem;
}

// ===========================================================================
// Tau solver kernels: one thread per live mode (tausolver.cpp, nse.cpp:479)
// ===========================================================================
__device__ TauView make_view(const Geom& g, const TauSet& s, int m, double nu, bool taucorr) {
    const int ikx = m % g.nkx, ikz = m / g.nkx;
    const int kx = kx_of(g, ikx), kz = ikz;
    const double pi2 = PI * PI;
    const double kappa2 = 4 * pi2 * ((kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz));
    const double c = 4.0 * pi2 * nu;
    const double lambda = s.lambda_t + c * ((kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz));
    double* cm = s.coef + (long)m * TAU_NA * g.Ny;
    auto A = [&](int k) { return SV{cm + (long)k * g.Ny, 1}; };
    TauView t;
    t.ph = HelmholtzView{A(0), A(1), A(2), kappa2, g.Ny};
    t.vh = HelmholtzView{A(3), A(4), A(5), lambda, g.Ny};
    t.Pp = A(6);
    t.vp = A(7);
    t.P0 = A(8);
    t.v0 = A(9);
    t.scal = s.scal + (long)m * 6;
    t.sstride = 1;
    t.nu = nu;
    t.a = g.a;
    t.b = g.b;
    t.kx2pi = 2 * PI * kx / g.Lx;
    t.kz2pi = 2 * PI * kz / g.Lz;
    t.zero_mode = (kx == 0 && kz == 0);
    t.taucorrection = taucorr;
    return t;
}

// TauSolver constructor per mode (tausolver.cpp:81-176), T modes per block,
// one thread each. ALL: the mode's whole working set in LDS, its 10 tau
// profiles (array a at element (a*Ny + n)*T + t), 6 scalars and 2 scratch
// profiles, copied to the mode-major tau set with contiguous writes at the end.
// Otherwise (tall grids, where a block of 64 KB would hold fewer than 8 such
// working sets) the profiles and scalars are built in place in the tau set and
// only the 2 scratch profiles are in LDS. The arithmetic is tau_setup's either
// way (the sequential set-up, bit for bit the oracle's); only the memory the
// recurrences store to and reload from moves.
template <bool ALL>
__global__ void k_tau_setup(Geom g, TauSet s, double nu, int taucorr) {
    extern __shared__ double sl[];
    const int T = blockDim.x, t = threadIdx.x;
    const int m0 = blockIdx.x * T, m = m0 + t;
    const int Ny = g.Ny;
    const long arr = (long)Ny * T;  // one profile of the block's modes
    if (m < g.M) {
        TauView v = make_view(g, s, m, nu, taucorr != 0);
        auto A = [&](int a) { return SV{sl + a * arr + t, T}; };
        if constexpr (ALL) {
            v.ph.band = A(0);
            v.ph.up = A(1);
            v.ph.invd = A(2);
            v.vh.band = A(3);
            v.vh.up = A(4);
            v.vh.invd = A(5);
            v.Pp = A(6);
            v.vp = A(7);
            v.P0 = A(8);
            v.v0 = A(9);
            v.scal = sl + (TAU_NA + 2) * arr + t;
            v.sstride = T;
            tau_setup(v, A(TAU_NA), A(TAU_NA + 1));
        } else {
            tau_setup(v, A(0), A(1));
        }
    }
    if constexpr (ALL) {
        __syncthreads();
        const int nm = min(T, g.M - m0);
        __attribute__((address_space(1))) double* coef = gmem_w(s.coef) + (long)m0 * TAU_NA * Ny;
        for (int i = t; i < nm * TAU_NA * Ny; i += T) {
            const int mm = i / (TAU_NA * Ny), r = i - mm * (TAU_NA * Ny), a = r / Ny, n = r - a * Ny;
            coef[i] = sl[a * arr + (long)n * T + mm];
        }
        __attribute__((address_space(1))) double* scal = gmem_w(s.scal) + (long)m0 * 6;
        for (int i = t; i < nm * 6; i += T) scal[i] = sl[(TAU_NA + 2) * arr + (long)(i % 6) * T + i / 6];
    }
}

// modes per block of the set-up within 64 KB of LDS, at most 64: whole working
// sets (12 profiles and 6 scalars each) where 8 or more fit, else scratch
// profiles only (2 each)
static int tau_setup_modes(int Ny, bool* all) {
    const long whole = ((TAU_NA + 2L) * Ny + 6) * (long)sizeof(double), scratch = 2L * Ny * (long)sizeof(double);
    const long T = (64L * 1024) / whole;
    *all = T >= 8;
    return (int)std::max(1L, std::min(64L, (64L * 1024) / (*all ? whole : scratch)));
}

void launch_tau_setup(const Geom& g, const TauSet& s, double nu, bool taucorr, hipStream_t st) {
    bool all = false;
    const int T = tau_setup_modes(g.Ny, &all);
    const dim3 grid((g.M + T - 1) / T);
    if (all) {
        const size_t lds = (size_t)((TAU_NA + 2L) * g.Ny + 6) * T * sizeof(double);
        k_tau_setup<true><<<grid, T, lds, st>>>(g, s, nu, taucorr ? 1 : 0);
    } else {
        const size_t lds = (size_t)2 * g.Ny * T * sizeof(double);
        k_tau_setup<false><<<grid, T, lds, st>>>(g, s, nu, taucorr ? 1 : 0);
    }
}

// Tau solve (NSE::solve, nse.cpp:479-575; TauSolver::solve, tausolver.cpp:347-450,
// with solve_P_and_v :193-251). The operators of a mode are real, and the real
// and imaginary parts of its equations couple only as (v, P real; u, w
// imaginary) and (v, P imaginary; u, w real): two independent real problems
//   P'' - kappa^2 P = Ry' - s (kx Rx + kz Rz),  v from P' - Ry,
//   u from s kx P - Rx,  w from s kz P - Rz,
// s = +1 with (Ry.re, Rx.im, Rz.im) and s = -1 with (Ry.im, Rx.re, Rz.re). Each
// runs on its own W-lane segment of a wavefront.

// The right-hand-side rows of a block's modes, [comp][n] at rows row0 .. row0 +
// nrow (row = comp Ny + n): sum_j coef_j in_j (the multistep / Runge-Kutta
// combination, dnsalgo.cpp:218-224, 668-673), handed to put(mode slot, row, re,
// im). The term count is a template parameter and UNR rows are loaded per pass,
// so the NT x UNR loads of a pass are all in flight before the first is summed
// (36 or 54 in flight were no faster: 192x129x192 136-138 us against 130).
template <int NT, int MPB, class Put>
__device__ __forceinline__ void tau_stage_rhs(const TauMember& me, const Geom& g, int m0, int nthr, Put&& put) {
    constexpr int UNR = NT <= 2 ? 8 : 16 / NT;  // 16 loads in flight at most
    const __attribute__((address_space(1))) dvec2* in[NT];
    double coef[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        in[j] = gmem(reinterpret_cast<const dvec2*>(me.in[j]));
        coef[j] = me.coef[j];
    }
    const int ww = threadIdx.x % MPB, nrow = 3 * g.Ny, step = nthr / MPB;
    const int mm = min(m0 + ww, g.M - 1);  // slots past the last mode repeat it
    for (int row = threadIdx.x / MPB; row < nrow; row += UNR * step) {
        dvec2 v[UNR][NT];
#pragma unroll
        for (int r = 0; r < UNR; ++r) {
            // rows past the end repeat the last one, so that every load is issued unconditionally
            const long off = (long)min(row + r * step, nrow - 1) * g.M + mm;
#pragma unroll
            for (int j = 0; j < NT; ++j) v[r][j] = in[j][off];
        }
#pragma unroll
        for (int r = 0; r < UNR; ++r) {
            dvec2 acc = dvec2{0.0, 0.0};
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                acc.x += coef[j] * v[r][j].x;
                acc.y += coef[j] * v[r][j].y;
            }
            if (row + r * step < nrow) put(ww, row + r * step, acc);
        }
    }
}
template <int MPB, class Put>
__device__ __forceinline__ void tau_stage(const TauMember& me, const Geom& g, int m0, int nthr, Put&& put) {
    switch (me.nterms) {
        case 1: tau_stage_rhs<1, MPB>(me, g, m0, nthr, put); break;
        case 2: tau_stage_rhs<2, MPB>(me, g, m0, nthr, put); break;
        case 3: tau_stage_rhs<3, MPB>(me, g, m0, nthr, put); break;
        case 4: tau_stage_rhs<4, MPB>(me, g, m0, nthr, put); break;
        case 5: tau_stage_rhs<5, MPB>(me, g, m0, nthr, put); break;
        case 6: tau_stage_rhs<6, MPB>(me, g, m0, nthr, put); break;
        case 7: tau_stage_rhs<7, MPB>(me, g, m0, nthr, put); break;
        default: tau_stage_rhs<MAX_TERMS, MPB>(me, g, m0, nthr, put); break;
    }
}

// LDS of a tau-solve block of MPB modes: the rows of its 2 MPB real problems,
// [mode][part][comp] of tau_pitch(Ny) doubles, then the rows of B (3 of 2KW
// doubles, zero past Ny).
__host__ __device__ constexpr int tau_pitch(int Ny) { return Ny + 1; }  // even (Ny is odd): 16-byte pairs
// Doubles of a row per lane (wrow_pos): padded above 16 lanes at K = 4 (128x193x128 with
// 8 doubles 120 us, with 10 107)
constexpr int tau_lp(int K) { return K == 4 ? 2 * K + 2 : 2 * K; }
template <int K>
__host__ __device__ constexpr int tau_row(int Ny) { return (wrow_pos<K, tau_lp(K)>(Ny) + 2) / 2 * 2; }
constexpr size_t tau_lds(int row, int lane, int W, int MPB) {
    return ((size_t)MPB * 6 * row + (size_t)3 * lane * W) * sizeof(double);
}

// Waves per SIMD a variant is compiled for, where its registers fit without
// spilling more than a few values (K = 5: 256 registers; a third wave at K = 3
// spills 164 bytes, one 64^3 field 14.6 -> 21.3 us).
constexpr int tau_waves(int K) { return K == 1 ? 4 : K == 2 ? 3 : K <= 5 ? 2 : 1; }

// The kx = kz = 0 mode: P from Ry', v = 0, u and w from the velocity operator; real
// parts only. For a whole block, c and seg as in the kernels below.
template <int K, int W, int NTHR, int LP, class Op>
__device__ __forceinline__ void tau_mean_mode(const Geom& g, const TauMember& me, const TauSet& s, double nu,
                                              const gcdouble coef, double* const R, int RP, int seg, const WCtx& c,
                                              __attribute__((address_space(1))) dvec2* __restrict__ u,
                                              __attribute__((address_space(1))) dvec2* __restrict__ q) {
    const int Ny = g.Ny;
    auto at = [&](int row) { return LP == 2 * K ? row + row / Ny * (RP - Ny) : row / Ny * RP + wrow_pos<K, LP>(row % Ny); };
    for (int row = threadIdx.x; row < 3 * Ny; row += NTHR) {
        double acc = 0.0;
        for (int j = 0; j < me.nterms; ++j) acc += me.coef[j] * gmem(me.in[j])[2L * row * g.M];
        R[at(row)] = acc;
    }
    __syncthreads();
    const SolveConst zc = me.sc;
    // segment 0 solves for P, the first two from the next wavefront on for u and w
    constexpr int U0 = 64 / W;
    static_assert(NTHR / W >= U0 + 2, "the block has these segments");
    if (seg == 0) {
        const Op op(coef, Ny, 0, 0u, 0.0, c);
        WV<K> y[1], f[1], x[1];
        y[0] = wrow_load<K, W, LP>(R + RP, c);
        wdiff_n<K, W, 1>(y, c, f);
        op.template solve<1>(f, c, x);
        wrow_store<K, W, LP>(R + RP, c, x[0]);
    } else if (seg == U0 || seg == U0 + 1) {
        const int cc = seg - U0;
        double* const S = R + 2 * cc * RP;
        const Op op(coef, Ny, 3, 0u, s.lambda_t, c);
        const WV<K> r = wrow_load<K, W, LP>(S, c);
        const WV<K> Byy = wload<K, W>(gmem(cc == 0 ? zc.nuUbaseyy : zc.nuWbaseyy), c);
        WV<K> f[1], x[1];  // nse.cpp:505-527: nu U'' (nu W''), and a fixed mean gradient
        for (int i = 0; i < K; ++i) {
            f[0].e[i] = -(r.e[i] + Byy.e[i]);
            f[0].o[i] = -(r.o[i] + Byy.o[i]);
        }
        if (zc.bulk) {  // bulk-velocity constraint (tausolver.cpp:404-450, helmholtz.cpp:158-213)
            WV<K> two[2], sol[2];
            two[0] = f[0];
            two[1] = wzero<K, W>();
            if (c.lane == 0) two[1].e[0] = nu;
            op.template solve<2>(two, c, sol);
            const double uamean = wmean<K, W>(sol[0], c), ucmean = wmean<K, W>(sol[1], c);
            const double mu = nu * ((cc == 0 ? zc.umean : zc.wmean) - uamean) / ucmean;
            if (c.lane == 0) {
                f[0].e[0] += mu;
                *(cc == 0 ? zc.dPdx_out : zc.dPdz_out) = mu;
            }
        } else if (c.lane == 0) {
            f[0].e[0] += cc == 0 ? zc.dPdxRef : zc.dPdzRef;
        }
        op.template solve<1>(f, c, x);
        wrow_store<K, W, LP>(S, c, x[0]);
    }
    __syncthreads();
    for (int row = threadIdx.x; row < 3 * Ny; row += NTHR) {
        const double v = R[at(row)];
        const bool mid = row >= Ny && row < 2 * Ny;
        if (mid) q[(long)(row - Ny) * g.M] = dvec2{v, 0.0};
        u[(long)row * g.M] = dvec2{mid ? 0.0 : v, 0.0};
    }
}

// Blocks of a launch, in XCD order: per member the block of the kx = kz = 0
// mode alone (its mean-flow solves would run one after the other with the
// general path of the modes beside it), then blocks of MPB consecutive modes;
// the general path also passes over mode 0, and its result there is dropped.
//
// What bounds it: for one field the instruction chain of a wave, for a batch
// HBM and that chain (24 x 32^3: 63 MB in 20.8 us, one round of blocks), for
// one large field HBM (192x129x192: 434 MB in 116 us, 3.7 TB/s, of which the
// right-hand-side rows are 256-byte pieces 130 KB apart). The set keeps P+ and v+
// only: with P- and v- stored and loaded too 128^3 took 47.2 us, not 44.4,
// 192x129x192 121.0, 96^3 23.6, not 22.4, 4 of 96^3 85.6, not 83.3. Against a segment per
// complex mode with the scan multipliers recomputed for every right-hand side
// and every lane past a system masked (8557 instructions at K = 3, now about
// 2200): one 32^3 field 20.5 -> 9.2 us, 64^3 31.3 -> 14.6, 96^3 39.5 -> 23.5,
// 128^3 66.7 -> 48.0, 192x129x192 138.7 -> 120.8, 24 x 32^3 26.8 -> 20.8.
template <int K, int W, int MPB>
__global__ void __launch_bounds__(2 * W * MPB) __attribute__((amdgpu_waves_per_eu(tau_waves(K))))
k_tau_solve_wave(Geom g, const double* __restrict__ hb, int nmem, const TauMember* __restrict__ tab) {
    extern __shared__ double2 lds2[];
    double* const lds = reinterpret_cast<double*>(lds2);
    constexpr int nthr = 2 * W * MPB, HP = 2 * K * W;
    int mblk, mem;
    xcd_block(nmem, mblk, mem);
    const TauMember& me = tab[mem];
    const TauSet s = me.set;
    const double nu = me.nu;
    const int taucorr = me.taucorr;
    __attribute__((address_space(1))) dvec2* __restrict__ u = gmem_w(reinterpret_cast<dvec2*>(me.u));
    __attribute__((address_space(1))) dvec2* __restrict__ q = gmem_w(reinterpret_cast<dvec2*>(me.q));
    const int Ny = g.Ny, RP = tau_pitch(Ny);
    double* const hbl = lds + MPB * 6 * RP;
    for (int i = threadIdx.x; i < 3 * HP; i += nthr) {
        const int r = i / HP, n = i % HP;
        hbl[i] = n < Ny ? hb[r * Ny + n] : 0.0;
    }
    for (int i = threadIdx.x; i < 6 * MPB; i += nthr) lds[i * RP + Ny] = 0.0;  // the rows' padding
    WCtx c;
    c.N = Ny;
    c.Me = (Ny + 1) / 2;
    c.Mo = (Ny - 1) / 2;
    c.Nb = Ny - 1;
    c.Nc = Ny - 1;
    c.lane = threadIdx.x % W;
    c.L = g.b - g.a;
    c.hb = hbl;
    const int seg = threadIdx.x / W;
    const gcdouble coef = gmem(s.coef);
    const double pi2 = PI * PI;

    if (mblk == 0) {
        tau_mean_mode<K, W, nthr, 2 * K, HelmOp<K, W>>(g, me, s, nu, coef, lds, RP, seg, c, u, q);
        return;
    }

    const int m0 = (mblk - 1) * MPB;
    const int w = seg >> 1, part = seg & 1;
    const int m = min(m0 + w, g.M - 1);
    // part 0 takes Ry.re, Rx.im, Rz.im; part 1 Ry.im, Rx.re, Rz.re
    auto slot = [&](int ww, int pt, int row) {
        const int comp = (row >= Ny) + (row >= 2 * Ny);
        return ((ww * 2 + pt) * 3 + comp) * RP + row - comp * Ny;
    };
    const unsigned fo = (unsigned)m * (TAU_NA * Ny);  // this mode's factors
    tau_stage<MPB>(me, g, m0, nthr, [&](int ww, int row, dvec2 v) {
        const bool mid = row >= Ny && row < 2 * Ny;
        lds[slot(ww, 0, row)] = mid ? v.x : v.y;
        lds[slot(ww, 1, row)] = mid ? v.y : v.x;
    });
    __syncthreads();
    const int ikx = m % g.nkx, ikz = m / g.nkx;
    const int kx = kx_of(g, ikx), kz = ikz;
    const double kk = (kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz);
    const double kappa2 = 4 * pi2 * kk;
    const double lambda = s.lambda_t + (4.0 * pi2 * nu) * kk;
    const double sgn = part ? -1.0 : 1.0;
    const double ax = sgn * (2 * PI * kx / g.Lx), az = sgn * (2 * PI * kz / g.Lz);
    double* const Sx = lds + (seg * 3 + 0) * RP;
    double* const Sy = lds + (seg * 3 + 1) * RP;
    double* const Sz = lds + (seg * 3 + 2) * RP;
    WV<K> P[1], v[1];
    {
        WV<K> f[1], t[1];
        t[0] = wrow_load<K, W>(Sy, c);
        wdiff_n<K, W, 1>(t, c, f);
        const WV<K> X = wrow_load<K, W>(Sx, c), Z = wrow_load<K, W>(Sz, c);
        for (int k = 0; k < K; ++k) {
            f[0].e[k] -= ax * X.e[k] + az * Z.e[k];
            f[0].o[k] -= ax * X.o[k] + az * Z.o[k];
        }
        const HelmOp<K, W> op(wfac3<K, W>(coef, Ny, 0, fo, c), kappa2, c);
        op.template solve<1>(f, c, P);
    }
    const HelmOp<K, W> vop(wfac3<K, W>(coef, Ny, 3, fo, c), lambda, c);  // velocity operator: v, then u and w
    {
        WV<K> f[1], t[1];
        wdiff_n<K, W, 1>(P, c, f);
        t[0] = wrow_load<K, W>(Sy, c);
        for (int k = 0; k < K; ++k) {
            f[0].e[k] -= t[0].e[k];
            f[0].o[k] -= t[0].o[k];
        }
        vop.template solve<1>(f, c, v);
        // influence-matrix correction (tausolver.cpp:178-191)
        double dvb[1], dva[1];
        wdiff_n<K, W, 1>(v, c, f);
        wends_n<K, W, 1>(f, c, dvb, dva);
        const gcdouble sc = gmem(s.scal) + 6L * m;
        const double dplus = -sc[0] * dvb[0] - sc[1] * dva[0];
        const double dminus = -sc[2] * dvb[0] - sc[3] * dva[0];
        // P- and v- are the mirrors of P+ and v+: (e, -o) and (-e, o)
        const WV<K> Pp = wfac<K, W>(coef, Ny, 6, fo, c), vp = wfac<K, W>(coef, Ny, 7, fo, c);
        for (int k = 0; k < K; ++k) {
            P[0].e[k] += dplus * Pp.e[k] + dminus * Pp.e[k];
            P[0].o[k] += dplus * Pp.o[k] - dminus * Pp.o[k];
            v[0].e[k] += dplus * vp.e[k] - dminus * vp.e[k];
            v[0].o[k] += dplus * vp.o[k] + dminus * vp.o[k];
        }
        if (taucorr) {
            const int Nb = c.Nb;
            const WV<K> P0 = wfac<K, W>(coef, Ny, 8, fo, c), v0 = wfac<K, W>(coef, Ny, 9, fo, c);
            const double sigma1_Nb = lambda * wtop<K, W>(v[0], c) - Sy[Nb];
            double sigma1_Nb1 = lambda * wtop1<K, W>(v[0], c) - Sy[Nb - 1];
            sigma1_Nb1 += (4.0 / c.L) * Nb * wtop<K, W>(P[0], c);
            const double sigmaNb = sigma1_Nb / (1.0 - sc[5]);
            const double sigmaNb1 = sigma1_Nb1 / (1.0 - sc[4]);
            for (int k = 0; k < K; ++k) {
                P[0].e[k] += sigmaNb1 * P0.e[k];
                P[0].o[k] += sigmaNb * P0.o[k];
                v[0].e[k] += sigmaNb * v0.e[k];
                v[0].o[k] += sigmaNb1 * v0.o[k];
            }
        }
    }
    wrow_store<K, W>(Sy, c, v[0]);  // the rows are this segment's alone
    // u and w, one parity at a time (fewer live registers)
    auto solve_uw = [&](const HelmPar<K, W>& op, const double (&Pk)[K], int par, int M) {
        double f[2][K], x[2][K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int n = 2 * min(K * c.lane + k, M - 1) + par;
            f[0][k] = ax * Pk[k] - Sx[n];
            f[1][k] = az * Pk[k] - Sz[n];
        }
        op.template solve<2>(f, hbl + 2 * K * c.lane + par, HP, c, x);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int i = K * c.lane + k;
            if (i < M) {
                Sx[2 * i + par] = x[0][k];
                Sz[2 * i + par] = x[1][k];
            }
        }
    };
    solve_uw(vop.e, P[0].e, 0, c.Me);
    solve_uw(vop.o, P[0].o, 1, c.Mo);
    __syncthreads();
    const int ww = threadIdx.x % MPB, mm = m0 + ww;
    const bool out = mm > 0 && mm < g.M;
    for (int row = threadIdx.x / MPB; row < 3 * Ny; row += nthr / MPB) {
        const double a = lds[slot(ww, 0, row)], b = lds[slot(ww, 1, row)];
        const bool mid = row >= Ny && row < 2 * Ny;
        if (out) u[(long)row * g.M + mm] = mid ? dvec2{a, b} : dvec2{b, a};
    }
    __syncthreads();
    wrow_store<K, W>(Sy, c, P[0]);
    __syncthreads();
    for (int row = Ny + threadIdx.x / MPB; row < 2 * Ny; row += nthr / MPB) {
        const double a = lds[slot(ww, 0, row)], b = lds[slot(ww, 1, row)];
        if (out) q[(long)(row - Ny) * g.M + mm] = dvec2{a, b};
    }
}

// The same above Ny = 191, where a mode's profiles take 32 or 64 lanes. A block of 4
// modes (64-byte pieces of a row) is 4 wavefronts, and what decides is how many blocks
// a compute unit holds, so that one loads its rows while another solves: the velocity
// operator is not held from v's solve to u's and w's, but formed one parity system at a
// time (HelmParts), which leaves 2 wavefronts per SIMD. Held, K = 4 on 32 lanes took 298
// registers and K = 6 408: a block alone on its compute unit. NP: real parts per
// segment. At NP = 2 (K = 3 on 64 lanes, above Ny = 255) both parts of a mode share its
// operators, and a block of 4 modes still has 4 wavefronts. LP: doubles of an LDS row
// per lane (wrow_pos).
// us per launch, SBDF3: a segment per complex mode / this kernel's shapes with the
// operator held / now. Ny = 193: one field of 32xNyx32 37.0 / 25.4 / 25.0, 128xNyx128 107.0 /
// 128.4 / 98.9, 8 of 32xNyx32 54.6 / 59.1 / 44.1, 24 of them 142.1 / 176.4 / 143.5; Ny = 257:
// 43.0 / 30.2 / 31.8, 138.7 / 162.5 / 132.8, 65.1 / 74.0 / 63.7, 196.1 / 223.9 / 194.4; Ny = 321:
// 45.4 / 33.4 / 34.6, 158.5 / 182.1 / 151.2, 76.5 / 86.6 / 73.9, 228.7 / 264.2 / 231.0.
template <int K, int W, int MPB, int NP>
__global__ void __launch_bounds__(2 * W * MPB / NP) __attribute__((amdgpu_waves_per_eu(2)))
k_tau_solve_tall(Geom g, const double* __restrict__ hb, int nmem, const TauMember* __restrict__ tab) {
    extern __shared__ double2 lds2[];
    double* const lds = reinterpret_cast<double*>(lds2);
    constexpr int nthr = 2 * W * MPB / NP, LP = tau_lp(K), HP = LP * W;
    using Op = HelmParts<K, W, LP>;
    auto pos = [](int n) { return wrow_pos<K, LP>(n); };
    int mblk, mem;
    xcd_block(nmem, mblk, mem);
    const TauMember& me = tab[mem];
    const TauSet s = me.set;
    const double nu = me.nu;
    const int taucorr = me.taucorr;
    __attribute__((address_space(1))) dvec2* __restrict__ u = gmem_w(reinterpret_cast<dvec2*>(me.u));
    __attribute__((address_space(1))) dvec2* __restrict__ q = gmem_w(reinterpret_cast<dvec2*>(me.q));
    const int Ny = g.Ny, RP = tau_row<K>(Ny);
    double* const hbl = lds + MPB * 6 * RP;
    for (int i = threadIdx.x; i < 3 * HP; i += nthr) {
        const int r = i / HP, at = i % HP, n = at % LP < 2 * K ? 2 * K * (at / LP) + at % LP : Ny;
        hbl[i] = n < Ny ? hb[r * Ny + n] : 0.0;
    }
    for (int i = threadIdx.x; i < 6 * MPB; i += nthr) lds[i * RP + pos(Ny)] = 0.0;  // the rows' padding
    WCtx c;
    c.N = Ny;
    c.Me = (Ny + 1) / 2;
    c.Mo = (Ny - 1) / 2;
    c.Nb = Ny - 1;
    c.Nc = Ny - 1;
    c.lane = threadIdx.x % W;
    c.L = g.b - g.a;
    c.hb = hbl;
    const int seg = threadIdx.x / W;
    const gcdouble coef = gmem(s.coef);
    if (mblk == 0) {
        tau_mean_mode<K, W, nthr, LP, Op>(g, me, s, nu, coef, lds, RP, seg, c, u, q);
        return;
    }

    const int m0 = (mblk - 1) * MPB;
    // the segment's mode and its first part: part 0 takes Ry.re, Rx.im, Rz.im; part 1 Ry.im, Rx.re, Rz.re
    const int w = NP == 2 ? seg : seg >> 1, part = NP == 2 ? 0 : seg & 1;
    const int m = min(m0 + w, g.M - 1);
    auto slot = [&](int ww, int pt, int row) {
        const int comp = (row >= Ny) + (row >= 2 * Ny);
        return ((ww * 2 + pt) * 3 + comp) * RP + pos(row - comp * Ny);
    };
    const unsigned fo = (unsigned)m * (TAU_NA * Ny);  // this mode's factors
    tau_stage<MPB>(me, g, m0, nthr, [&](int ww, int row, dvec2 v) {
        const bool mid = row >= Ny && row < 2 * Ny;
        lds[slot(ww, 0, row)] = mid ? v.x : v.y;
        lds[slot(ww, 1, row)] = mid ? v.y : v.x;
    });
    __syncthreads();
    const int ikx = m % g.nkx, ikz = m / g.nkx;
    const int kx = kx_of(g, ikx), kz = ikz;
    const double kk = (kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz);
    const double kappa2 = 4 * (PI * PI) * kk;
    const double lambda = s.lambda_t + (4.0 * (PI * PI) * nu) * kk;
    auto each = [](auto&& fn) {  // for each of the segment's parts
        fn(0);
        if constexpr (NP == 2) fn(1);
    };
    double ax[NP], az[NP];
    double *Sx[NP], *Sy[NP], *Sz[NP];
    each([&](int p) {
        const double sgn = part + p ? -1.0 : 1.0;
        ax[p] = sgn * (2 * PI * kx / g.Lx);
        az[p] = sgn * (2 * PI * kz / g.Lz);
        Sx[p] = lds + ((seg * NP + p) * 3 + 0) * RP;
        Sy[p] = lds + ((seg * NP + p) * 3 + 1) * RP;
        Sz[p] = lds + ((seg * NP + p) * 3 + 2) * RP;
    });
    WV<K> P[NP], v[NP];
    {
        WV<K> f[NP], t[NP];
        each([&](int p) { t[p] = wrow_load<K, W, LP>(Sy[p], c); });
        wdiff_n<K, W, NP>(t, c, f);
        each([&](int p) {
            const WV<K> X = wrow_load<K, W, LP>(Sx[p], c), Z = wrow_load<K, W, LP>(Sz[p], c);
            for (int k = 0; k < K; ++k) {
                f[p].e[k] -= ax[p] * X.e[k] + az[p] * Z.e[k];
                f[p].o[k] -= ax[p] * X.o[k] + az[p] * Z.o[k];
            }
        });
        const Op op(coef, Ny, 0, fo, kappa2, c);
        op.template solve<NP>(f, c, P);
    }
    const Op vop(coef, Ny, 3, fo, lambda, c);  // velocity operator: v, then u and w
    {
        WV<K> f[NP], t[NP];
        wdiff_n<K, W, NP>(P, c, f);
        each([&](int p) {
            t[p] = wrow_load<K, W, LP>(Sy[p], c);
            for (int k = 0; k < K; ++k) {
                f[p].e[k] -= t[p].e[k];
                f[p].o[k] -= t[p].o[k];
            }
        });
        vop.template solve<NP>(f, c, v);
        // influence-matrix correction (tausolver.cpp:178-191)
        double dvb[NP], dva[NP];
        wdiff_n<K, W, NP>(v, c, f);
        wends_n<K, W, NP>(f, c, dvb, dva);
        const gcdouble sc = gmem(s.scal) + 6L * m;
        double dplus[NP], dminus[NP];
        each([&](int p) {
            dplus[p] = -sc[0] * dvb[p] - sc[1] * dva[p];
            dminus[p] = -sc[2] * dvb[p] - sc[3] * dva[p];
        });
        // P- and v- are the mirrors of P+ and v+: (e, -o) and (-e, o)
        const WV<K> Pp = wfac<K, W>(coef, Ny, 6, fo, c), vp = wfac<K, W>(coef, Ny, 7, fo, c);
        each([&](int p) {
            for (int k = 0; k < K; ++k) {
                P[p].e[k] += dplus[p] * Pp.e[k] + dminus[p] * Pp.e[k];
                P[p].o[k] += dplus[p] * Pp.o[k] - dminus[p] * Pp.o[k];
                v[p].e[k] += dplus[p] * vp.e[k] - dminus[p] * vp.e[k];
                v[p].o[k] += dplus[p] * vp.o[k] + dminus[p] * vp.o[k];
            }
        });
        if (taucorr) {
            const int Nb = c.Nb;
            const WV<K> P0 = wfac<K, W>(coef, Ny, 8, fo, c), v0 = wfac<K, W>(coef, Ny, 9, fo, c);
            each([&](int p) {
                const double sigma1_Nb = lambda * wtop<K, W>(v[p], c) - Sy[p][pos(Nb)];
                double sigma1_Nb1 = lambda * wtop1<K, W>(v[p], c) - Sy[p][pos(Nb - 1)];
                sigma1_Nb1 += (4.0 / c.L) * Nb * wtop<K, W>(P[p], c);
                const double sigmaNb = sigma1_Nb / (1.0 - sc[5]);
                const double sigmaNb1 = sigma1_Nb1 / (1.0 - sc[4]);
                for (int k = 0; k < K; ++k) {
                    P[p].e[k] += sigmaNb1 * P0.e[k];
                    P[p].o[k] += sigmaNb * P0.o[k];
                    v[p].e[k] += sigmaNb * v0.e[k];
                    v[p].o[k] += sigmaNb1 * v0.o[k];
                }
            });
        }
    }
    each([&](int p) { wrow_store<K, W, LP>(Sy[p], c, v[p]); });  // the rows are this segment's alone
    // u and w, one parity at a time (fewer live registers)
    auto solve_uw = [&](double (WV<K>::*const Pk)[K], int par, int M) {
        double f[2 * NP][K], x[2 * NP][K];
        const HelmPar<K, W> op = vop.part(par, M, c);
        each([&](int p) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int n = pos(2 * min(K * c.lane + k, M - 1) + par);
                f[2 * p][k] = ax[p] * (P[p].*Pk)[k] - Sx[p][n];
                f[2 * p + 1][k] = az[p] * (P[p].*Pk)[k] - Sz[p][n];
            }
        });
        op.template solve<2 * NP>(f, hbl + LP * c.lane + par, HP, c, x);
        each([&](int p) {
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int i = K * c.lane + k, at = wrow_own<K, LP>(c.lane, i, k) + par;
                if (i < M) {
                    Sx[p][at] = x[2 * p][k];
                    Sz[p][at] = x[2 * p + 1][k];
                }
            }
        });
    };
    __builtin_amdgcn_sched_barrier(0);
    solve_uw(&WV<K>::e, 0, c.Me);
    __builtin_amdgcn_sched_barrier(0);
    solve_uw(&WV<K>::o, 1, c.Mo);
    __syncthreads();
    const int ww = threadIdx.x % MPB, mm = m0 + ww;
    const bool out = mm > 0 && mm < g.M;
    for (int row = threadIdx.x / MPB; row < 3 * Ny; row += nthr / MPB) {
        const double a = lds[slot(ww, 0, row)], b = lds[slot(ww, 1, row)];
        const bool mid = row >= Ny && row < 2 * Ny;
        if (out) u[(long)row * g.M + mm] = mid ? dvec2{a, b} : dvec2{b, a};
    }
    __syncthreads();
    each([&](int p) { wrow_store<K, W, LP>(Sy[p], c, P[p]); });
    __syncthreads();
    for (int row = Ny + threadIdx.x / MPB; row < 2 * Ny; row += nthr / MPB) {
        const double a = lds[slot(ww, 0, row)], b = lds[slot(ww, 1, row)];
        if (out) q[(long)(row - Ny) * g.M + mm] = dvec2{a, b};
    }
}

// PressureSolver::solve (poissonsolver.cpp:326-431) per mode, after the
// nonlinear term f of u + U: p'' - kappa^2 p = -div f with p = 0 at the walls,
// solved with the pressure factors of the tau data (the same Helmholtz operator,
// nu = 1), then for every mode but (0,0) the wall correction
// g = c exp(-mu (y-a)) + d exp(mu (y-b)), mu^2 = kappa^2, that makes
// dp/dy = nu v'' at y = a, b; g's coefficients are Ti times its values at the
// Chebyshev points.
template <int K, int W, int MPB>
__global__ void __launch_bounds__(W * MPB) k_pressure_wave(Geom g, YMats ym, PressArgs pa, const double* __restrict__ hb) {
    extern __shared__ double2 lds[];  // [MPB][4][Ny]: f0, f1, f2, v; then the B rows [3][Ny]
    const int Ny = g.Ny;
    double* hbl = reinterpret_cast<double*>(lds + 4 * Ny * MPB);
    for (int i = threadIdx.x; i < 3 * Ny; i += W * MPB) hbl[i] = hb[i];
    const long M = g.M;
    const int m0 = blockIdx.x * MPB, w = threadIdx.x / W;
    const long m = m0 + w;
    const bool valid = m < M;
    const double2* __restrict__ f = reinterpret_cast<const double2*>(pa.f);
    const double2* __restrict__ u = reinterpret_cast<const double2*>(pa.u);
    double2* __restrict__ q = reinterpret_cast<double2*>(pa.q);
    for (int idx = threadIdx.x; idx < 4 * Ny * MPB; idx += W * MPB) {
        const int ww = idx % MPB, rest = idx / MPB, n = rest % Ny, comp = rest / Ny;
        const long mm = m0 + ww;
        double2 v = make_double2(0.0, 0.0);
        if (mm < M) v = comp < 3 ? f[((long)comp * Ny + n) * M + mm] : u[((long)Ny + n) * M + mm];
        lds[(ww * 4 + comp) * Ny + n] = v;
    }
    __syncthreads();
    WCtx c;
    c.N = Ny;
    c.Me = (Ny + 1) / 2;
    c.Mo = (Ny - 1) / 2;
    c.Nb = Ny - 1;
    c.Nc = Ny - 1;
    c.lane = threadIdx.x % W;
    c.L = g.b - g.a;
    c.hb = hbl;
    if (valid) {
        const int ikx = (int)(m % g.nkx), ikz = (int)(m / g.nkx);
        const int kx = kx_of(g, ikx), kz = ikz;
        const bool zero = (kx == 0 && kz == 0);
        const double pi2 = PI * PI;
        const double kappa2 = 4 * pi2 * ((kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz));
        const double ax = 2 * PI * kx / g.Lx, az = 2 * PI * kz / g.Lz;
        const double* cm = pa.set.coef + m * TAU_NA * Ny;
        WV<K> Fxr, Fxi, Fyr, Fyi, Fzr, Fzi;
        wload_c<K, W>(lds + (w * 4 + 0) * Ny, c, Fxr, Fxi);
        wload_c<K, W>(lds + (w * 4 + 1) * Ny, c, Fyr, Fyi);
        wload_c<K, W>(lds + (w * 4 + 2) * Ny, c, Fzr, Fzi);
        const WV<K> Dr = wdiff<K, W>(Fyr, c), Di = wdiff<K, W>(Fyi, c);
        WV<K> Rr, Ri;  // -div f (diffops.cpp:2488-2516)
        for (int k = 0; k < K; ++k) {
            Rr.e[k] = -((-ax * Fxi.e[k] - az * Fzi.e[k]) + Dr.e[k]);
            Rr.o[k] = -((-ax * Fxi.o[k] - az * Fzi.o[k]) + Dr.o[k]);
            Ri.e[k] = -((ax * Fxr.e[k] + az * Fzr.e[k]) + Di.e[k]);
            Ri.o[k] = -((ax * Fxr.o[k] + az * Fzr.o[k]) + Di.o[k]);
        }
        WV<K> Pr = whelm<K, W>(Rr, cm, cm + Ny, cm + 2L * Ny, kappa2, 0.0, 0.0, c);
        WV<K> Pi = whelm<K, W>(Ri, cm, cm + Ny, cm + 2L * Ny, kappa2, 0.0, 0.0, c);
        if (!zero) {  // dp/dy = nu v'' at the walls (poissonsolver.cpp:356-427)
            WV<K> Vr, Vi;
            wload_c<K, W>(lds + (w * 4 + 3) * Ny, c, Vr, Vi);
            double pbr, par_, pbi, pai, vbr, var_, vbi, vai;
            wends<K, W>(wdiff<K, W>(Pr, c), c, pbr, par_);
            wends<K, W>(wdiff<K, W>(Pi, c), c, pbi, pai);
            wends<K, W>(wdiff<K, W>(wdiff<K, W>(Vr, c), c), c, vbr, var_);
            wends<K, W>(wdiff<K, W>(wdiff<K, W>(Vi, c), c), c, vbi, vai);
            const double alr = pa.nu * var_ - par_, ali = pa.nu * vai - pai;
            const double ber = pa.nu * vbr - pbr, bei = pa.nu * vbi - pbi;
            const double mu = sqrt(kappa2), H = g.b - g.a, e = exp(-mu * H);
            const double delta = mu * (1 - exp(-2 * mu * H));
            const double ccr = (-alr + ber * e) / delta, cci = (-ali + bei * e) / delta;
            const double ddr = (ber - alr * e) / delta, ddi = (bei - ali * e) / delta;
            const double piN = PI / (Ny - 1), rad = (g.b - g.a) / 2, cen = (g.b + g.a) / 2;  // chebypoints
            for (int par = 0; par < 2; ++par)
                for (int k = 0; k < K; ++k) {
                    const int n = 2 * (K * c.lane + k) + par;
                    if (n >= Ny) continue;
                    double sr = 0.0, si = 0.0;
                    for (int j = 0; j < Ny; ++j) {
                        const double y = cen + rad * cos(j * piN);
                        const double e1 = exp(-mu * (y - g.a)), e2 = exp(mu * (y - g.b));
                        const double t = ym.Ti[(long)n * Ny + j];
                        sr += t * (ccr * e1 + ddr * e2);
                        si += t * (cci * e1 + ddi * e2);
                    }
                    if (par == 0) {
                        Pr.e[k] += sr;
                        Pi.e[k] += si;
                    } else {
                        Pr.o[k] += sr;
                        Pi.o[k] += si;
                    }
                }
        }
        wstore_c<K, W>(lds + (w * 4 + 0) * Ny, c, Pr, Pi);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < Ny * MPB; idx += W * MPB) {
        const int ww = idx % MPB, n = idx / MPB;
        const long mm = m0 + ww;
        if (mm < M) q[(long)n * M + mm] = lds[(ww * 4 + 0) * Ny + n];
    }
}

void launch_pressure(const Geom& g, const YMats& ym, const double* hb, const PressArgs& pa, hipStream_t st) {
    const int Me = (g.Ny + 1) / 2;
    auto go = [&](auto kern, int w) {
        const int mpb = 256 / w;
        const dim3 grid((unsigned)((g.M + mpb - 1) / mpb));
        const size_t lds = (size_t)4 * g.Ny * mpb * sizeof(double2) + (size_t)3 * g.Ny * sizeof(double);
        allow_lds(kern, lds);
        kern<<<grid, 256, lds, st>>>(g, ym, pa, hb);
    };
    if (Me <= 16) go(k_pressure_wave<1, 16, 16>, 16);
    else if (Me <= 32) go(k_pressure_wave<1, 32, 8>, 32);
    else if (Me <= 64) go(k_pressure_wave<1, 64, 4>, 64);
    else if (Me <= 128) go(k_pressure_wave<2, 64, 4>, 64);
    else go(k_pressure_wave<3, 64, 4>, 64);
}

void launch_tau_solve(const Geom& g, const double* hb, int n, const TauMember* tab, hipStream_t st) {
    const int Me = (g.Ny + 1) / 2;  // even coefficients: at most K per lane of a W-lane segment
    auto launch = [&](auto kern, int mpb, int threads, size_t lds) {
        const long nblk = ((long)((g.M + mpb - 1) / mpb) + 1) * n;
        if (nblk > 0x7fffffffL) throw std::runtime_error("tau solve: too many blocks in one launch");
        allow_lds(kern, lds);
        kern<<<dim3((unsigned)nblk), threads, lds, st>>>(g, hb, n, tab);
    };
    auto go = [&](auto kern, int k, int w, int mpb) {
        launch(kern, mpb, 2 * w * mpb, tau_lds(tau_pitch(g.Ny), 2 * k, w, mpb));
    };
    // 16-lane segments (every shuffle a DPP row move) as far as their
    // coefficients fit the registers, 32 and 64 lanes above. 8 modes per block: with 16
    // a lone 32^3 field took 12.4 us, not 9.2, 64^3 17.1, not 14.6, and 24 of
    // 32^3 26.7, not 20.8. At 65-80 coefficients, where a block of 8 leaves
    // half-filled 256-byte runs of every row, 16 modes per block are faster once
    // one field fills the chip with them (192x129x192 122.5 -> 120.8 us, 128^3,
    // 224 blocks, 53.3 -> 48.0). The rule looks at the grid alone: a member's
    // result must not depend on which instance its batch runs.
    if (Me <= 16) go(k_tau_solve_wave<1, 16, 8>, 1, 16, 8);
    else if (Me <= 32) go(k_tau_solve_wave<2, 16, 8>, 2, 16, 8);
    else if (Me <= 48) go(k_tau_solve_wave<3, 16, 8>, 3, 16, 8);
    else if (Me <= 64) go(k_tau_solve_wave<4, 16, 8>, 4, 16, 8);
    else if (Me <= 80 && g.M >= 192 * 16) go(k_tau_solve_wave<5, 16, 16>, 5, 16, 16);
    else if (Me <= 80) go(k_tau_solve_wave<5, 16, 8>, 5, 16, 8);
    else if (Me <= 96) go(k_tau_solve_wave<6, 16, 8>, 6, 16, 8);
    else if (Me <= 128) launch(k_tau_solve_tall<4, 32, 4, 1>, 4, 256, tau_lds(tau_row<4>(g.Ny), tau_lp(4), 32, 4));
    else launch(k_tau_solve_tall<3, 64, 4, 2>, 4, 256, tau_lds(tau_row<3>(g.Ny), tau_lp(3), 64, 4));
}

// ===========================================================================
// NSE::linear on live modes (nse.cpp:393-477)
// ===========================================================================
// For each velocity component L = nu (u'' - kappa^2 u) - grad q, plus on kx = kz = 0
// nu U'', nu W'' and the mean pressure gradient (the bulk-velocity branch takes dPdx
// from nu (du/dy(b) - du/dy(a)) / Ly, nse.cpp:437-472). The real parts couple as in
// the tau solve, (v, q real; u, w imaginary) and (v, q imaginary; u, w real), and
// each set runs on its own W-lane segment; MPB modes per block, member blockIdx.y.
//
// What bounds it: for one field the latency of a block, for a batch HBM. The rows of
// a block's modes are staged in LDS with MPB consecutive modes per access; loaded by
// the segments themselves, whose lanes are rows apart, every 8 bytes were a request
// of their own. us per launch, before -> after: one 32^3 field 9.0 -> 5.4, 54x57x72
// 11.5 -> 6.4, 64^3 10.6 -> 7.9, 96^3 16.7 -> 10.3, 128^3 22.9 -> 18.5, 192x129x192
// 57.8 -> 36.7 (177 MB, 4.8 TB/s), 48x193x48 17.0 -> 11.3, 16 of 48^3 16.4 -> 14.3, 16
// of 64^3 39.3 -> 36.0.
template <int K, int W, int MPB>
__global__ void __launch_bounds__(2 * W * MPB) k_linear_wave(Geom g, const LinearMember* __restrict__ tab) {
    extern __shared__ double2 lds2[];
    double* const lds = reinterpret_cast<double*>(lds2);  // [mode][part][u v w q] of tau_pitch(Ny)
    constexpr int nthr = 2 * W * MPB, step = nthr / MPB, UNR = 8;
    const LinearMember& me = tab[blockIdx.y];
    const double nu = me.nu;
    const LinearConst lc = me.c;
    const int Ny = g.Ny, RP = tau_pitch(Ny), nrow = 4 * Ny;
    const int m0 = blockIdx.x * MPB;
    const int ww = threadIdx.x % MPB, mm = m0 + ww;
    // part 0 takes v.re, q.re, u.im, w.im; part 1 v.im, q.im, u.re, w.re
    auto slot = [&](int pt, int comp, int n) { return ((ww * 2 + pt) * 4 + comp) * RP + n; };
    auto comp_of = [&](int row) { return (row >= Ny) + (row >= 2 * Ny) + (row >= 3 * Ny); };
    {
        const auto u = gmem(reinterpret_cast<const dvec2*>(me.u));
        const auto q = gmem(reinterpret_cast<const dvec2*>(me.q));
        const int mc = min(mm, g.M - 1);  // slots past the last mode repeat it
        for (int row = threadIdx.x / MPB; row < nrow; row += UNR * step) {
            dvec2 v[UNR];
#pragma unroll
            for (int r = 0; r < UNR; ++r) {
                const int rr = min(row + r * step, nrow - 1);
                v[r] = rr < 3 * Ny ? u[(long)rr * g.M + mc] : q[(long)(rr - 3 * Ny) * g.M + mc];
            }
#pragma unroll
            for (int r = 0; r < UNR; ++r) {
                const int rr = row + r * step, comp = comp_of(rr), n = rr - comp * Ny;
                if (rr >= nrow) continue;
                const bool odd = comp & 1;  // v, q
                lds[slot(0, comp, n)] = odd ? v[r].x : v[r].y;
                lds[slot(1, comp, n)] = odd ? v[r].y : v[r].x;
            }
        }
    }
    const int seg = threadIdx.x / W;
    for (int i = threadIdx.x; i < 2 * MPB * 4; i += nthr) lds[i * RP + Ny] = 0.0;  // the rows' padding
    __syncthreads();
    {
        WCtx c;
        c.N = Ny;
        c.Me = (Ny + 1) / 2;
        c.Mo = (Ny - 1) / 2;
        c.Nb = Ny - 1;
        c.Nc = Ny - 1;
        c.lane = threadIdx.x % W;
        c.L = g.b - g.a;
        c.hb = nullptr;
        const int m = min(m0 + (seg >> 1), g.M - 1), part = seg & 1;
        const int ikx = m % g.nkx, kz = m / g.nkx, kx = kx_of(g, ikx);
        const bool mean = kx == 0 && kz == 0 && part == 1;  // the mean flow's real parts
        const double kappa2 = 4 * PI * PI * ((kx / g.Lx) * (kx / g.Lx) + (kz / g.Lz) * (kz / g.Lz));
        const double sgn = part ? 1.0 : -1.0;
        double* const R = lds + seg * 4 * RP;
        const WV<K> Pq = wrow_load<K, W>(R + 3 * RP, c);
        WV<K> s0[3], s1[3], s2[3];
#pragma unroll
        for (int comp = 0; comp < 3; ++comp) {
            s0[comp] = wrow_load<K, W>(R + comp * RP, c);
#pragma unroll
            for (int k = 0; k < K; ++k) {
                s0[comp].e[k] *= nu;
                s0[comp].o[k] *= nu;
            }
        }
        wdiff_n<K, W, 3>(s0, c, s1);
        double dPd[3] = {0.0, 0.0, 0.0};
        if (mean && lc.bulk) {
            double eb[3], ea[3];
            wends_n<K, W, 3>(s1, c, eb, ea);
            for (int comp = 0; comp < 3; comp += 2) dPd[comp] = (eb[comp] - ea[comp]) / c.L;
        }
        wdiff_n<K, W, 3>(s1, c, s2);  // nu u''
        WV<K> p1[1] = {Pq}, dq[1];
        wdiff_n<K, W, 1>(p1, c, dq);
#pragma unroll
        for (int comp = 0; comp < 3; ++comp) {
            // dq/dy; i k q: the real part of u meets -k q.im, the imaginary part k q.re
            const double d = sgn * (comp == 0 ? 2 * PI * kx / g.Lx : 2 * PI * kz / g.Lz);
            WV<K> o;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                o.e[k] = s2[comp].e[k] - kappa2 * s0[comp].e[k];
                o.o[k] = s2[comp].o[k] - kappa2 * s0[comp].o[k];
                o.e[k] += comp == 1 ? -dq[0].e[k] : d * Pq.e[k];
                o.o[k] += comp == 1 ? -dq[0].o[k] : d * Pq.o[k];
            }
            if (mean && comp != 1) {
                const WV<K> base = wload<K, W>(gmem(comp == 0 ? lc.nuUbaseyy : lc.nuWbaseyy), c);
                for (int k = 0; k < K; ++k) {
                    o.e[k] += base.e[k];
                    o.o[k] += base.o[k];
                }
                if (c.lane == 0) {
                    if (!lc.bulk) o.e[0] -= comp == 0 ? lc.dPdxRef : lc.dPdzRef;
                    else o.e[0] -= dPd[comp] + (comp == 0 ? lc.nuUbase_slope : lc.nuWbase_slope);
                }
            }
            wrow_store<K, W>(R + comp * RP, c, o);  // the rows are this segment's alone
        }
    }
    __syncthreads();
    if (mm >= g.M) return;
    const auto out = gmem_w(reinterpret_cast<dvec2*>(me.out));
    for (int row = threadIdx.x / MPB; row < 3 * Ny; row += step) {
        const int comp = comp_of(row), n = row - comp * Ny;
        const double a = lds[slot(0, comp, n)], b = lds[slot(1, comp, n)];
        out[(long)row * g.M + mm] = comp == 1 ? dvec2{a, b} : dvec2{b, a};
    }
}

void launch_linear(const Geom& g, int n, const LinearMember* tab, hipStream_t st) {
    const int Me = (g.Ny + 1) / 2;
    auto go = [&](auto kern, int w, int mpb) {
        const size_t lds = (size_t)mpb * 8 * tau_pitch(g.Ny) * sizeof(double);
        allow_lds(kern, lds);
        kern<<<dim3((g.M + mpb - 1) / mpb, n), 2 * w * mpb, lds, st>>>(g, tab);
    };
    // 16-lane segments and 8 modes per block as far as in the tau solve; above, 4 modes
    // keep a block within 100 KB of LDS, at 64-byte pieces of a row (at 65 coefficients,
    // 32 lanes and 4 modes against 16 and 8: 128^3 26.3 -> 18.5 us, 192x129x192 54 -> 37).
    // At 81-96 coefficients 8 modes on 16 lanes are the faster ones where one field fills
    // the chip with their blocks (128x161x128 30.7 us, 32.7 with 4 modes; 32x161x32 10.8
    // against 9.2, 24 of them 43.4 against 40.7).
    if (Me <= 16) go(k_linear_wave<1, 16, 8>, 16, 8);
    else if (Me <= 32) go(k_linear_wave<2, 16, 8>, 16, 8);
    else if (Me <= 48) go(k_linear_wave<3, 16, 8>, 16, 8);
    else if (Me <= 64) go(k_linear_wave<4, 16, 8>, 16, 8);
    else if (Me <= 80) go(k_linear_wave<5, 16, 8>, 16, 8);
    else if (Me <= 96 && g.M >= 192 * 16) go(k_linear_wave<6, 16, 8>, 16, 8);
    else if (Me <= 96) go(k_linear_wave<3, 32, 4>, 32, 4);
    else if (Me <= 128) go(k_linear_wave<4, 32, 4>, 32, 4);
    else if (Me <= 192) go(k_linear_wave<6, 32, 4>, 32, 4);
    else throw std::runtime_error("NSE::linear: Ny above 383 is not supported");
}

}  // namespace cfg
