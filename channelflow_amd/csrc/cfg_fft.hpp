// FFTs (FP64): LDS Stockham FFTs of a block's lines, and FFTs of lines held in
// the registers of a wavefront.
#pragma once

#include "cfg_dev.hpp"

namespace cfg {

// LDS layout of FFT lines: element i of a line sits at pidx(i) = i + i/8 (one
// pad slot per 8 complex values spreads the power-of-two strides of the
// Stockham passes over distinct banks), and consecutive lines are lpitch(N) =
// N + N/8 + 1 slots apart (odd, so walks across lines are conflict-free too).
__host__ __device__ constexpr int pidx(int i) { return i + (i >> 3); }
__host__ __device__ constexpr int lpitch(int N) { return N + N / 8 + 1; }

// ---------------------------------------------------------------------------
// LDS Stockham FFTs over nlines contiguous lines of length N. sign -1 forward
// (exp(-i...)), +1 backward; unnormalised. tw is the table exp(-2 pi i j/N),
// j < N, staged in LDS. The result lands in a or b (returned). All threads of
// the block must call them.
// ---------------------------------------------------------------------------
template <int R, int SIGN>
__device__ __forceinline__ void dft_small(double2 (&v)[4]) {
    double2 o[4];
    if constexpr (R == 2) {
        o[0] = cadd(v[0], v[1]);
        o[1] = csub(v[0], v[1]);
    } else if constexpr (R == 4) {
        const double2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const double2 s13 = cadd(v[1], v[3]), d13 = csub(v[1], v[3]);
        const double2 jd = (SIGN < 0) ? make_double2(d13.y, -d13.x) : make_double2(-d13.y, d13.x);
        o[0] = cadd(s02, s13);
        o[1] = cadd(d02, jd);
        o[2] = csub(s02, s13);
        o[3] = csub(d02, jd);
    } else {
        const double s3 = (SIGN < 0) ? -0.86602540378443864676 : 0.86602540378443864676;
        const double2 s12 = cadd(v[1], v[2]), d12 = csub(v[1], v[2]);
        const double2 m = make_double2(v[0].x - 0.5 * s12.x, v[0].y - 0.5 * s12.y);
        o[0] = cadd(v[0], s12);
        o[1] = make_double2(fma(-s3, d12.y, m.x), fma(s3, d12.x, m.y));  // m + q, q = i s3 d12
        o[2] = make_double2(fma(s3, d12.y, m.x), fma(-s3, d12.x, m.y));  // m - q
    }
    for (int r = 0; r < R; ++r) v[r] = o[r];
}

// radix 8, decimation in frequency: sums and differences of v_k, v_{k+4}, the
// differences turned by w^k (w = exp(SIGN 2 pi i/8)), then two radix-4 DFTs
// give the even and the odd outputs. The 1/sqrt(2) of w and w^3 is applied in
// the odd radix-4's first sums, as fused multiply-adds: with p1 = w b1 sqrt2
// and p3 = w^3 b3 sqrt2, b1 + b3 = h (p1 + p3) and b1 - b3 = h (p1 - p3).
template <int R, int SIGN>
__device__ __forceinline__ void dft_small(double2 (&v)[8]) {
    static_assert(R == 8, "radix-8 overload");
    constexpr double h = 0.70710678118654752440;  // 1/sqrt(2)
    double2 a[4], b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a[k] = cadd(v[k], v[k + 4]);
        b[k] = csub(v[k], v[k + 4]);
    }
    double2 p1, p3;
    if constexpr (SIGN < 0) {  // w = (1 - i)/sqrt2, w^2 = -i, w^3 = -(1 + i)/sqrt2
        p1 = make_double2(b[1].x + b[1].y, b[1].y - b[1].x);
        p3 = make_double2(b[3].y - b[3].x, -(b[3].x + b[3].y));
        b[2] = make_double2(b[2].y, -b[2].x);
    } else {  // w = (1 + i)/sqrt2, w^2 = i, w^3 = (-1 + i)/sqrt2
        p1 = make_double2(b[1].x - b[1].y, b[1].x + b[1].y);
        p3 = make_double2(-(b[3].x + b[3].y), b[3].x - b[3].y);
        b[2] = make_double2(-b[2].y, b[2].x);
    }
    dft_small<4, SIGN>(a);
    // radix 4 of (b0, h p1, b2, h p3), as in dft_small<4>
    const double2 s02 = cadd(b[0], b[2]), d02 = csub(b[0], b[2]);
    const double2 s13 = cadd(p1, p3), d13 = csub(p1, p3);                                // over h
    const double2 jd = (SIGN < 0) ? make_double2(d13.y, -d13.x) : make_double2(-d13.y, d13.x);  // over h
    b[0] = make_double2(fma(h, s13.x, s02.x), fma(h, s13.y, s02.y));
    b[1] = make_double2(fma(h, jd.x, d02.x), fma(h, jd.y, d02.y));
    b[2] = make_double2(fma(-h, s13.x, s02.x), fma(-h, s13.y, s02.y));
    b[3] = make_double2(fma(-h, jd.x, d02.x), fma(-h, jd.y, d02.y));
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        v[2 * m] = a[m];
        v[2 * m + 1] = b[m];
    }
}

template <int R, int SIGN>
__device__ __forceinline__ void stockham_bfly(const double2* __restrict__ s, double2* __restrict__ d, const double2* tw,
                                              int j, int k, int NR, int NS, int tstep) {
    double2 v[4];
    for (int r = 0; r < R; ++r) v[r] = s[pidx(j + r * NR)];
    if (k != 0) {
        for (int r = 1; r < R; ++r) {
            double2 t = tw[r * k * tstep];
            if (SIGN > 0) t.y = -t.y;
            v[r] = cmul(v[r], t);
        }
    }
    dft_small<R, SIGN>(v);
    const int o = (j / NS) * NS * R + k;
    for (int r = 0; r < R; ++r) d[pidx(o + r * NS)] = v[r];
}

template <int SIGN>
__device__ double2* fft_lds(double2* a, double2* b, const FFTPlan& P, const double2* tw, int nlines) {
    double2* src = a;
    double2* dst = b;
    const int N = P.N;
    int Ns = 1;
    for (int p = 0; p < P.npass; ++p) {
        const int R = P.radix[p];
        const int NR = N / R;
        const int tstep = N / (Ns * R);
        for (int w = threadIdx.x; w < nlines * NR; w += blockDim.x) {
            const int line = w / NR;
            const int j = w - line * NR;
            const int k = j % Ns;
            const int lo = line * lpitch(N);
            if (R == 4) stockham_bfly<4, SIGN>(src + lo, dst + lo, tw, j, k, NR, Ns, tstep);
            else if (R == 2) stockham_bfly<2, SIGN>(src + lo, dst + lo, tw, j, k, NR, Ns, tstep);
            else stockham_bfly<3, SIGN>(src + lo, dst + lo, tw, j, k, NR, Ns, tstep);
        }
        __syncthreads();
        double2* t = src;
        src = dst;
        dst = t;
        Ns *= R;
    }
    return src;
}

// stage the twiddle table of P into LDS
__device__ __forceinline__ void stage_tw(double2* dst, const FFTPlan& P) {
    for (int i = threadIdx.x; i < P.N; i += blockDim.x) dst[i] = P.tw[i];
}

// ---- wave-local FFTs ---------------------------------------------------------
// A z-line of length N = N1 N2 lives on G lanes of one wavefront (G the power
// of two >= N1, N2; 64/G lines per wavefront), in one of two layouts:
//   spectral: lane j < N1 holds Z[j + N1 r], r < N2;
//   physical: lane j < N2 holds x[j + N2 m], m < N1.
// The inverse transform is an N2-point DFT in registers, the twiddles
// w_N^(j k1), a transpose through the line's own LDS rows and an N1-point DFT
// in registers; the forward transform runs the same steps the other way. All
// fields of a line share the physical layout, so the products are lane-local,
// and a wavefront never waits for another one.
// Lengths 2^a 3^b. Those between the powers of two run here as well: against
// the LDS FFTs, whose every pass ends in a block barrier and whose runtime plan
// divides by its strides, a 54x57x72 field (divergence form) takes 11.9 us for
// its z pass, not 36.2, 4.8 and 6.3 us for its inverse and forward x-FFTs, not
// 8.6 and 11.9; 16 members of 48x59x18 step 2.2x as fast, of 48x53x36 2.3x.
template <int NZ>
struct ZWShape {
    static constexpr int N1 = 0, N2 = 0;
};
template <> struct ZWShape<16> { static constexpr int N1 = 4, N2 = 4; };
template <> struct ZWShape<18> { static constexpr int N1 = 3, N2 = 6; };
template <> struct ZWShape<24> { static constexpr int N1 = 4, N2 = 6; };
template <> struct ZWShape<32> { static constexpr int N1 = 4, N2 = 8; };
template <> struct ZWShape<36> { static constexpr int N1 = 6, N2 = 6; };
template <> struct ZWShape<48> { static constexpr int N1 = 6, N2 = 8; };
template <> struct ZWShape<54> { static constexpr int N1 = 6, N2 = 9; };
template <> struct ZWShape<64> { static constexpr int N1 = 8, N2 = 8; };
template <> struct ZWShape<72> { static constexpr int N1 = 6, N2 = 12; };
template <> struct ZWShape<96> { static constexpr int N1 = 8, N2 = 12; };
template <> struct ZWShape<108> { static constexpr int N1 = 9, N2 = 12; };
template <> struct ZWShape<128> { static constexpr int N1 = 8, N2 = 16; };
template <> struct ZWShape<144> { static constexpr int N1 = 9, N2 = 16; };
template <> struct ZWShape<162> { static constexpr int N1 = 9, N2 = 18; };
template <> struct ZWShape<192> { static constexpr int N1 = 12, N2 = 16; };
template <> struct ZWShape<256> { static constexpr int N1 = 16, N2 = 16; };

constexpr int pow2_at_least(int n) {
    int p = 1;
    while (p < n) p *= 2;
    return p;
}

// A line of N values on G lanes of a wavefront, 64/G lines per wavefront:
//   spectral layout  lane s < SL holds Z[s + SL r], r < SV;
//   physical layout  lane p < PL holds x[p + PL m], m < PV.
template <int NZ>
struct ZW {
    static constexpr int N1 = ZWShape<NZ>::N1, N2 = ZWShape<NZ>::N2, N = N1 * N2;
    static constexpr int SL = N1, SV = N2, PL = N2, PV = N1;
    static constexpr int NMAX = N1 > N2 ? N1 : N2;
    static constexpr int G = pow2_at_least(NMAX);  // lanes per line
    static constexpr int LPW = 64 / G;             // lines per wavefront
    static constexpr int LBUF = N + NMAX;          // LDS slots per line (transposes, padded rows)
    static constexpr int TWN = N;                  // twiddles: w_N^i
    static __device__ __forceinline__ int tw_power(int i) { return i; }
};

// The same in three steps, N = A B C with the physical values A per lane: two
// transposes, but fewer values per lane and transform. QG: groups of B values a
// lane holds in the middle step. P1, P2: LDS pitches of the transposes, [C][B A] and
// [A][B C]. The middle step's lanes run over C first, so that every access is
// contiguous or at the odd pitch P1 across lanes; P2 keeps the A-groups of a
// 16-lane read on different banks. With rows of A or B values instead, lanes a row
// apart, conflicts took a quarter of the rotational 192-bin z pass (9.4 M cycles, now
// 2.0 M). us per launch, before -> after: 192x129x192 rotational 63 -> 57, 128^3
// convection 48 -> 44, rotational 31.4 -> 30.6, skew-symmetric 64x49x108 19.5 -> 17.9,
// 64x49x144 21.8 -> 20.4, 64x33x256 24.5 -> 20.9; at 72 and 96 the same.
template <int NZ>
struct ZW3Shape {
    static constexpr int A = 0, B = 0, C = 0, QG = 1, P1 = 1, P2 = 1;
};
template <> struct ZW3Shape<72> { static constexpr int A = 3, B = 4, C = 6, QG = 1, P1 = 13, P2 = 30; };
template <> struct ZW3Shape<96> { static constexpr int A = 3, B = 4, C = 8, QG = 1, P1 = 13, P2 = 40; };
template <> struct ZW3Shape<108> { static constexpr int A = 6, B = 3, C = 6, QG = 2, P1 = 19, P2 = 22; };
template <> struct ZW3Shape<128> { static constexpr int A = 4, B = 4, C = 8, QG = 1, P1 = 17, P2 = 40; };
template <> struct ZW3Shape<144> { static constexpr int A = 6, B = 4, C = 6, QG = 2, P1 = 25, P2 = 30; };
template <> struct ZW3Shape<162> { static constexpr int A = 6, B = 3, C = 9, QG = 3, P1 = 19, P2 = 41; };
template <> struct ZW3Shape<192> { static constexpr int A = 6, B = 4, C = 8, QG = 2, P1 = 25, P2 = 40; };
template <> struct ZW3Shape<256> { static constexpr int A = 8, B = 4, C = 8, QG = 2, P1 = 33, P2 = 40; };

template <int NZ>
struct ZW3 {
    static constexpr int A = ZW3Shape<NZ>::A, B = ZW3Shape<NZ>::B, C = ZW3Shape<NZ>::C, QG = ZW3Shape<NZ>::QG;
    static constexpr int P1 = ZW3Shape<NZ>::P1, P2 = ZW3Shape<NZ>::P2, PT = C | 1;
    static constexpr int N = A * B * C;
    static constexpr int SL = A * B, SV = C, PL = B * C, PV = A, QL = A * C / QG;
    static constexpr int G = pow2_at_least(PL > SL ? PL : SL);
    static constexpr int LPW = 64 / G;
    static constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }
    static constexpr int LBUF = max3(C * P1, A * P2, N);
    // twiddles: w_N^(j k) at j P2 + k (j < A, k < PL), then w_PL^(b m) at b PT + m (b < B, m < C)
    static constexpr int TWN = A * P2 + B * PT;
    static_assert(QL <= G && A % QG == 0 && P1 >= SL && P2 >= PL, "the middle step's lanes and the pitches");
    // entry i as a power of w_N
    static __device__ __forceinline__ int tw_power(int i) {
        if (i < A * P2) return i / P2 * (i % P2 < PL ? i % P2 : 0);
        i -= A * P2;
        return A * (i / PT) * (i % PT < C ? i % PT : 0);
    }
};

// the lengths with a wavefront FFT
#define CFG_FFT_SIZES(X) \
    X(16) X(18) X(24) X(32) X(36) X(48) X(54) X(64) X(72) X(96) X(108) X(128) X(144) X(162) X(192) X(256)
constexpr bool zwave_size(int n) {
#define CFG_IS_SIZE(N) || n == N
    return false CFG_FFT_SIZES(CFG_IS_SIZE);
#undef CFG_IS_SIZE
}

// Orders the LDS accesses of one wavefront (its lanes read what other lanes of
// the same wavefront wrote): a compiler barrier between wavefront-scope fences.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- DFTs held in registers: sum_n v_n exp(SIGN 2 pi i n k / R) ----
template <int R, int SIGN>
__device__ __forceinline__ void dft_reg(double2 (&v)[R]);

constexpr int inv_mod(int a, int m) {
    for (int x = 1; x < m; ++x)
        if ((a * x) % m == 1) return x;
    return 1;
}

// prime-factor (Good-Thomas) DFT of length A B with gcd(A, B) = 1: input
// n = (B a + A b) mod AB, output k with k = ka (mod A), k = kb (mod B); no twiddles
template <int A, int B, int SIGN>
__device__ __forceinline__ void dft_pfa(double2 (&v)[A * B]) {
    constexpr int R = A * B, BI = inv_mod(B, A), AI = inv_mod(A, B);
    double2 t[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        double2 s[A];
#pragma unroll
        for (int a = 0; a < A; ++a) s[a] = v[(B * a + A * b) % R];
        dft_reg<A, SIGN>(s);
#pragma unroll
        for (int a = 0; a < A; ++a) t[b][a] = s[a];
    }
#pragma unroll
    for (int ka = 0; ka < A; ++ka) {
        double2 s[B];
#pragma unroll
        for (int b = 0; b < B; ++b) s[b] = t[b][ka];
        dft_reg<B, SIGN>(s);
#pragma unroll
        for (int kb = 0; kb < B; ++kb) v[(B * BI * ka + A * AI * kb) % R] = s[kb];
    }
}

// exp(i m pi / 8), m <= 9, from cos(pi/8), sin(pi/8) and 1/sqrt(2)
__device__ __forceinline__ constexpr double2 w16(int m) {
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, h = 0.70710678118654752440;
    return m == 1 ? double2{c1, s1} : m == 2 ? double2{h, h} : m == 3 ? double2{s1, c1} : m == 4 ? double2{0.0, 1.0}
         : m == 5 ? double2{-s1, c1} : m == 6 ? double2{-h, h} : m == 7 ? double2{-c1, s1} : m == 8 ? double2{-1.0, 0.0}
         : m == 9 ? double2{-c1, -s1} : double2{1.0, 0.0};
}

// length 16 as 4 x 4 (Cooley-Tukey, twiddles exp(SIGN 2 pi i n2 k1 / 16))
template <int SIGN>
__device__ __forceinline__ void dft_ct44(double2 (&v)[16]) {
    double2 t[4][4];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        double2 s[4];
#pragma unroll
        for (int n1 = 0; n1 < 4; ++n1) s[n1] = v[4 * n1 + n2];
        dft_small<4, SIGN>(s);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            if (n2 * k1 == 0) {
                t[n2][k1] = s[k1];
            } else {
                double2 w = w16(n2 * k1);
                if (SIGN < 0) w.y = -w.y;
                t[n2][k1] = cmul(s[k1], w);
            }
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        double2 s[4];
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) s[n2] = t[n2][k1];
        dft_small<4, SIGN>(s);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = s[k2];
    }
}

// exp(2 pi i m / 9), m = 1, 2, 4
__device__ __forceinline__ constexpr double2 w9(int m) {
    return m == 1 ? double2{0.76604444311897803520, 0.64278760968653932632}
         : m == 2 ? double2{0.17364817766693034885, 0.98480775301220805937}
                  : double2{-0.93969262078590838405, 0.34202014332566873304};
}

// length 9 as 3 x 3 (Cooley-Tukey, twiddles exp(SIGN 2 pi i n2 k1 / 9))
template <int SIGN>
__device__ __forceinline__ void dft_ct33(double2 (&v)[9]) {
    double2 t[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
        double2 s[3];
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1) s[n1] = v[3 * n1 + n2];
        dft_reg<3, SIGN>(s);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            if (n2 * k1 == 0) {
                t[n2][k1] = s[k1];
            } else {
                double2 w = w9(n2 * k1);
                if (SIGN < 0) w.y = -w.y;
                t[n2][k1] = cmul(s[k1], w);
            }
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        double2 s[3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) s[n2] = t[n2][k1];
        dft_reg<3, SIGN>(s);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = s[k2];
    }
}

template <int R, int SIGN>
__device__ __forceinline__ void dft_reg(double2 (&v)[R]) {
    if constexpr (R == 2 || R == 3 || R == 4) {
        double2 t[4];
#pragma unroll
        for (int i = 0; i < R; ++i) t[i] = v[i];
        dft_small<R, SIGN>(t);
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = t[i];
    } else if constexpr (R == 8) {
        dft_small<8, SIGN>(v);
    } else if constexpr (R == 6) {
        dft_pfa<2, 3, SIGN>(v);
    } else if constexpr (R == 9) {
        dft_ct33<SIGN>(v);
    } else if constexpr (R == 18) {
        dft_pfa<2, 9, SIGN>(v);
    } else if constexpr (R == 12) {
        dft_pfa<4, 3, SIGN>(v);
    } else if constexpr (R == 16) {
        dft_ct44<SIGN>(v);
    } else {
        static_assert(R == 0, "no register DFT of this length");
    }
}

// DFT (sign SIGN) of a line held in layout A, v[r] = Z[j + N1 r] on lane
// j < N1, into layout B, u[m] = X[j + N2 m] on lane j < N2:
// X[k1 + N2 k2] = sum_j w_N1^(j k2) w_N^(j k1) sum_r Z[j + N1 r] w_N2^(r k1).
template <int N, int SIGN>
__device__ __forceinline__ void zw_a2b(double2 (&v)[ZW<N>::N2], double2 (&u)[ZW<N>::N1], int j, double2* T,
                                       const double2* tw) {
    constexpr int N1 = ZW<N>::N1, N2 = ZW<N>::N2;
    dft_reg<N2, SIGN>(v);
    const int jt = j < N1 ? j : N1 - 1;
#pragma unroll
    for (int k1 = 1; k1 < N2; ++k1) {
        double2 t = tw[jt * k1];
        if (SIGN > 0) t.y = -t.y;
        v[k1] = cmul(v[k1], t);
    }
    wave_lds_sync();
    if (j < N1) {
#pragma unroll
        for (int k1 = 0; k1 < N2; ++k1) T[k1 * (N1 + 1) + j] = v[k1];
    }
    wave_lds_sync();
    const int row = j < N2 ? j : N2 - 1;
#pragma unroll
    for (int i = 0; i < N1; ++i) u[i] = T[row * (N1 + 1) + i];
    dft_reg<N1, SIGN>(u);
}

// the same from layout B, u[m] = x[j + N2 m] on lane j < N2, into layout A,
// v[p] = X[j + N1 p] on lane j < N1
template <int N, int SIGN>
__device__ __forceinline__ void zw_b2a(double2 (&u)[ZW<N>::N1], double2 (&v)[ZW<N>::N2], int j, double2* T,
                                       const double2* tw) {
    constexpr int N1 = ZW<N>::N1, N2 = ZW<N>::N2;
    dft_reg<N1, SIGN>(u);
    const int jt = j < N2 ? j : N2 - 1;
#pragma unroll
    for (int q = 1; q < N1; ++q) {
        double2 t = tw[jt * q];
        if (SIGN > 0) t.y = -t.y;
        u[q] = cmul(u[q], t);
    }
    wave_lds_sync();
    if (j < N2) {
#pragma unroll
        for (int q = 0; q < N1; ++q) T[q * (N2 + 1) + j] = u[q];
    }
    wave_lds_sync();
    const int row = j < N1 ? j : N1 - 1;
#pragma unroll
    for (int i = 0; i < N2; ++i) v[i] = T[row * (N2 + 1) + i];
    dft_reg<N2, SIGN>(v);
}

// The three-step transforms, between the same layouts. With n = s + SL c,
// s = j + A b (j < A, b < B, c < C) and k = k1 + PL k2, k1 = m1 + C m2:
// X[k] = sum_j w_A^(j k2) w_N^(j k1) sum_b w_B^(b m2) w_PL^(b m1) sum_c Z w_C^(c m1).
template <int NZ, int SIGN>
__device__ __forceinline__ void zw3_s2p(double2 (&v)[ZW3<NZ>::SV], double2 (&u)[ZW3<NZ>::PV], int l, double2* T,
                                        const double2* tw) {
    using S = ZW3<NZ>;
    constexpr int A = S::A, B = S::B, C = S::C, P1 = S::P1, P2 = S::P2;
    auto turn = [&](double2 x, int i) {
        double2 t = tw[i];
        if (SIGN > 0) t.y = -t.y;
        return cmul(x, t);
    };
    asm volatile("" : "+v"(l));  // addresses formed anew in each transform, not held between them
    dft_reg<C, SIGN>(v);
    const int b = (l < S::SL ? l : S::SL - 1) / A;
    wave_lds_sync();
    if (l < S::SL) {
        T[l] = v[0];
#pragma unroll
        for (int m1 = 1; m1 < C; ++m1) T[m1 * P1 + l] = turn(v[m1], A * P2 + b * S::PT + m1);
    }
    wave_lds_sync();
    double2 w[S::QG][B];
    const int q = l < S::QL ? l : S::QL - 1, j0 = q / C, m1 = q - j0 * C;
#pragma unroll
    for (int g = 0; g < S::QG; ++g) {
#pragma unroll
        for (int i = 0; i < B; ++i) w[g][i] = T[m1 * P1 + i * A + j0 + A / S::QG * g];
        dft_reg<B, SIGN>(w[g]);
    }
    wave_lds_sync();
    if (l < S::QL) {
#pragma unroll
        for (int g = 0; g < S::QG; ++g) {
            const int at = (j0 + A / S::QG * g) * P2 + m1;
#pragma unroll
            for (int m2 = 0; m2 < B; ++m2) T[at + C * m2] = turn(w[g][m2], at + C * m2);
        }
    }
    wave_lds_sync();
    const int p = l < S::PL ? l : S::PL - 1;
#pragma unroll
    for (int i = 0; i < A; ++i) u[i] = T[i * P2 + p];
    dft_reg<A, SIGN>(u);
}

template <int NZ, int SIGN>
__device__ __forceinline__ void zw3_p2s(double2 (&u)[ZW3<NZ>::PV], double2 (&v)[ZW3<NZ>::SV], int l, double2* T,
                                        const double2* tw) {
    using S = ZW3<NZ>;
    constexpr int A = S::A, B = S::B, C = S::C, P1 = S::P1, P2 = S::P2;
    auto turn = [&](double2 x, int i) {
        double2 t = tw[i];
        if (SIGN > 0) t.y = -t.y;
        return cmul(x, t);
    };
    asm volatile("" : "+v"(l));  // addresses formed anew in each transform, not held between them
    dft_reg<A, SIGN>(u);
    wave_lds_sync();
    if (l < S::PL) {
        T[l] = u[0];
#pragma unroll
        for (int q = 1; q < A; ++q) T[q * P2 + l] = turn(u[q], q * P2 + l);
    }
    wave_lds_sync();
    double2 w[S::QG][B];
    const int q = l < S::QL ? l : S::QL - 1, j0 = q / C, i1 = q - j0 * C;
#pragma unroll
    for (int g = 0; g < S::QG; ++g) {
#pragma unroll
        for (int i = 0; i < B; ++i) w[g][i] = T[(j0 + A / S::QG * g) * P2 + i1 + C * i];
        dft_reg<B, SIGN>(w[g]);
    }
    wave_lds_sync();
    if (l < S::QL) {
#pragma unroll
        for (int g = 0; g < S::QG; ++g) {
            const int at = i1 * P1 + j0 + A / S::QG * g;
            T[at] = w[g][0];
#pragma unroll
            for (int p1 = 1; p1 < B; ++p1) T[at + p1 * A] = turn(w[g][p1], A * P2 + p1 * S::PT + i1);
        }
    }
    wave_lds_sync();
    const int s = l < S::SL ? l : S::SL - 1;
#pragma unroll
    for (int i = 0; i < C; ++i) v[i] = T[i * P1 + s];
    dft_reg<C, SIGN>(v);
}

// spectral -> physical and back by either kind of line
template <class S>
constexpr bool three_step = false;
template <int N>
constexpr bool three_step<ZW3<N>> = true;
template <class S, int SIGN>
__device__ __forceinline__ void line_s2p(double2 (&v)[S::SV], double2 (&u)[S::PV], int l, double2* T, const double2* tw) {
    if constexpr (three_step<S>) zw3_s2p<S::N, SIGN>(v, u, l, T, tw);
    else zw_a2b<S::N, SIGN>(v, u, l, T, tw);
}
template <class S, int SIGN>
__device__ __forceinline__ void line_p2s(double2 (&u)[S::PV], double2 (&v)[S::SV], int l, double2* T, const double2* tw) {
    if constexpr (three_step<S>) zw3_p2s<S::N, SIGN>(u, v, l, T, tw);
    else zw_b2a<S::N, SIGN>(u, v, l, T, tw);
}

}  // namespace cfg
