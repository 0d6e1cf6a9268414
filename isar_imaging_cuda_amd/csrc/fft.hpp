// fft.hpp — the device FFT: transforms of 64 ... 16384 points held in registers, exchanged through
// LDS between passes.
//
// A transform of length N is computed by T = N / E threads, each holding E elements in
// registers. A pass with radix R processes N / R butterflies; thread t owns butterflies
// j = t + b T, b < E / R, and holds x[j + r N / R] for r < R on entry. After the last pass the
// thread holds the outputs at the same positions j + r N / R_last, so the first-pass load and
// the last-pass store are both unit-stride across threads (coalesced against global memory).
// Between passes the data goes through a padded LDS buffer (self-sorting passes, Stockham). Lengths
// 2^k take radices 16 and one of 2, 4, 8 with 16 elements per thread, lengths 3 * 2^k radices 4, 6
// and 12 with 12.
//
// From 192 points on the first and last radix are equal, so a transform ends in the layout it
// started from and the next one can follow without an exchange. The two-pass lengths 64 and 128
// cannot have that; REV = true runs their radices in reverse order, from the output layout of the
// plain order back to its input layout.
//
// Bound by FP32 vector issue (autofocus, chirp-z) a pass is arranged for few instructions. Input r
// of a butterfly carries the twiddle w^r, w = exp(j theta): the outputs are the polynomial
// sum_r x_r z^r at z = w exp(j 2 pi q / R), evaluated by halving (even and odd part, z -> z^2).
// Every step is a +- z b for one of a few z, kept as z = c (1 + j t), t = tan: two fused
// multiply-adds form (1 + j t) b and four add c times it to +-a, six instructions where a rotation
// and two sums take eight, and no separate twiddle products (radix 16: 192 instructions instead of
// 168 for the butterfly, 60 for the twiddles and up to 52 to form their powers; E. N. Linzer and E. Feig,
// "Implementation of efficient FFT algorithms on fused multiply-add architectures", 1993). c and t are each
// rounded once from FP64 (fft_table); the rounding of (1 + j t) b is relative to that sum,
// which c brings back to the size of b, so a large t costs no accuracy, only range (fft_overflowed). 512, 4096 and 16384 points
// are 0.95, 1.15 and 1.26e-7 off the FP64 transform (relative, random data; 4096 points with products
// of rounded twiddles 1.97e-7). A 512-point transform with its 2-point pass takes 388 vector
// instructions instead of 700, and what is bound by their issue is that much faster: the autofocus
// of 40 frames of 512 pulses 2.7 instead of 4.3 ms.
#pragma once

namespace isar {

// ------------------------------------------------------------------------------------------
// Twiddle constants: z = c (1 + j t), c = cos, t = tan of an angle. An angle of exactly pi / 2
// takes c = 2^-30, t = 2^30, which is off by 1e-9.
// ------------------------------------------------------------------------------------------
struct FftCT {
    float c, t;
};
// n of them for one pass of one thread
template <int n>
struct FftCTs {
    FftCT v[n > 0 ? n : 1];
};

namespace fft_table {
// sin and cos of pi x for 0 <= x <= 1/4 by their Taylor series (terms below 1e-19 left out)
constexpr double sin_pi(double x) {
    const double a = 3.14159265358979323846 * x, a2 = a * a;
    double term = a, sum = 0.0;
    for (int k = 1; k < 24; k += 2) {
        sum += term;
        term *= -a2 / ((k + 1) * (k + 2));
    }
    return sum;
}
constexpr double cos_pi(double x) {
    const double a = 3.14159265358979323846 * x, a2 = a * a;
    double term = 1.0, sum = 0.0;
    for (int k = 0; k < 24; k += 2) {
        sum += term;
        term *= -a2 / ((k + 1) * (k + 2));
    }
    return sum;
}
// c and t of the angle 2 pi k / d, given sin and cos on the first eighth of the circle
template <typename Octant>
constexpr FftCT ct(int k, int d, const Octant& oct) {
    const int q = (8 * (k % d)) / d;   // octant
    const int e = d / 4, r = k % d;
    double c = 0.0, s = 0.0;
    switch (q) {
    case 0: c = oct.c[r]; s = oct.s[r]; break;
    case 1: c = oct.s[e - r]; s = oct.c[e - r]; break;
    case 2: c = -oct.s[r - e]; s = oct.c[r - e]; break;
    case 3: c = -oct.c[2 * e - r]; s = oct.s[2 * e - r]; break;
    case 4: c = -oct.c[r - 2 * e]; s = -oct.s[r - 2 * e]; break;
    case 5: c = -oct.s[3 * e - r]; s = -oct.c[3 * e - r]; break;
    case 6: c = oct.s[r - 3 * e]; s = -oct.c[r - 3 * e]; break;
    default: c = oct.c[4 * e - r]; s = -oct.s[4 * e - r]; break;
    }
    constexpr double tiny = 1.0 / 1073741824.0;
    if (c < tiny && c > -tiny) c = tiny;
    // t from the rounded c, so that c t is the sine
    const float cf = static_cast<float>(c);
    return FftCT{cf, static_cast<float>(s / static_cast<double>(cf))};
}
template <int D>
struct Octant {
    double c[D / 8 + 1], s[D / 8 + 1];
    constexpr Octant() : c(), s() {
        for (int k = 0; k <= D / 8; ++k) {
            c[k] = cos_pi(2.0 * k / D);
            s[k] = sin_pi(2.0 * k / D);
        }
    }
};
// Row k: the constants of a radix-16 pass whose inputs carry w^r, w = exp(j theta), theta = 2 pi k / 16384:
// 8 theta; 4 theta; 2 theta + {0, pi/4}; theta + {0, pi/8, pi/4, 3 pi/8}.
struct Pow2 {
    FftCT row[1024][8];
    constexpr Pow2() : row() {
        constexpr int d = 16384;
        const Octant<d> oct;
        for (int k = 0; k < 1024; ++k) {
            row[k][0] = ct(8 * k, d, oct);
            row[k][1] = ct(4 * k, d, oct);
            row[k][2] = ct(2 * k, d, oct);
            row[k][3] = ct(2 * k + d / 8, d, oct);
            for (int i = 0; i < 4; ++i) row[k][4 + i] = ct(k + i * (d / 16), d, oct);
        }
    }
};
struct ThreePow2 {   // entry k: the angle 2 pi k / 768
    FftCT at[768];
    constexpr ThreePow2() : at() {
        const Octant<768> oct;
        for (int k = 0; k < 768; ++k) at[k] = ct(k, 768, oct);
    }
};
}  // namespace fft_table

alignas(64) static __device__ constexpr fft_table::Pow2 kFftPow2{};
alignas(64) static __device__ constexpr fft_table::ThreePow2 kFftThreePow2{};

// ------------------------------------------------------------------------------------------
// Butterflies. DIR = -1 forward (exp(-j ...)), +1 inverse.
// ------------------------------------------------------------------------------------------
// y0, y1 = a +- w b, w = c (1 + DIR j t) (DIR j)^jp
template <int DIR>
__device__ __forceinline__ void fft_butterfly(float2 a, float2 b, FftCT w, int jp, float2& y0, float2& y1) {
    const float t = DIR < 0 ? -w.t : w.t;
    const float u = fmaf(-t, b.y, b.x), v = fmaf(t, b.x, b.y);
    const float p = jp ? (DIR < 0 ? v : -v) : u, q = jp ? (DIR < 0 ? -u : u) : v;
    y0 = make_float2(fmaf(w.c, p, a.x), fmaf(w.c, q, a.y));
    y1 = make_float2(fmaf(-w.c, p, a.x), fmaf(-w.c, q, a.y));
}
// y0, y1 = a +- (DIR j)^jp b
template <int DIR>
__device__ __forceinline__ void fft_butterfly_unit(float2 a, float2 b, int jp, float2& y0, float2& y1) {
    const float2 r = jp ? cmul_i<DIR>(b) : b;
    y0 = cadd(a, r);
    y1 = csub(a, r);
}
// y0, y1 = a +- exp(DIR j pi / 4) (DIR j)^jp b
template <int DIR>
__device__ __forceinline__ void fft_butterfly_eighth(float2 a, float2 b, int jp, float2& y0, float2& y1) {
    constexpr float h = 0.70710678118654752440f;
    const float u = DIR < 0 ? b.x + b.y : b.x - b.y, v = DIR < 0 ? b.y - b.x : b.y + b.x;
    const float p = jp ? (DIR < 0 ? v : -v) : u, q = jp ? (DIR < 0 ? -u : u) : v;
    y0 = make_float2(fmaf(h, p, a.x), fmaf(h, q, a.y));
    y1 = make_float2(fmaf(-h, p, a.x), fmaf(-h, q, a.y));
}

// DFT of the L values x[S i] (i < L = 2^k), natural order, no twiddles. HALF: the values of the whole
// transform's upper half are zero and not read.
template <int L, int S, int DIR, bool HALF = false>
__device__ __forceinline__ void dft_unit(const float2* x, float2 (&y)[L]) {
    if constexpr (L == 1) {
        y[0] = x[0];
    } else if constexpr (L == 2 && HALF) {
        y[0] = y[1] = x[0];
    } else {
        float2 e[L / 2], o[L / 2];
        dft_unit<L / 2, 2 * S, DIR, HALF>(x, e);
        dft_unit<L / 2, 2 * S, DIR, HALF>(x + S, o);
#pragma unroll
        for (int q = 0; q < L / 2; ++q) {
            const int quarter = L >= 4 ? L / 4 : 1, i = L >= 4 ? q % quarter : 0, jp = L >= 4 ? q / quarter : 0;
            if (i == 0) fft_butterfly_unit<DIR>(e[q], o[q], jp, y[q], y[q + L / 2]);
            else if (8 * i == L) fft_butterfly_eighth<DIR>(e[q], o[q], jp, y[q], y[q + L / 2]);
            else
                fft_butterfly<DIR>(e[q], o[q],
                                   i == 1 ? FftCT{0.92387953251128675613f, 0.41421356237309504880f}
                                          : FftCT{0.38268343236508977173f, 2.41421356237309504880f},
                                   jp, y[q], y[q + L / 2]);
        }
    }
}

// sum_r x[S r] z^r at z = w exp(DIR j 2 pi q / L), q < L: the DFT of L values with twiddles w^r, w = exp(DIR j theta).
// ct: a row of fft_table::Pow2 for the angle theta L / 16, of which entries 0 ... L / 2 - 1 are used.
template <int L, int S, int DIR, int n>
__device__ __forceinline__ void dft_twiddled(const float2* x, const FftCTs<n>& ct, float2 (&y)[L]) {
    if constexpr (L == 1) {
        y[0] = x[0];
    } else {
        constexpr int entry = L / 4, quarter = L >= 4 ? L / 4 : 1;   // entries per quarter turn
        float2 e[L / 2], o[L / 2];
        dft_twiddled<L / 2, 2 * S, DIR>(x, ct, e);
        dft_twiddled<L / 2, 2 * S, DIR>(x + S, ct, o);
#pragma unroll
        for (int q = 0; q < L / 2; ++q)
            fft_butterfly<DIR>(e[q], o[q], ct.v[entry + q % quarter], q / quarter, y[q], y[q + L / 2]);
    }
}

// The same for group b of the B = 16 / R groups that a thread holds in the last pass of a length of
// B T points or fewer, whose twiddle base is w exp(DIR j 2 pi b / 16): sum_r x[S r] z^r (r < L) at
// z = (w exp(DIR j 2 pi (b + q B) / 16))^(R / L). ct: entries FIRST ... 7 of the row of w.
template <int L, int S, int R, int DIR, int FIRST, int n>
__device__ __forceinline__ void dft_twiddled_group(const float2* x, const FftCTs<n>& ct, int b, float2 (&y)[L]) {
    if constexpr (L == 1) {
        y[0] = x[0];
    } else {
        constexpr int B = 16 / R, m = R / L;
        constexpr int entry = (m == 4 ? 1 : m == 2 ? 2 : 4) - FIRST;
        constexpr int quarter = 4 / m;
        float2 e[L / 2], o[L / 2];
        dft_twiddled_group<L / 2, 2 * S, R, DIR, FIRST>(x, ct, b, e);
        dft_twiddled_group<L / 2, 2 * S, R, DIR, FIRST>(x + S, ct, b, o);
#pragma unroll
        for (int q = 0; q < L / 2; ++q) {
            const int i = b + q * B;
            fft_butterfly<DIR>(e[q], o[q], ct.v[entry + i % quarter], i / quarter, y[q], y[q + L / 2]);
        }
    }
}

// x <- the DFT of its 16 values with twiddles w^r (row: the constants of w).
template <int DIR>
__device__ __forceinline__ void dft16_twiddled(float2 (&x)[16], const FftCTs<8>& row) {
    float2 y[16];
    dft_twiddled<16, 1, DIR>(x, row, y);
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = y[e];
}

template <int DIR>
__device__ __forceinline__ void dft3(float2& a0, float2& a1, float2& a2) {
    constexpr float h = 0.86602540378443864676f;   // sqrt(3)/2
    const float2 t = cadd(a1, a2), d = csub(a1, a2);
    const float2 m = make_float2(fmaf(-0.5f, t.x, a0.x), fmaf(-0.5f, t.y, a0.y));
    const float2 r = cmul_i<DIR>(d);
    a0 = cadd(a0, t);
    a1 = make_float2(fmaf(h, r.x, m.x), fmaf(h, r.y, m.y));
    a2 = make_float2(fmaf(-h, r.x, m.x), fmaf(-h, r.y, m.y));
}
// DFT of R = 3 P values (P = 2 or 4) by the prime-factor mapping: n = 3 n1 + P n2 (mod R) in, k = k1 mod P and
// k2 mod 3 out, P-point and 3-point transforms with no twiddles between them.
template <int R, int DIR>
__device__ __forceinline__ void dft_3p(float2 (&x)[R]) {
    constexpr int P = R / 3;
    float2 a[P][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
        float2 in[P], out[P];
#pragma unroll
        for (int n1 = 0; n1 < P; ++n1) in[n1] = x[(3 * n1 + P * n2) % R];
        dft_unit<P, 1, DIR>(in, out);
#pragma unroll
        for (int k1 = 0; k1 < P; ++k1) a[k1][n2] = out[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) dft3<DIR>(a[k1][0], a[k1][1], a[k1][2]);
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = a[k % P][k % 3];
}

// ------------------------------------------------------------------------------------------
// Plans
// ------------------------------------------------------------------------------------------
// Radix sequence per transform length for E elements per thread.
template <int N, int E>
struct FftPlan;

// E = 16 plans
template <> struct FftPlan<16384, 16> { static constexpr int NP = 4; static constexpr int R[4] = {16, 16, 4, 16}; };
template <> struct FftPlan<8192, 16>  { static constexpr int NP = 4; static constexpr int R[4] = {16, 16, 2, 16}; };
template <> struct FftPlan<4096, 16>  { static constexpr int NP = 3; static constexpr int R[3] = {16, 16, 16}; };
template <> struct FftPlan<2048, 16>  { static constexpr int NP = 3; static constexpr int R[3] = {16, 8, 16}; };
template <> struct FftPlan<1024, 16>  { static constexpr int NP = 3; static constexpr int R[3] = {16, 4, 16}; };
template <> struct FftPlan<512, 16>   { static constexpr int NP = 3; static constexpr int R[3] = {16, 2, 16}; };
template <> struct FftPlan<256, 16>   { static constexpr int NP = 2; static constexpr int R[2] = {16, 16}; };
template <> struct FftPlan<128, 16>   { static constexpr int NP = 2; static constexpr int R[2] = {16, 8}; };
template <> struct FftPlan<64, 16>    { static constexpr int NP = 2; static constexpr int R[2] = {16, 4}; };
// E = 12 plans (3 * 2^k lengths)
template <> struct FftPlan<192, 12>   { static constexpr int NP = 3; static constexpr int R[3] = {4, 12, 4}; };
template <> struct FftPlan<384, 12>   { static constexpr int NP = 4; static constexpr int R[4] = {4, 6, 4, 4}; };
template <> struct FftPlan<768, 12>   { static constexpr int NP = 4; static constexpr int R[4] = {4, 12, 4, 4}; };

// a sequence with equal first and last radix keeps its layout and always runs in the plain order
template <int N, int E, bool REV>
inline constexpr bool kFftReversed = REV && FftPlan<N, E>::R[0] != FftPlan<N, E>::R[FftPlan<N, E>::NP - 1];

template <int N, int E, bool REV>
struct FftOrder {
    using Plan = FftPlan<N, E>;
    static constexpr int NP = Plan::NP;
    static constexpr int T = N / E;
    static constexpr int radix(int p) { return Plan::R[kFftReversed<N, E, REV> ? NP - 1 - p : p]; }
    static constexpr int stride(int p) { return p == 0 ? 1 : stride(p - 1) * radix(p - 1); }
    // all groups of a thread share one twiddle base
    static constexpr bool shared(int p) { return radix(p) == E || T % stride(p) == 0; }
    // twiddle constants of pass p per thread: E = 16 takes entries 0 ... R / 2 - 1 of a row of Pow2 where the
    // groups share their base and entries first(p) ... 7 where they do not (the last pass of 64 and
    // 128 points), E = 12 the angles of w^r (radix 6, 12) or of w^2 and w per group (radix 4)
    static constexpr int first(int p) { return radix(p) == 8 ? 1 : 2; }
    static constexpr int count(int p) {
        if (p == 0 || p >= NP) return 0;
        if (E == 16) return shared(p) ? radix(p) / 2 : 8 - first(p);
        const int per_group = radix(p) == 4 ? 2 : radix(p) - 1;
        return per_group * (shared(p) ? 1 : E / radix(p));
    }
};

// Element position held in register slot e before and after a transform: the thread's index plus an offset
// that depends on the slot alone.
template <int N, int E, int R>
__host__ __device__ constexpr int fft_slot_offset(int e) {
    return (e / R) * (N / E) + (e % R) * (N / R);
}
template <int N, int E, bool REV = false>
__host__ __device__ constexpr int fft_in_offset(int e) {
    return fft_slot_offset<N, E, FftOrder<N, E, REV>::radix(0)>(e);
}
template <int N, int E, bool REV = false>
__host__ __device__ constexpr int fft_out_offset(int e) {
    using O = FftOrder<N, E, REV>;
    return fft_slot_offset<N, E, O::radix(O::NP - 1)>(e);
}
template <int N, int E, bool REV = false>
__device__ __forceinline__ int fft_in_pos(int tid, int e) { return tid + fft_in_offset<N, E, REV>(e); }
template <int N, int E, bool REV = false>
__device__ __forceinline__ int fft_out_pos(int tid, int e) { return tid + fft_out_offset<N, E, REV>(e); }

// The constants of pass P for thread tid.
template <int N, int E, bool REV, int P>
__device__ __forceinline__ FftCTs<FftOrder<N, E, REV>::count(P)> fft_constants(int tid) {
    using O = FftOrder<N, E, REV>;
    FftCTs<O::count(P)> ct;
    if constexpr (P > 0 && P < O::NP) {
        constexpr int R = O::radix(P), Ns = O::stride(P);
        if constexpr (E == 16) {
            // groups of one base w = exp(j 2 pi k / (Ns R)), k = tid mod Ns, or the last pass with
            // w exp(j 2 pi b / 16), w = exp(j 2 pi tid / N), as the base of group b
            static_assert(O::shared(P) || ((R == 4 || R == 8) && Ns * R == N), "bases of a pass's groups");
            const FftCT* row = O::shared(P) ? kFftPow2.row[(tid % Ns) * (1024 / Ns)] : kFftPow2.row[tid * (16384 / N)] + O::first(P);
#pragma unroll
            for (int i = 0; i < O::count(P); ++i) ct.v[i] = row[i];
        } else {
            constexpr int B = E / R, T = O::T, unit = 768 / (Ns * R);
#pragma unroll
            for (int b = 0; b < (O::shared(P) ? 1 : B); ++b) {
                const int k = ((tid + b * T) % Ns) * unit;
                if constexpr (R == 4) {
                    ct.v[2 * b] = kFftThreePow2.at[2 * k];
                    ct.v[2 * b + 1] = kFftThreePow2.at[k];
                } else {
#pragma unroll
                    for (int r = 1; r < R; ++r) ct.v[r - 1] = kFftThreePow2.at[(k * r) % 768];
                }
            }
        }
    }
    return ct;
}

// Twiddle constants of every pass of a transform for one thread, kept in registers.
template <int N, int E, bool REV = false>
struct FftTwiddles {
    using O = FftOrder<N, E, REV>;
    FftCTs<O::count(1)> p1;
    FftCTs<O::count(2)> p2;
    FftCTs<O::count(3)> p3;
    template <int P>
    __device__ __forceinline__ const auto& pass(int) const {
        if constexpr (P == 1) return p1;
        else if constexpr (P == 2) return p2;
        else return p3;
    }
};
template <int N, int E, bool REV = false>
__device__ __forceinline__ FftTwiddles<N, E, kFftReversed<N, E, REV>> fft_twiddles(int tid) {
    constexpr bool V = kFftReversed<N, E, REV>;
    return {fft_constants<N, E, V, 1>(tid), fft_constants<N, E, V, 2>(tid), fft_constants<N, E, V, 3>(tid)};
}

// The same with the constants of the second pass (stride 16) in LDS: it needs only 16 rows (tid mod 16),
// kFft16Row apart so that the 16-byte reads of 16 lanes hit different banks. For kernels whose
// registers are needed elsewhere. Constants read from memory at each use instead would wait for the
// kernel's earlier stores too (one in-order counter): 7.5 instead of 6.2 ms for the level-0
// kernel at 1024 frames of 256 x 4096.
constexpr int kFft16Row = 10;   // FftCT per row: 8 and a pad of 16 bytes
constexpr int kFft16Bytes = 16 * kFft16Row * static_cast<int>(sizeof(FftCT));
template <int N, int E>
struct FftTwiddlesLds {
    using O = FftOrder<N, E, false>;
    static_assert(O::NP >= 3 && O::stride(1) == 16, "the second of three or four passes has stride 16");
    const FftCT* rows;
    FftCTs<O::count(2)> p2;
    FftCTs<O::count(3)> p3;
    template <int P>
    __device__ __forceinline__ decltype(auto) pass(int tid) const {
        if constexpr (P == 1) {
            const FftCT* row = rows + (opaque(tid) & 15) * kFft16Row;
            FftCTs<O::count(1)> ct;
#pragma unroll
            for (int i = 0; i < O::count(1); ++i) ct.v[i] = row[i];
            return ct;
        } else if constexpr (P == 2) {
            return (p2);
        } else {
            return (p3);
        }
    }
};
// Every thread of the workgroup calls it; `rows`: kFft16Bytes of LDS, 16-byte aligned. The first
// transform's first barrier orders the copy before any use.
template <int N, int E>
__device__ __forceinline__ FftTwiddlesLds<N, E> fft_twiddles_lds(int tid, FftCT* rows) {
    // without a branch, so that the kernel's other loads are not held back: with more than 128 threads some
    // entries are written twice, with the same value
#pragma unroll
    for (int i = 0; i < 128; i += N / E) {
        const int k = (tid + i) & 127;
        rows[(k >> 3) * kFft16Row + (k & 7)] = kFftPow2.row[(k >> 3) * 64][k & 7];
    }
    return {rows, fft_constants<N, E, false, 2>(tid), fft_constants<N, E, false, 3>(tid)};
}

// ------------------------------------------------------------------------------------------
// Passes
// ------------------------------------------------------------------------------------------
// Orders the LDS accesses of an FFT's passes. WAVE = false: a workgroup barrier. WAVE = true: the
// transform lives in one wave, whose LDS instructions the hardware performs in issue order, so
// only the compiler has to be kept from moving accesses across (a wavefront-scope fence needs no
// wait and no barrier instruction).
template <bool WAVE>
__device__ __forceinline__ void fft_sync() {
#ifdef ISAR_EMU
    __syncthreads();   // every thread of the block calls the transform together
#else
    if constexpr (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
#endif
}

// LDS layout of a transform: a padding slot every 32 elements (256 bytes, the width of the LDS), so that with the
// passes' strides only the 8-byte stores of stride 16 meet a bank twice (with one every 16 elements
// every load did). Up to 1024 points one every 16 elements measured better all the same (autofocus of
// 40 frames of 512 pulses 2.70 instead of 2.93 ms); up to 256 points several transforms share 32
// lanes, and their buffers are N/E (mod 32) apart for N/E lanes each.
__host__ __device__ constexpr int lds_pad_every(int n) { return n <= 1024 ? 16 : 32; }
__host__ __device__ constexpr int lds_padded_size(int n) {
    return n == 192 ? 208 : n + n / lds_pad_every(n) + (n > 256 ? 1 : 0);
}
template <int N>
__host__ __device__ constexpr int lds_pad(int i) { return i + i / lds_pad_every(N); }
// For a constant off, lds_pad(i + off) = lds_pad(i) + lds_pad(off), so that an access is a base address
// and an immediate offset, where no carry crosses a pad: off a multiple of the padding distance, or
// off a multiple of m and i below m modulo that distance, m a power of two up to it.
template <int N>
__host__ __device__ constexpr bool lds_pad_aligned(int n) {
    return n % lds_pad_every(N) == 0 || lds_pad_every(N) % n == 0;
}

template <int N, int E, int R, int Ns>
__device__ __forceinline__ void stockham_store(const float2 (&x)[E], float2* lds, int tid) {
    constexpr int T = N / E;
    constexpr int B = E / R;
    // element r of group j goes to (j / Ns) Ns R + j mod Ns + r Ns
    constexpr int P = lds_pad_every(N);
    constexpr bool kLinear = Ns % P == 0 || (P % Ns == 0 && lds_pad_aligned<N>(Ns * R));
    constexpr bool kOneBase = kLinear && T % Ns == 0 && (T * R) % P == 0;   // group b lies b T R further on
    auto at_group = [&](int b) {
        const int j = tid + b * T;
        return (j / Ns) * Ns * R + j % Ns;
    };
    float2* const base = lds + lds_pad<N>(at_group(0));
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (kOneBase) base[lds_pad<N>(b * T * R) + lds_pad<N>(r * Ns)] = x[b * R + r];
            else if constexpr (kLinear) (lds + lds_pad<N>(at_group(b)))[lds_pad<N>(r * Ns)] = x[b * R + r];
            else lds[lds_pad<N>(at_group(b) + r * Ns)] = x[b * R + r];
        }
    }
}

template <int N, int E, int R>
__device__ __forceinline__ void stockham_load(float2 (&x)[E], const float2* lds, int tid) {
    constexpr int T = N / E, S = N / R, P = lds_pad_every(N);   // inputs S apart, groups below S
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int b = e / R, r = e % R;
        if constexpr (S % P == 0 && T % P == 0) x[e] = (lds + lds_pad<N>(tid))[lds_pad<N>(b * T + r * S)];
        else if constexpr (lds_pad_aligned<N>(S)) x[e] = (lds + lds_pad<N>(tid + b * T))[lds_pad<N>(r * S)];
        else x[e] = lds[lds_pad<N>(tid + b * T + r * S)];
    }
}

// The butterflies of pass P on a thread's registers.
template <int N, int E, int DIR, int P, bool REV, typename TW>
__device__ __forceinline__ void fft_compute(float2 (&x)[E], int tid, const TW& tw) {
    using O = FftOrder<N, E, REV>;
    constexpr int R = O::radix(P), B = E / R;
    if constexpr (P == 0) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            float2 y[R];
            dft_unit<R, 1, DIR>(x + b * R, y);
#pragma unroll
            for (int r = 0; r < R; ++r) x[b * R + r] = y[r];
        }
    } else {
        const auto& ct = tw.template pass<P>(tid);
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if constexpr (E == 16) {
                float2 y[R];
                if constexpr (O::shared(P)) dft_twiddled<R, 1, DIR>(x + b * R, ct, y);
                else dft_twiddled_group<R, 1, R, DIR, O::first(P)>(x + b * R, ct, b, y);
#pragma unroll
                for (int r = 0; r < R; ++r) x[b * R + r] = y[r];
            } else if constexpr (R == 4) {
                const FftCT w2 = ct.v[O::shared(P) ? 0 : 2 * b], w1 = ct.v[O::shared(P) ? 1 : 2 * b + 1];
                float2 e0, e1, o0, o1;
                fft_butterfly<DIR>(x[b * 4], x[b * 4 + 2], w2, 0, e0, e1);
                fft_butterfly<DIR>(x[b * 4 + 1], x[b * 4 + 3], w2, 0, o0, o1);
                fft_butterfly<DIR>(e0, o0, w1, 0, x[b * 4], x[b * 4 + 2]);
                fft_butterfly<DIR>(e1, o1, w1, 1, x[b * 4 + 1], x[b * 4 + 3]);
            } else {
                static_assert(R % 3 == 0 && O::shared(P), "radix 6 or 12 with one twiddle base per thread");
                float2 v[R];
                v[0] = x[b * R];
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    const float2 a = x[b * R + r];
                    const float t = DIR < 0 ? -ct.v[r - 1].t : ct.v[r - 1].t;
                    v[r] = make_float2(ct.v[r - 1].c * fmaf(-t, a.y, a.x), ct.v[r - 1].c * fmaf(t, a.x, a.y));
                }
                dft_3p<R, DIR>(v);
#pragma unroll
                for (int r = 0; r < R; ++r) x[b * R + r] = v[r];
            }
        }
    }
}

template <int N, int E, int DIR, int P, bool WAVE, bool REV, typename TW>
struct FftPasses {
    using O = FftOrder<N, E, REV>;
    // passes P ... NP - 1; x holds the layout of pass P on entry
    __device__ __forceinline__ static void run(float2 (&x)[E], float2* lds, int tid, const TW& tw) {
        fft_compute<N, E, DIR, P, REV>(x, tid, tw);
        after(x, lds, tid, tw);
    }
    // the exchange after the butterflies of pass P and the passes that follow
    __device__ __forceinline__ static void after(float2 (&x)[E], float2* lds, int tid, const TW& tw) {
        static_assert(!WAVE || (N / E <= 64 && 64 % (N / E) == 0), "a wave-ordered transform must lie in one wave");
        if constexpr (P + 1 < O::NP) {
            stockham_store<N, E, O::radix(P), O::stride(P)>(x, lds, tid);
            fft_sync<WAVE>();
            stockham_load<N, E, O::radix(P + 1)>(x, lds, tid);
            fft_sync<WAVE>();
            FftPasses<N, E, DIR, P + 1, WAVE, REV, TW>::run(x, lds, tid, tw);
        }
    }
};

// In-register/LDS transform. On entry x[e] = in[fft_in_pos<N, E, REV>(tid, e)], on exit
// x[e] = out[fft_out_pos<N, E, REV>(tid, e)]. lds must hold lds_padded_size(N) float2 for this
// transform. All threads of the workgroup must call the transform together (it uses
// __syncthreads). With WAVE = true the passes are ordered by fft_sync<true> instead: for
// transforms of at most 64 threads, aligned within a wave, that touch only their own LDS buffer
// (N/E <= 64 and 64 % (N/E) == 0); the caller orders other waves' accesses to that buffer with
// barriers of its own.
template <int N, int E, int DIR, bool WAVE = false, bool REV = false, typename TW>
__device__ __forceinline__ void fft(float2 (&x)[E], float2* lds, int tid, const TW& tw) {
    FftPasses<N, E, DIR, 0, WAVE, REV, TW>::run(x, lds, tid, tw);
}
// The factor t of a butterfly is up to 2^30, so that values whose transform FP32 holds can overflow on the
// way, from about 2^83 on at 16384 points. A kernel that takes any input does a transform over on
// kFftLarge times its values where the workgroup's results are not all finite (which an overflow
// always leaves so), and divides the results by it. Every thread of the workgroup calls it.
constexpr float kFftLarge = 0x1p-60f;
template <int E>
__device__ __forceinline__ bool fft_overflowed(const float2 (&x)[E]) {
    float m = 0.0f;   // not finite if any value is not
#pragma unroll
    for (int e = 0; e < E; ++e) m = fmaf(x[e].x, 0.0f, fmaf(x[e].y, 0.0f, m));
    return __syncthreads_or(!(m == 0.0f));
}
// A kernel's only transform: the constants are loaded ahead of its first pass.
template <int N, int E, int DIR, bool WAVE = false, bool REV = false>
__device__ __forceinline__ void fft(float2 (&x)[E], float2* lds, int tid) {
    const auto tw = fft_twiddles<N, E, REV>(tid);
    fft<N, E, DIR, WAVE, REV>(x, lds, tid, tw);
}
// The same transform with its first pass done by the caller.
template <int N, int E, int DIR, bool WAVE = false, typename TW>
__device__ __forceinline__ void fft_after_first(float2 (&x)[E], float2* lds, int tid, const TW& tw) {
    FftPasses<N, E, DIR, 0, WAVE, false, TW>::after(x, lds, tid, tw);
}
// A transform whose input is zero from N / 2 on (x[8 ... 15], not read; first radix 16).
template <int N, int DIR, bool WAVE = false>
__device__ __forceinline__ void fft_zero_half(float2 (&x)[16], float2* lds, int tid) {
    static_assert(FftPlan<N, 16>::R[0] == 16, "slots 8 ... 15 hold the upper half");
    const auto tw = fft_twiddles<N, 16>(tid);
    float2 y[16];
    dft_unit<16, 1, DIR, true>(x, y);
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = y[e];
    fft_after_first<N, 16, DIR, WAVE>(x, lds, tid, tw);
}

}  // namespace isar
