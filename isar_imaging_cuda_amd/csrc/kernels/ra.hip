// ra.hip — range alignment (range_alignment.cu:4-201) for gfx950.
//
// The reference inverse-transforms all M rows at every merge level and once more at the end.
// Here each row's spectrum S0 (HPC, Hamming window and (-1)^n centring applied) is formed once
// and stored; a row is transformed again only when its cumulative lag changes, by re-reading S0
// and applying its lag ramp on the fly. Group energies sum_{rows} |IFFT(row)|^2 / N^2 are kept per
// group head row and merged level by level, E^{l+1}_g = E^l_{2g} + E~^l_{2g+1} (E~ = the second
// group after its shift). Row m moves for the last time at level floor(log2 m) (it moves at level
// l exactly when bit l of m is set), so its aligned profile is written then, and no final pass
// over all rows is needed.
#include "../dev_common.hpp"
#include "../launchers.hpp"

namespace isar {

namespace {

constexpr int kE = 16;   // elements per thread for the row transforms

// Range cell (or bin) of register slot e of a thread, before and after a row transform.
template <int N>
__device__ __forceinline__ int row_pos(int tid, int e) {
    static_assert(FftPlan<N, kE>::R[0] == 16 && FftPlan<N, kE>::R[FftPlan<N, kE>::NP - 1] == 16, "one layout");
    return tid + e * (N / kE);
}

// Dynamic LDS of the row kernels: the transform buffer (lds_padded_size(N) float2), 64 floats of
// reductions, then the constants of the stride-16 pass.
constexpr int row_words(int N) { return (lds_padded_size(N) * 2 + 64 + 3) & ~3; }   // 4-byte words before the constants
template <int N>
__device__ __forceinline__ FftCT* stride16_rows(float2* lds) {
    return reinterpret_cast<FftCT*>(reinterpret_cast<float*>(lds) + row_words(N));
}

// Spectrum of row m of frame f with HPC (FP64 phase), window and (-1)^n centring applied, in
// the first-pass layout (range_alignment.cu:13-18, high_speed_compensation.cu:4-54). With
// if_hrrp the STRETCH rows carry the window twice (getHRRP windows them in place first,
// common.cu:563-566) unless ONE_WINDOW asks for the rows as getHRRP transforms them.
//
// The HPC phase exp(j pi vk n^2) at the first-pass positions n = tid + e S, S = N / 16, is
// factorised as exp(j pi vk tid^2) * d^e * exp(j pi vk S^2 e^2) with d = exp(j pi 2 vk S tid):
// three FP64-reduced evaluations per thread (tid^2, d, d^4) and one per lane e < 16 of each wave
// (the e^2 factor, read by the other lanes), instead of sixteen. exp(j pi vk tid^2) d^e is walked
// along each group of four elements by one product with d, and the group base steps by d^4, so
// no factor is more than six products from an FP64-reduced value and only the running factor,
// the group base, d, d^4 and the lane's e^2 factor stay live beside the row. Every FP64 argument
// is a part of vk n^2 and is reduced at least as exactly as vk n^2 itself.
//
// The row's samples and window values are loaded first (RowSamples::load), together, and turned into
// the spectrum later (spectrum), every element times `scale`, a power of two.
//
// IFDS: the rows pass the pre-stage first (isar_main.cu:15-27: ifftshift, IFFT / N, ifftshift). Both
// shifts by N / 2 are by eight register slots, so that transform runs where the row is
// (prestage) instead of in a kernel of its own with a pass over memory each way: for 96 frames of
// 256 x 4096 that took 305 us beside pair 0's 456, together they take 550.
template <int N, bool ONE_WINDOW = false, bool IFDS = false>
struct RowSamples {
    static_assert(FftPlan<N, kE>::R[0] == 16, "factorised phase assumes a radix-16 first pass");
    float2 v[kE];
    float w[kE];
    double velocity;   // for the compensation phase (0 without)

    __device__ __forceinline__ void load(const Job& J, int f, int m, int tid_) {
        const int tid = opaque(tid_);
        const long long erow = echo_first_row(J, f) + m;
        const float2* row = J.echo + static_cast<size_t>(erow) * N;
        velocity = !IFDS && J.if_hpc ? J.velocity[erow] : 0.0;
#pragma unroll
        for (int e = 0; e < kE; ++e) v[e] = elem_u32(row + (IFDS ? e ^ 8 : e) * (N / kE), tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) w[e] = elem_u32(J.win_range + e * (N / kE), tid);
        issue_point();
    }

    // The IFDS pre-stage of the loaded row but for its 1 / N. getHRRP for IFDS (common.cu:546-558) undoes
    // the stage, ifftshift(FFT(ifftshift(pre))) = the input row, so the profile is the row itself.
    __device__ __forceinline__ void prestage(const Job& J, int f, int m, float2* lds, int tid_,
                                             const FftTwiddlesLds<N, kE>& tw) {
        if (J.hrrp) {
            const int tid = opaque(tid_);
            float2* dst = J.hrrp + (static_cast<size_t>(f) * J.M + m) * N;
#pragma unroll
            for (int e = 0; e < kE; ++e) elem_u32(dst + (e ^ 8) * (N / kE), tid) = v[e];
        }
        fft<N, kE, +1>(v, lds, tid_, tw);
#pragma unroll
        for (int e = 0; e < kE / 2; ++e) {
            const float2 t = v[e];
            v[e] = v[e + 8];
            v[e + 8] = t;
        }
    }

    __device__ __forceinline__ void spectrum(float2 (&x)[kE], const Job& J, int tid_, float scale) const {
        const int tid = opaque(tid_);
        const bool hpc = !IFDS && J.if_hpc;
        const bool hrrp_window = !IFDS && !ONE_WINDOW && J.if_hrrp;
        // N/16 is even, so the sign (-1)^n is that of the thread
        const float sign = (tid & 1) ? -1.0f : 1.0f;
        auto window = [&](int e) { return sign * (hrrp_window ? w[e] * w[e] : w[e]); };
        if (!hpc) {
#pragma unroll
            for (int e = 0; e < kE; ++e) x[e] = cscale(v[e], scale * window(e));
            return;
        }
        constexpr double S = N / kE;
        const double vk = uniform(J.hpc_k * velocity);
        const double t = static_cast<double>(tid);
        const double lin = 2.0 * S * vk * t;
        const float2 d1 = expjpi_reduced(lin);
        const float2 d4 = expjpi_reduced(4.0 * lin);
        float2 base = cscale(expjpi_reduced(vk * t * t), scale);
        const double e0 = static_cast<double>(tid & 15);
        const float2 c = expjpi_reduced((S * S) * vk * (e0 * e0));
        issue_point();
#pragma unroll
        for (int q = 0; q < kE / 4; ++q) {
            float2 h = base;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = 4 * q + r;
                const float2 ce = make_float2(wave_read_lane(c.x, e), wave_read_lane(c.y, e));
                x[e] = cscale(cmul(v[e], cmul(h, ce)), window(e));
                if (r < 3) h = cmul(h, d1);
            }
            if (q + 1 < kE / 4) base = cmul(base, d4);
        }
    }
};

// Stored spectrum S0 of row m times its lag ramp exp(-j 2 pi n lag / N), lag = before + by, after the first pass of
// its inverse transform. With n = tid + e N/16 the ramp factors into exp(j pi b tid) * u^e,
// u = exp(j pi b N / 16) = exp(-j pi lag / 8), b = -2 lag / N. The powers of u are taken by the
// pass itself, as its twiddle: the eight constants (fft_table::Pow2) are the same for every
// thread, so lane l < 8 of each wave forms the l-th and the others read it. exp(j pi b tid) is one
// product per element. Arguments are reduced in FP64.
template <int N>
__device__ __forceinline__ void load_row_shifted(float2 (&x)[kE], const Job& J, int f, int m, double before, double by,
                                                 int tid_) {
    static_assert(FftPlan<N, kE>::R[0] == 16, "factorised ramp assumes a radix-16 first pass");
    const int tid = opaque(tid_);
    const float2* row = J.pre + (static_cast<size_t>(f) * J.M + m) * N;
#pragma unroll
    for (int e = 0; e < kE; ++e) x[e] = elem_u32(row + e * (N / kE), tid);
    issue_point();
    const double lag = uniform(before + by);
    const float2 w0 = expjpi_reduced(-2.0 * lag / N * tid);
    const int l = tid & 7;
    const double turns = (l == 0 ? 8.0 : l == 1 ? 4.0 : l < 4 ? 2.0 : 1.0) * (-0.125 * lag) +
                         (l == 3 ? 0.25 : l < 4 ? 0.0 : 0.125 * (l - 4));
    const float2 cs = expjpi_reduced(turns);
    const float c = fabsf(cs.x) < 0x1p-30f ? 0x1p-30f : cs.x;
    const float r = rcp_hw(c);
    float t = cs.y * r;
    t = fmaf(fmaf(-t, c, cs.y), r, t);   // cs.y / c to an ulp
    FftCTs<8> ramp;
#pragma unroll
    for (int i = 0; i < 8; ++i) ramp.v[i] = FftCT{wave_read_lane(c, i), wave_read_lane(t, i)};
#pragma unroll
    for (int e = 0; e < kE; ++e) x[e] = cmul(x[e], w0);
    dft16_twiddled<+1>(x, ramp);
}

// Energy profile of group g at merge stride s >= 2. Level 1 (s = 2)
// energies are complete (written by the fused level-0 pass); from level 2 on, the shifted second
// subgroup of the previous level is added from its row-chunk partial sums.
template <int N>
__device__ __forceinline__ void group_energy(float (&a)[kE], const Job& J, int f, int g, int s, int tid) {
    const int M = J.M;
    const float* base = J.egrp + (static_cast<size_t>(f) * M + static_cast<size_t>(g) * s) * N;
#pragma unroll
    for (int e = 0; e < kE; ++e) a[e] = elem_u32(base, row_pos<N>(tid, e));
    if (s > 2) {
        const int s2 = s / 2;
        const int r0 = (2 * g + 1) * s2;
        if (r0 < M) {
            const int r1 = min(r0 + s2, M);
            const int R = min(s2, J.ra_chunk);
            const float* pp = J.epart + (static_cast<size_t>(f) * M + r0) * N;
            const size_t step = static_cast<size_t>(R) * N;
            int left = (r1 - r0 + R - 1) / R;
            constexpr int kAtOnce = N >= 8192 ? 2 : 4;   // partial sums with their loads in flight together
            for (; left >= kAtOnce; left -= kAtOnce, pp += kAtOnce * step) {
                float v[kAtOnce][kE];
#pragma unroll
                for (int q = 0; q < kAtOnce; ++q)
#pragma unroll
                    for (int e = 0; e < kE; ++e) v[q][e] = elem_u32(pp + q * step, row_pos<N>(tid, e));
                issue_point();
#pragma unroll
                for (int q = 0; q < kAtOnce; ++q)
#pragma unroll
                    for (int e = 0; e < kE; ++e) a[e] += v[q][e];
            }
            for (; left > 0; --left, pp += step) {
#pragma unroll
                for (int e = 0; e < kE; ++e) a[e] += elem_u32(pp, row_pos<N>(tid, e));
            }
        }
    }
}

// Correlation of two non-negative profiles given as energies: the argmax of
// |c| after ifftshift, lowest index on ties (range_alignment.cu:45-61, 108-168). The real
// correlation comes from one complex FFT of gA + j gB, whose spectrum lands in the layout that the
// inverse transform takes, so only the mirrored bins N - k go through LDS. Every thread gets the
// argmax.
template <int N>
__device__ int correlation_argmax(const float (&a)[kE], const float (&b)[kE], float2* lds, float* redv, int* redi,
                                  int tid, const FftTwiddlesLds<N, kE>& tw) {
    constexpr int NT = N / kE;
    float2 x[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) x[e] = make_float2(sqrt_hw(a[e]), sqrt_hw(b[e]));
    fft<N, kE, -1>(x, lds, tid, tw);
    // bin k = tid + e T; its mirror N - k = (T - tid) + (15 - e) T, which is 0 (not N) for k = 0
    constexpr int T = N / kE;
    static_assert(FftPlan<N, kE>::R[0] == 16 && T % lds_pad_every(N) == 0, "bins of a thread T apart");
    {
        float2* at = lds + lds_pad<N>(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) at[lds_pad<N>(e * T)] = x[e];
    }
    __syncthreads();
    const float2* mirror = lds + lds_pad<N>(T - tid);
    const float2* mirror0 = tid == 0 ? lds : mirror + lds_pad<N>(15 * T);
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const float2 zk = x[e], zn = e == 0 ? *mirror0 : mirror[lds_pad<N>((15 - e) * T)];
        const float2 ga = make_float2(0.5f * (zk.x + zn.x), 0.5f * (zk.y - zn.y));
        const float2 gb = make_float2(0.5f * (zk.y + zn.y), -0.5f * (zk.x - zn.x));
        x[e] = cmulc(ga, gb);
    }
    __syncthreads();
    fft<N, kE, +1>(x, lds, tid, tw);
    float best = -1.0f;
    int bi = 0;
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const int i = (row_pos<N>(tid, e) + N / 2) & (N - 1);
        const float v = fabsf(x[e].x);
        if (v > best || (v == best && i < bi)) { best = v; bi = i; }
    }
    // the transform's last LDS reads precede the reduction's barriers
    block_argmax<NT>(best, bi, redv, redi);
    return bi;
}

// sqrt(x) to about 1e-14 relative for x >= 0: the hardware FP32 root (within 1 ulp) refined by one
// Newton step in FP64, s + (x - s^2) / (2 s); the step's own factor 1 / (2 s) needs only the
// hardware reciprocal's accuracy (1 ulp). A few FP64 operations instead of the long correctly rounded
// FP64 square root.
__device__ __forceinline__ double sqrt_refined(float x) {
    const float s = sqrt_hw(x);
    const double sd = static_cast<double>(s);
    const double d = fma(-sd, sd, static_cast<double>(x));
    return s > 0.0f ? fma(d, static_cast<double>(0.5f * rcp_hw(s)), sd) : 0.0;
}

// Parabolic lag around the argmax bi (binomialFixDevice, range_alignment.cu:121-131). The three
// samples c[bi-1], c[bi], c[bi+1] are formed again as direct sums sum_n gA[n] gB[n - l] in FP64,
// not read from the FP32 transform: near a broad peak the second
// difference f1 + f3 - 2 f2 cancels most of its digits, and the transform's rounding alone moved
// the vertex by up to 2.4e-4 cell at 1024 x 16384, which 120 autofocus iterations amplify into a
// 1e-3 image difference. The vertex and the lag are FP64. a, b: the two energy profiles. Must follow
// correlation_argmax (its barriers end the LDS use). Thread 0 records the lag and argmax; every thread
// gets the lag.
template <int N>
__device__ double parabola_lag(const float (&a)[kE], const float (&b)[kE], int bi, float2* lds, int tid,
                               double* lag_out, int32_t* imax_out) {
    constexpr int NT = N / kE;
    // cl[i] = c[i - N/2] and c[l] = sum_n gA[n] gB[n - l] (mod N): the samples at bi - 1, bi,
    // bi + 1 are lags l0 - 1, l0, l0 + 1 with l0 = bi - N/2. gB goes to LDS by range cell, its first
    // two cells once more behind the last, so that the three cells of a product follow each other (N + 2
    // doubles fit the transform's padded N float2); each thread sums over its own cells. The
    // per-wave sums follow gB in LDS and are added in wave order, so the result does not depend
    // on scheduling.
    // The profiles are the square roots of the FP32 energies to FP64 accuracy (the hardware FP32
    // root alone is off by up to 1 ulp, which the vertex would see). The energies pass through
    // opaque() so that the roots are not shared with the transform input above and kept live
    // across its transforms.
    double* gb = reinterpret_cast<double*>(lds);
    double* red = gb + N + 2;
    auto pos = [&](int e) { return row_pos<N>(tid, e); };
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const double g = sqrt_refined(opaque(b[e]));
        gb[pos(e)] = g;
        if (e == 0 && tid < 2) gb[N + tid] = g;
    }
    __syncthreads();
    const int l0 = bi - N / 2;
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const double ga = sqrt_refined(opaque(a[e]));
        const double* g = gb + ((pos(e) - l0 - 1) & (N - 1));
        s1 = fma(ga, g[2], s1);
        s2 = fma(ga, g[1], s2);
        s3 = fma(ga, g[0], s3);
    }
    s1 = wave_sum_d(s1);
    s2 = wave_sum_d(s2);
    s3 = wave_sum_d(s3);
    const int w = tid >> 6;
    if ((tid & 63) == 0) {
        red[3 * w] = s1;
        red[3 * w + 1] = s2;
        red[3 * w + 2] = s3;
    }
    __syncthreads();
    if (tid == 0) {
        double f1 = 0.0, f2 = 0.0, f3 = 0.0;
#pragma unroll
        for (int k = 0; k < (NT + 63) / 64; ++k) {
            f1 += red[3 * k];
            f2 += red[3 * k + 1];
            f3 += red[3 * k + 2];
        }
        double delta = 0.0;
        if (bi > 0 && bi < N - 1) {   // Q9a: no refinement at the row edge
            const double fa = (f1 + f3 - 2.0 * f2) / 2.0, fb = (f3 - f1) / 2.0;
            if (fa != 0.0) delta = -fb / (2.0 * fa);
            if (!(delta == delta) || fabs(delta) > 1e30) delta = 0.0;
        }
        const double lag = static_cast<double>(l0) + delta;
        *lag_out = lag;
        *imax_out = bi;
        red[0] = lag;
    }
    __syncthreads();
    const double lag = uniform(red[0]);
    __syncthreads();
    return lag;
}

}  // namespace

// IFDS pre-stage (isar_main.cu:15-27): ifftshift, IFFT / N, ifftshift of every row, for stage reads (a
// run does it in k_ra_pair0).
template <int N>
__global__ __launch_bounds__(N / kE) void k_ifds_pre(Job J) {
    HIP_DYNAMIC_SHARED(float2, lds);
    const int m = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
    const size_t off = (static_cast<size_t>(f) * J.M + m) * N;
    const float2* src = J.echo + static_cast<size_t>(echo_first_row(J, f) + m) * N;
    float2 x[kE];
#pragma unroll
    for (int e = 0; e < kE; ++e) x[e] = src[(row_pos<N>(tid, e) + N / 2) & (N - 1)];
    fft<N, kE, +1>(x, lds, tid);
    const float inv = 1.0f / N;
#pragma unroll
    for (int e = 0; e < kE; ++e) J.pre[off + ((row_pos<N>(tid, e) + N / 2) & (N - 1))] = cscale(x[e], inv);
}

// getHRRP for STRETCH (common.cu:561-571): ifftshift(FFT(hamming_N * row)) of the compensated
// rows, one workgroup per row. The ifftshift is the (-1)^n modulation RowSamples applies.
template <int N>
__global__ __launch_bounds__(N / kE) void k_hrrp(Job J) {
    HIP_DYNAMIC_SHARED(float2, lds);
    const int m = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
    float2 x[kE];
    RowSamples<N, true> row;
    float2* dst = J.hrrp + (static_cast<size_t>(f) * J.M + m) * N;
#pragma unroll 1
    for (float scale = 1.0f;; scale = kFftLarge) {
        const int t = opaque(tid);   // nothing is kept in registers for the second time
        row.load(J, f, m, t);
        row.spectrum(x, J, t, scale);
        fft<N, kE, -1>(x, lds, t);
#pragma unroll
        for (int e = 0; e < kE; ++e) dst[row_pos<N>(t, e)] = cscale(x[e], 1.0f / scale);
        if (scale != 1.0f || !fft_overflowed(x)) break;
    }
}

// Merge level 0 fused with the spectrum preparation (range_alignment.cu:13-18 and :34-73 at
// stride 1), one workgroup per row pair (2p, 2p+1): S0 of both rows (stored for the later
// levels), both energy profiles, their correlation and lag, the shift of row 2p+1 and the
// merged level-1 energy. Rows 0 and 1 never move again: their aligned profiles and column sums
// are written here. The spectra carry the inverse transforms' 1 / N (a power of two), so no
// profile or energy is scaled later.
// Bound by memory and by vector issue alike: 256 frames of 256 x 4096 take 1.21 ms, in which it moves
// 23.2 MB a frame at 4.9 TB/s (a plain copy reaches 4.7) and issues 2.66 M vector instructions a
// frame, 1.11 of the rate of one in 4 cycles; 1024 frames take 5.5 ms. (S0 of row 2p+1 kept in registers
// instead of read again saves 4.2 MB a frame, but then the fourth wave of a SIMD does not fit: 5.7 ms.)
template <int N, bool IFDS>
__global__ __launch_bounds__(N / kE, 4) void k_ra_pair0(Job J) {
    HIP_DYNAMIC_SHARED(float2, lds);
    constexpr int NT = N / kE;
    float* redv = reinterpret_cast<float*>(lds + lds_padded_size(N));
    int* redi = reinterpret_cast<int*>(redv + 16);
    const int p = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
    const int M = J.M;
    const int ra = 2 * p, rb = 2 * p + 1;
    constexpr float invN = 1.0f / N;
    const bool final_rows = (p == 0);
    float2* s0a = J.pre + (static_cast<size_t>(f) * M + ra) * N;
    float2* s0b = J.pre + (static_cast<size_t>(f) * M + rb) * N;
    float* dst = J.egrp + (static_cast<size_t>(f) * M + ra) * N;
    float* ap = J.arp_part + static_cast<size_t>(f) * (M / 2) * N;
    RowSamples<N, false, IFDS> row;
    row.load(J, f, ra, tid);
    const auto tw = fft_twiddles_lds<N, kE>(tid, stride16_rows<N>(lds));
    float2 x[kE];
    float ea[kE], eb[kE];
    constexpr float scale = IFDS ? invN * invN : invN;
    float mx = 0.0f;
    // Every global location below is re-read only by the thread that wrote it, and the stores
    // into the S0 rows (which st aliases) are ordered by the barriers inside each transform.
    // row 2p: S0, profile, energy (kept in registers as the first term of the merged energy)
    if constexpr (IFDS) row.prestage(J, f, ra, lds, tid, tw);
    row.spectrum(x, J, tid, scale);
    {
        const int t = opaque(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) elem_u32(s0a + e * (N / kE), t) = x[e];
    }
    fft<N, kE, +1>(x, lds, tid, tw);
    if (final_rows) {   // row 0 is the reference of the merge tree and never moves
        const int t = opaque(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const int pos = row_pos<N>(t, e);
            elem_u32(s0a, pos) = x[e];
            const float av = cabs_hw(x[e]);
            elem_u32(ap, pos) = av;
            mx = fmaxf(mx, av);
        }
    }
#pragma unroll
    for (int e = 0; e < kE; ++e) ea[e] = cabs2(x[e]);
    // row 2p+1: S0 and energy
    row.load(J, f, rb, tid);
    if constexpr (IFDS) row.prestage(J, f, rb, lds, tid, tw);
    row.spectrum(x, J, tid, scale);
    {
        const int t = opaque(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) elem_u32(s0b + e * (N / kE), t) = x[e];
    }
    fft<N, kE, +1>(x, lds, tid, tw);
#pragma unroll
    for (int e = 0; e < kE; ++e) eb[e] = cabs2(x[e]);
    const size_t idx = static_cast<size_t>(f) * (M - 1) + p;
    const int bi = correlation_argmax<N>(ea, eb, lds, redv, redi, tid, tw);
    const double lag = parabola_lag<N>(ea, eb, bi, lds, tid, J.lags + idx, J.imax + idx);
    // shift row 2p+1 by the lag and merge (range_alignment.cu:66-69)
    load_row_shifted<N>(x, J, f, rb, 0.0, lag, tid);
    fft_after_first<N, kE, +1>(x, lds, tid, tw);
    {
        const int t = opaque(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) elem_u32(dst + e * (N / kE), t) = ea[e] + cabs2(x[e]);
    }
    if (tid == 0) {
        J.lagsum[static_cast<size_t>(f) * M + ra] = 0.0;
        J.lagsum[static_cast<size_t>(f) * M + rb] = lag;
    }
    if (final_rows) {   // row 1 never moves again either
        const int t = opaque(tid);
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const int pos = row_pos<N>(t, e);
            elem_u32(s0b, pos) = x[e];
            const float av = cabs_hw(x[e]);
            elem_u32(ap, pos) += av;
            mx = fmaxf(mx, av);
        }
        mx = block_max<NT>(mx, redv);
        if (tid == 0) J.max_part[static_cast<size_t>(f) * (M / 2)] = mx;
    }
}

// One merge level s >= 2: group energies of pair p and their correlation (range_alignment.cu:
// 45-61). The first group's energy is kept for the next level.
template <int N>
__global__ __launch_bounds__(N / kE, 4) void k_ra_corr(Job J, int s, int pair_base) {
    HIP_DYNAMIC_SHARED(float2, lds);
    float* redv = reinterpret_cast<float*>(lds + lds_padded_size(N));
    int* redi = reinterpret_cast<int*>(redv + 16);
    const int p = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
    const int M = J.M;
    const int ngroups = (M + s - 1) / s, npairs = ngroups / 2;
    const bool unpaired = (p == npairs);
    const int gA = unpaired ? ngroups - 1 : 2 * p;
    const auto tw = fft_twiddles_lds<N, kE>(tid, stride16_rows<N>(lds));
    float a[kE], b[kE];
    group_energy<N>(a, J, f, gA, s, tid);
    {   // keep the first group's energy for the next level (same head row, same thread)
        float* dst = J.egrp + (static_cast<size_t>(f) * M + static_cast<size_t>(gA) * s) * N;
#pragma unroll
        for (int e = 0; e < kE; ++e) elem_u32(dst, row_pos<N>(tid, e)) = a[e];
    }
    if (unpaired) return;
    group_energy<N>(b, J, f, gA + 1, s, tid);
    const size_t idx = static_cast<size_t>(f) * (M - 1) + pair_base + p;
    const int bi = correlation_argmax<N>(a, b, lds, redv, redi, tid, tw);
    (void)parabola_lag<N>(a, b, bi, lds, tid, J.lags + idx, J.imax + idx);
}

// Shift the rows of the second group of pair p by the pair's lag (range_alignment.cu:66-69)
// and accumulate their new energies; each workgroup handles up to J.ra_chunk rows. The rows of
// pair 0 move for the last time at this level: their aligned profiles replace their spectra and
// their column sums feed HRRP centring.
// PART selects the grid: kUpdAll, the chunks of every pair (final rows where p = 0, one launch
// per level); kUpdFinal, the chunks of pair 0 only; kUpdRest, those of pairs 1, 2, ... Apart
// from the final-row work the three run the same code.
// Bound by memory: 1024 frames of 256 x 4096 read S0 of half the rows at each of seven levels and write
// all profiles once, 41.6 GB in 8.3 ms.
constexpr int kUpdAll = 0, kUpdFinal = 1, kUpdRest = 2;
template <int N, int PART>
__global__ __launch_bounds__(N / kE, 4) void k_ra_upd(Job J, int s, int pair_base) {
    HIP_DYNAMIC_SHARED(float2, lds);
    const int b = blockIdx.x, f = blockIdx.y, tid = threadIdx.x;
    const int M = J.M;
    const int R = min(s, J.ra_chunk);
    const int cpp = (s + R - 1) / R;
    const int p = b / cpp + (PART == kUpdRest ? 1 : 0), i = b % cpp;
    const int gend = min((2 * p + 2) * s, M);
    const int r0 = (2 * p + 1) * s + i * R;
    const int r1 = min(r0 + R, gend);
    if (r0 >= r1) return;
    const double lag = uniform(J.lags[static_cast<size_t>(f) * (M - 1) + pair_base + p]);
    const bool final_rows = PART == kUpdFinal || (PART == kUpdAll && p == 0);
    float acc[kE];
    float mx = 0.0f;
#pragma unroll
    for (int e = 0; e < kE; ++e) acc[e] = 0.0f;
    float2 x[kE];
    const auto tw = fft_twiddles_lds<N, kE>(tid, stride16_rows<N>(lds));
    // column sums of |profile| over the final rows of this chunk, in registers (added in place in memory
    // they cost a final row as many bytes again: 40 frames of 512 x 8192 took 2.16 instead of 1.75 ms)
    constexpr bool kFinal = PART != kUpdRest;
    float* ap = J.arp_part + (static_cast<size_t>(f) * (M / 2) + r0 / 2) * N;
    float arp[kFinal ? kE : 1];
#pragma unroll
    for (int e = 0; e < (kFinal ? kE : 1); ++e) arp[e] = 0.0f;
#pragma unroll 1
    for (int m = r0; m < r1; ++m) {
        load_row_shifted<N>(x, J, f, m, J.lagsum[static_cast<size_t>(f) * M + m], lag, tid);
        fft_after_first<N, kE, +1>(x, lds, tid, tw);
#pragma unroll
        for (int e = 0; e < kE; ++e) acc[e] += cabs2(x[e]);
        if (final_rows) {   // S0 of row m was read before the transform's first barrier
            float2* st = J.st + (static_cast<size_t>(f) * M + m) * N;
            const int t = opaque(tid);
#pragma unroll
            for (int e = 0; e < kE; ++e) {
                const int pos = row_pos<N>(t, e);
                elem_u32(st, pos) = x[e];
                const float av = cabs_hw(x[e]);
                if constexpr (kFinal) arp[e] += av;
                mx = fmaxf(mx, av);
            }
        }
    }
    if (final_rows) {
        if constexpr (kFinal) {
            const int t = opaque(tid);
#pragma unroll
            for (int e = 0; e < kE; ++e) elem_u32(ap, row_pos<N>(t, e)) = arp[e];
        }
        float* red = reinterpret_cast<float*>(lds + lds_padded_size(N));
        mx = block_max<N / kE>(mx, red);
        if (tid == 0) J.max_part[static_cast<size_t>(f) * (M / 2) + r0 / 2] = mx;
    }
    __syncthreads();
    if (tid < r1 - r0) J.lagsum[static_cast<size_t>(f) * M + r0 + tid] += lag;
    float* dst = J.epart + (static_cast<size_t>(f) * M + r0) * N;
#pragma unroll
    for (int e = 0; e < kE; ++e) elem_u32(dst, row_pos<N>(tid, e)) = acc[e];
}

// k_ra_upd (kUpdAll) for batches that leave the GPU idle with one row of each chunk at a time: a
// workgroup takes G rows of its chunk at once, N / 16 threads each with a transform buffer of its
// own. The rows' energies go through those buffers, and every thread adds 16 / G cells over the rows
// in their order: the sums are k_ra_upd's bit for bit.
// Bound by latency (a row's loads, ramp and transform, one after the other): a level of 13 frames of
// 192 x 2048 in chunks of 8 takes 15 us instead of 36, of one frame of 256 x 4096 in chunks of 2 9
// instead of 14; imaging 32 such frames in chunks of 8 1.39 ms instead of 1.48.
template <int N, int G>
__global__ __launch_bounds__(N / kE * G) void k_ra_upd_rows(Job J, int s, int pair_base) {
    HIP_DYNAMIC_SHARED(float2, lds);   // G transform buffers, 64 floats of reductions, constants (rows_words)
    constexpr int T = N / kE, B = lds_padded_size(N), C = kE / G;
    const int b = blockIdx.x, f = blockIdx.y, g = threadIdx.x / T, tid = threadIdx.x % T;
    const int M = J.M;
    const int R = min(s, J.ra_chunk);
    const int cpp = (s + R - 1) / R;
    const int p = b / cpp, i = b % cpp;
    const int gend = min((2 * p + 2) * s, M);
    const int r0 = (2 * p + 1) * s + i * R;
    const int r1 = min(r0 + R, gend);
    if (r0 >= r1) return;
    const double lag = uniform(J.lags[static_cast<size_t>(f) * (M - 1) + pair_base + p]);
    const bool final_rows = p == 0;
    float* const red = reinterpret_cast<float*>(lds + G * B);
    const auto tw = fft_twiddles_lds<N, kE>(tid, reinterpret_cast<FftCT*>(red + 64));
    float2* const buf = lds + g * B;
    float acc[C], arp[C];
    float mx = 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = arp[c] = 0.0f;
#pragma unroll 1
    for (int m0 = r0; m0 < r1; m0 += G) {
        const int m = min(m0 + g, r1 - 1);   // past the chunk's end: the last row, not used
        float2 x[kE];
        load_row_shifted<N>(x, J, f, m, J.lagsum[static_cast<size_t>(f) * M + m], lag, tid);
        fft_after_first<N, kE, +1>(x, buf, tid, tw);
        if (final_rows && m0 + g < r1) {   // S0 of the row was read before the transform's first barrier
            float2* st = J.st + (static_cast<size_t>(f) * M + m) * N;
            const int t = opaque(tid);
#pragma unroll
            for (int e = 0; e < kE; ++e) elem_u32(st, row_pos<N>(t, e)) = x[e];
        }
        __syncthreads();   // the transforms' last reads
#pragma unroll
        for (int e = 0; e < kE; ++e) reinterpret_cast<float*>(buf)[row_pos<N>(tid, e)] = cabs2(x[e]);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < G; ++q) {
            if (m0 + q >= r1) break;
            const float* row = reinterpret_cast<const float*>(lds + q * B) + threadIdx.x;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float e = row[c * T * G];
                acc[c] += e;
                if (final_rows) {
                    const float av = sqrt_hw(e);
                    arp[c] += av;
                    mx = fmaxf(mx, av);
                }
            }
        }
        __syncthreads();
    }
    const size_t cell = threadIdx.x;
    if (final_rows) {
        float* ap = J.arp_part + (static_cast<size_t>(f) * (M / 2) + r0 / 2) * N + cell;
#pragma unroll
        for (int c = 0; c < C; ++c) ap[c * T * G] = arp[c];
        mx = block_max<T * G>(mx, red);
        if (threadIdx.x == 0) J.max_part[static_cast<size_t>(f) * (M / 2) + r0 / 2] = mx;
    }
    if (static_cast<int>(threadIdx.x) < r1 - r0) J.lagsum[static_cast<size_t>(f) * M + r0 + threadIdx.x] += lag;
    float* dst = J.epart + (static_cast<size_t>(f) * M + r0) * N + cell;
#pragma unroll
    for (int c = 0; c < C; ++c) dst[c * T * G] = acc[c];
}

// Range Hamming window 0.54 - 0.46 cos(2 pi n / (N - 1)) (genHammingVec, common.cu:260-266),
// evaluated in FP64 and rounded once to FP32.
__global__ __launch_bounds__(256) void k_range_window(int N, float* win) {
    const int n = blockIdx.x * 256 + threadIdx.x;
    if (n < N) win[n] = static_cast<float>(0.54 - 0.46 * cos(2.0 * 3.14159265358979323846 * n / (N - 1)));
}

// ------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------
namespace {
template <int N>
size_t ra_lds() { return row_words(N) * sizeof(float) + kFft16Bytes; }
template <int N, int G>
size_t ra_rows_lds() { return G * lds_padded_size(N) * sizeof(float2) + 64 * sizeof(float) + kFft16Bytes; }

// The rows that k_ra_upd_rows may take at once: up to 8, in workgroups of at most 1024 threads.
template <int N>
constexpr int kRowsMax = N >= 16384 ? 1 : N == 8192 ? 2 : N == 4096 ? 4 : 8;

// Rows at once of a level's chunks of R rows: doubled until the grid gives every SIMD four waves, which
// is what fits beside each other; with that many, chunks row by row do as well without the exchange.
template <int N>
int rows_at_once(int frames, int nblocks, int R) {
    const long long waves = static_cast<long long>(frames) * nblocks * (N / kE / 64);
    int g = 1;
    while (2 * g <= std::min(R, kRowsMax<N>) && waves * g < 4 * 4 * kComputeUnits) g *= 2;
    return g;
}

template <int N, int G>
void launch_upd_rows(const Job& J, int stride, int pair_base, int nblocks, hipStream_t s) {
    if constexpr (G <= kRowsMax<N>)
        ISAR_LAUNCH((k_ra_upd_rows<N, G>), dim3(nblocks, J.K), dim3(N / kE * G), (ra_rows_lds<N, G>()), s, J, stride, pair_base);
}
template <int N>
bool upd_rows(const Job& J, int stride, int pair_base, int nblocks, int R, hipStream_t s) {
    switch (rows_at_once<N>(J.K, nblocks, R)) {
    case 2: launch_upd_rows<N, 2>(J, stride, pair_base, nblocks, s); return true;
    case 4: launch_upd_rows<N, 4>(J, stride, pair_base, nblocks, s); return true;
    case 8: launch_upd_rows<N, 8>(J, stride, pair_base, nblocks, s); return true;
    default: return false;
    }
}

#define ISAR_RANGE_SWITCH(N, BODY)                     \
    switch (N) {                                       \
    case 1024: { constexpr int NN = 1024; BODY; } break;   \
    case 2048: { constexpr int NN = 2048; BODY; } break;   \
    case 4096: { constexpr int NN = 4096; BODY; } break;   \
    case 8192: { constexpr int NN = 8192; BODY; } break;   \
    case 16384: { constexpr int NN = 16384; BODY; } break; \
    default: break;                                    \
    }
}  // namespace

bool range_size_supported(int N) {
    return N == 1024 || N == 2048 || N == 4096 || N == 8192 || N == 16384;
}

hipError_t configure_ra_kernels() {
    hipError_t err = hipSuccess;
#ifndef ISAR_EMU
    auto set = [&](const void* fn, size_t bytes) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        if (e != hipSuccess) {
            err = e;
            report_config_error(__FILE__, bytes);
        }
    };
#define ISAR_SET_RA(NN)                                                        \
    set(reinterpret_cast<const void*>(&k_ifds_pre<NN>), ra_lds<NN>());         \
    set(reinterpret_cast<const void*>(&k_hrrp<NN>), ra_lds<NN>());             \
    set(reinterpret_cast<const void*>(&k_ra_pair0<NN, false>), ra_lds<NN>());  \
    set(reinterpret_cast<const void*>(&k_ra_pair0<NN, true>), ra_lds<NN>());   \
    set(reinterpret_cast<const void*>(&k_ra_corr<NN>), ra_lds<NN>());          \
    set(reinterpret_cast<const void*>(&k_ra_upd<NN, kUpdAll>), ra_lds<NN>());   \
    set(reinterpret_cast<const void*>(&k_ra_upd<NN, kUpdFinal>), ra_lds<NN>()); \
    set(reinterpret_cast<const void*>(&k_ra_upd<NN, kUpdRest>), ra_lds<NN>());
    ISAR_SET_RA(1024) ISAR_SET_RA(2048) ISAR_SET_RA(4096) ISAR_SET_RA(8192) ISAR_SET_RA(16384)
#undef ISAR_SET_RA
#define ISAR_SET_ROWS(NN, GG) set(reinterpret_cast<const void*>(&k_ra_upd_rows<NN, GG>), ra_rows_lds<NN, GG>());
    ISAR_SET_ROWS(1024, 2) ISAR_SET_ROWS(1024, 4) ISAR_SET_ROWS(1024, 8) ISAR_SET_ROWS(2048, 2) ISAR_SET_ROWS(2048, 4)
    ISAR_SET_ROWS(2048, 8) ISAR_SET_ROWS(4096, 2) ISAR_SET_ROWS(4096, 4) ISAR_SET_ROWS(8192, 2)
#undef ISAR_SET_ROWS
#endif
    return err;
}

void launch_range_window(int N, float* win, hipStream_t s) {
    ISAR_LAUNCH(k_range_window, dim3((N + 255) / 256), dim3(256), 0, s, N, win);
}

void launch_ifds_pre(const Job& J, hipStream_t s) {
    ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH(k_ifds_pre<NN>, dim3(J.M, J.K), dim3(NN / kE), ra_lds<NN>(), s, J));
}

void launch_hrrp(const Job& J, hipStream_t s) {
    ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH(k_hrrp<NN>, dim3(J.M, J.K), dim3(NN / kE), ra_lds<NN>(), s, J));
}
void launch_ra_pair0(const Job& J, hipStream_t s) {
    if (J.data_type == 1) {
        ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH((k_ra_pair0<NN, true>), dim3(J.M / 2, J.K), dim3(NN / kE), ra_lds<NN>(), s, J));
    } else {
        ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH((k_ra_pair0<NN, false>), dim3(J.M / 2, J.K), dim3(NN / kE), ra_lds<NN>(), s, J));
    }
}
void launch_ra_corr(const Job& J, int stride, int pair_base, int nblocks, hipStream_t s) {
    ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH(k_ra_corr<NN>, dim3(nblocks, J.K), dim3(NN / kE), ra_lds<NN>(), s, J,
                                       stride, pair_base));
}
void launch_ra_upd(const Job& J, int stride, int pair_base, int nblocks, hipStream_t s) {
    // nblocks = pairs x chunks per pair. Chunks that would leave SIMDs without work take several rows at
    // once. Batches of many frames launch pair 0 (final rows) and the other pairs apart, others together.
    const int R = std::min(stride, J.ra_chunk), cpp = (stride + R - 1) / R;
    if (J.ra_split == 0) {
        bool done = false;
        ISAR_RANGE_SWITCH(J.N, done = upd_rows<NN>(J, stride, pair_base, nblocks, R, s));
        if (done) return;
    }
    const bool split = J.ra_split == 2 || (J.ra_split == 0 && J.K >= kRaSplitFrames);
    if (!split) {
        ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH((k_ra_upd<NN, kUpdAll>), dim3(nblocks, J.K), dim3(NN / kE), ra_lds<NN>(),
                                           s, J, stride, pair_base));
        return;
    }
    const int rest = nblocks - cpp;
    ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH((k_ra_upd<NN, kUpdFinal>), dim3(cpp, J.K), dim3(NN / kE), ra_lds<NN>(), s, J,
                                       stride, pair_base));
    if (rest > 0)
        ISAR_RANGE_SWITCH(J.N, ISAR_LAUNCH((k_ra_upd<NN, kUpdRest>), dim3(rest, J.K), dim3(NN / kE), ra_lds<NN>(), s,
                                           J, stride, pair_base));
}

}  // namespace isar
