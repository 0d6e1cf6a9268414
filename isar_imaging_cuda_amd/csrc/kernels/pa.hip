// pa.hip — phase adjustment (phase_adjustment.cu:4-41, 167-346) for gfx950:
// Doppler-centroid tracking, column energy/entropy statistics, bin selection and the
// fast minimum-entropy autofocus with the selected bins kept resident per frame.
#include <algorithm>

#include "../dev_common.hpp"
#include "../launchers.hpp"

namespace isar {

namespace {

// phi[0] = 0, phi[m+1] = exp(-j theta_m), theta = inclusive scan of arg(r_m) (accumulated in
// FP64 and reduced before the FP32 sincos). r: M-1 adjacent-pulse products (LDS or global).
template <int NT>
__device__ void doppler_phase(const float2* r, int M, float2* phi, double* scratch, double* red) {
    for (int m = threadIdx.x; m < M - 1; m += NT) scratch[m] = static_cast<double>(atan2f(r[m].y, r[m].x));
    __syncthreads();
    block_inclusive_scan_d<NT>(scratch, M - 1, red);
    for (int m = threadIdx.x; m < M; m += NT) {
        if (m == 0) phi[0] = make_float2(0.0f, 0.0f);   // phase_adjustment.cu:29
        else phi[m] = expjpi_reduced(-scratch[m - 1] * 0.31830988618379067154);
    }
    __syncthreads();
}

// A float's bits as an unsigned number in the order of the floats, both zeros alike and NaNs last.
__device__ __forceinline__ unsigned order_key(float v) {
    if (!(v == v)) return 0xffffffffu;
    const unsigned b = __float_as_uint(v + 0.0f);
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}

// Rank of key[n] among key[0 ... count - 1] in LDS (ascending, equal keys by index), count at most W
// and a multiple of 4: the keys before n's wave count where they are no larger, those after it
// where they are smaller. All lanes of a wave read the same keys, four a load; a compare and an add
// each, so 512 keys cost W waves' 1024 instructions, where a bitonic sort passes 45 barriers or
// shuffles one after the other.
template <int W>
__device__ int rank_of(const unsigned* key, int count, int n) {
    const unsigned own = key[n];
    const int w0 = min(n & ~63, count), w1 = min(w0 + 64, count);
    int rank = 0;
    auto each = [&](int from, int to, auto before) {
#pragma unroll 4
        for (int k = from; k < to; k += 4) {
            const uint4 q = *reinterpret_cast<const uint4*>(key + k);
            rank += before(q.x, k) ? 1 : 0;
            rank += before(q.y, k + 1) ? 1 : 0;
            rank += before(q.z, k + 2) ? 1 : 0;
            rank += before(q.w, k + 3) ? 1 : 0;
        }
    };
    each(0, w0, [&](unsigned q, int) { return q <= own; });
    each(w0, w1, [&](unsigned q, int k) { return q < own || (q == own && k < n); });
    each(w1, count, [&](unsigned q, int) { return q < own; });
    return rank;
}

}  // namespace

// Doppler-centroid phase of the cut (dopplerTracking, phase_adjustment.cu:4-41) from the
// adjacent-pulse products k_cut formed: once per frame, for every column tile of k_pa_colfft.
template <int M>
__global__ __launch_bounds__(256) void k_pa_doppler(Job J) {
    HIP_DYNAMIC_SHARED(double, scr);   // M (scan) + 32 (its partial sums)
    const int f = blockIdx.x;
    doppler_phase<256>(J.rowdop + static_cast<size_t>(f) * M, M, J.dopphi + static_cast<size_t>(f) * M, scr,
                       scr + M);
}

// Per column tile: Doppler-tracked image column FFT, energy E_col, entropy H_col and the
// column maxima of |X| (phase_adjustment.cu:175-246).
template <int M>
__global__ __launch_bounds__(256) void k_pa_colfft(Job J) {
    using C = ColCfg<M>;
    constexpr int NT = C::NT, CT = C::CT, TPF = C::TPF, E = C::E;
    HIP_DYNAMIC_SHARED(float2, sm);
    float2* work = sm;                                   // tile / transform buffers
    const int tile = xcd_tile(blockIdx.x, gridDim.x), f = blockIdx.y, tid = threadIdx.x;
    const int W = J.W;
    const int g = tid / TPF, lane = tid % TPF;
    const int n0 = tile * CT, n = n0 + g;

    float2 phi[E];   // read ahead of the tile
    {
        const float2* d = J.dopphi + static_cast<size_t>(f) * M;
#pragma unroll
        for (int e = 0; e < E; ++e) phi[e] = elem_u32(d, static_cast<unsigned>(C::in(lane, e)));
    }
    load_column_tile<NT, CT>(J.x + static_cast<size_t>(f) * M * W, W, n0, M, work, tid);
    __syncthreads();
    float2 x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int pos = C::in(lane, e);
        x[e] = cmul(phi[e], work[pos * (CT + 1) + g]);
    }
    __syncthreads();
    float2* buf = work + g * lds_padded_size(M);
    fft<M, E, -1, true>(x, buf, lane);
    float p2[E];
    float esum = 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e) { p2[e] = cabs2(x[e]); esum += p2[e]; }
    const float Ecol = group_sum<TPF>(esum);
    float h = 0.0f;
    if (Ecol > 0.0f) {
        const float inv = 1.0f / Ecol;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float p = p2[e] * inv;
            if (p > 0.0f) h -= p * logf(p);
        }
    }
    const float H = group_sum<TPF>(h);
    if (lane == 0) {
        const int nb = (M + kCutBandRows - 1) / kCutBandRows;
        float cm = 0.0f;
        for (int b = 0; b < nb; ++b) cm = fmaxf(cm, J.colmax_part[(static_cast<size_t>(f) * nb + b) * W + n]);
        J.colmax[static_cast<size_t>(f) * W + n] = cm;
        J.colE[static_cast<size_t>(f) * W + n] = Ecol;
        J.colH[static_cast<size_t>(f) * W + n] = Ecol > 0.0f ? H : __int_as_float(0x7f800000);
    }
}

// Bin selection (phase_adjustment.cu:186-264): int-truncated mean of the column maxima,
// tgt_num bins above 1.48 * mean, the tgt_num most energetic (stable, descending), the
// unit2_num = nextPow2(tgt_num / 2) of those with the lowest entropy (stable, ascending),
// sorted by index. One workgroup of W threads per frame; the orders come from ranks (rank_of), the
// final one from a prefix sum over the bins. 13 us for a single frame, with three bitonic sorts 27.
template <int W>
__global__ __launch_bounds__(W) void k_pa_select(Job J) {
    HIP_DYNAMIC_SHARED(uint4, sm_sel);
    unsigned* key = reinterpret_cast<unsigned*>(sm_sel);   // W
    int* order1 = reinterpret_cast<int*>(key + W);         // W
    int* taken = order1 + W;                               // W
    int* ired = taken + W;                                 // 32
    const int f = blockIdx.x, n = threadIdx.x;
    const float mx = J.colmax[static_cast<size_t>(f) * W + n];
    const float E = J.colE[static_cast<size_t>(f) * W + n];
    const float H = J.colH[static_cast<size_t>(f) * W + n];
    // energy descending, index ascending on ties, NaN last
    key[n] = order_key((E == E) ? -E : __int_as_float(0x7f800000));
    taken[n] = 0;
    // thrust::reduce(..., 0, plus<int>()) (phase_adjustment.cu:186) converts every maximum to int
    // as the device does (truncation, clamped) and adds them in 32-bit arithmetic, which wraps
    unsigned utot = 0;
    (void)block_exclusive_scan<W, unsigned>(static_cast<unsigned>(trunc_sat_i32(mx)),
                                            reinterpret_cast<unsigned*>(ired), &utot);
    const int tot = static_cast<int>(utot);   // two's complement
    const float mean_val = static_cast<float>(tot) / static_cast<float>(W);
    const float threshold = 1.48f * mean_val;
    int tgt = 0;
    (void)block_exclusive_scan<W>(mx > threshold ? 1 : 0, ired, &tgt);
    int half = tgt / 2, U = 1;
    while (half >> 1) { U <<= 1; half >>= 1; }
    U <<= 1;   // nextPow2 (common.cu:521-529)
    const int rank1 = rank_of<W>(key, W, n);
    __syncthreads();
    // entropy ascending among the first tgt, rank ascending on ties
    key[rank1] = rank1 < tgt ? order_key(H) : 0xffffffffu;
    order1[rank1] = n;
    __syncthreads();
    // the first U of them
    if (n < tgt && rank_of<W>(key, (tgt + 3) & ~3, n) < U) taken[order1[n]] = 1;
    __syncthreads();
    // bin 0 fills positions beyond tgt, as std::vector growth does
    const int times = taken[n] + (n == 0 ? max(U - tgt, 0) : 0);
    int all = 0;
    const int at = block_exclusive_scan<W>(times, ired, &all);
    for (int i = 0; i < times; ++i) J.sel[static_cast<size_t>(f) * W + at + i] = n;
    if (n == 0) {
        J.dec[f].tgt_num = tgt;
        J.dec[f].unit2_num = U;
        J.dec[f].pa_threshold = threshold;
    }
}

// Fast minimum-entropy autofocus (phase_adjustment.cu:270-324): one workgroup per frame; the
// selected bins are gathered once into a column-major copy, then J.iterations fixed-point
// updates phi_m <- unit(sum_u conj(S[m,u]) IFFT(G |G|)[m,u] / M), G = FFT(diag(phi) S).
// CF columns are transformed at once (TPF threads each); when all U selected bins fit in one
// chunk they stay in registers for every iteration.
template <int M>
struct AfCfg {
    static constexpr int E = ColCfg<M>::E;
    static constexpr int TPF = ColCfg<M>::TPF;
    static constexpr int NT = M <= 384 ? 1024 : 512;
    static constexpr int CF = NT / TPF;                       // columns per chunk
    static constexpr int RPT = (M + NT - 1) / NT;             // rows per thread when M > NT
    static constexpr int Q = M <= NT ? (NT / M >= 16 ? 16 : NT / M >= 8 ? 8 : NT / M >= 4 ? 4 : NT / M >= 2 ? 2 : 1) : 1;
    // Summation order of the per-pulse sums: the selected bins in sub-chunks of SUB columns, each
    // summed column by column, the sub-chunk sums added in order. The one-workgroup form and the
    // split form (k_af_cols / k_af_phase) both follow it.
    static constexpr int SUB = CF / Q;
    static_assert(CF % Q == 0, "sub-chunks must tile a chunk");
};

// One term conj(S) IFFT(G |G|) / M of the per-pulse sums. Only the unit phasor of the sum is
// kept, so for a power-of-two M the 1/M is left out: scaling by 2^-k commutes with every rounding
// of the sum, its magnitude and the division, and the phases are the same bit for bit.
template <int M>
__device__ __forceinline__ float2 af_term(float2 s, float2 x, float invM) {
    if constexpr ((M & (M - 1)) == 0) return cconjmul(s, x);
    else return cscale(cconjmul(s, x), invM);
}

// The scale exponent of a frame's selected bins: 2^-e takes the largest selected |S| into [1, 2)
// (e = 0 for no finite positive maximum). cm: the workgroup's maximum of their column maxima.
__device__ __forceinline__ int af_scale_exponent(float cm) {
    return cm > 0.0f && cm <= 3.40282347e38f ? ilogbf(cm) : 0;
}

template <int M>
__global__ __launch_bounds__(AfCfg<M>::NT) void k_autofocus(Job J) {
    using A = AfCfg<M>;
    using C = ColCfg<M>;
    constexpr int NT = A::NT, E = A::E, TPF = A::TPF, CF = A::CF, RPT = A::RPT, Q = A::Q;
    HIP_DYNAMIC_SHARED(float2, sm);
    float2* phi = sm;                                     // M
    float2* rdop = phi + M;                               // M
    double* scr = reinterpret_cast<double*>(rdop + M);    // M
    double* red = scr + M;                                // NT
    float2* bufs = reinterpret_cast<float2*>(red + NT);   // CF * lds_padded_size(M)
    const int f = blockIdx.x, tid = threadIdx.x;
    const int W = J.W;
    const int U = J.dec[f].unit2_num;
    const int* sel = J.sel + static_cast<size_t>(f) * W;
    float2* su = J.su + static_cast<size_t>(f) * W * M;
    const float2* X = J.x + static_cast<size_t>(f) * M * W;
    if (J.af_redo && (J.dec[f].status & 2) == 0) return;   // the whole workgroup

    // gather the selected bins, column-major (selectRangeBins, :335-346), scaled by 2^-e so that
    // the largest selected |S| lies in [1, 2): the update takes the unit phasor of sums cubic in
    // S, and a power of two scales every product exactly, so the phases are those of the unscaled
    // bins while conj(S) IFFT(G |G|) stays far from FP32 overflow at any input level
    float cm = 0.0f;
    for (int u = tid; u < U; u += NT) cm = fmaxf(cm, J.colmax[static_cast<size_t>(f) * W + sel[u]]);
    cm = block_max<NT>(cm, reinterpret_cast<float*>(red));
    const int e = af_scale_exponent(cm);
    {   // the selected bins' indices in LDS (the transform buffers are free here), then the
        // gather with eight loads in flight per thread
        int* lsel = reinterpret_cast<int*>(bufs);
        for (int u = tid; u < U; u += NT) lsel[u] = sel[u];
        __syncthreads();
        for (int idx0 = tid; idx0 < U * M; idx0 += 8 * NT) {
            float2 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int idx = idx0 + i * NT;
                if (idx < U * M) v[i] = X[static_cast<size_t>(idx / U) * W + lsel[idx % U]];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int idx = idx0 + i * NT;
                if (idx < U * M)
                    su[static_cast<size_t>(idx % U) * M + idx / U] = make_float2(ldexpf(v[i].x, -e), ldexpf(v[i].y, -e));
            }
        }
    }
    __syncthreads();
    if (J.phi0_given) {
        for (int m = tid; m < M; m += NT) phi[m] = J.phi0_in[static_cast<size_t>(f) * M + m];
        __syncthreads();
    } else {
        // Doppler tracking of the selected bins without compensation (:282), the products added
        // in bin order with eight bins' loads in flight
        for (int m = tid; m < M - 1; m += NT) {
            float2 acc = make_float2(0.0f, 0.0f);
            for (int u0 = 0; u0 < U; u0 += 8) {
                float2 a[8], b[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (u0 + i < U) {
                        a[i] = su[static_cast<size_t>(u0 + i) * M + m];
                        b[i] = su[static_cast<size_t>(u0 + i) * M + m + 1];
                    }
                }
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (u0 + i < U) acc = cadd(acc, cconjmul(a[i], b[i]));
            }
            rdop[m] = acc;
        }
        __syncthreads();
        doppler_phase<NT>(rdop, M, phi, scr, red);
    }
    for (int m = tid; m < M; m += NT) J.phi0[static_cast<size_t>(f) * M + m] = phi[m];

    const int g = tid / TPF, lane = tid % TPF;
    float2* buf = bufs + g * lds_padded_size(M);
    const float invM = 1.0f / static_cast<float>(M);
    // the twiddle constants stay in registers for all iterations' transforms
    const auto fwd = fft_twiddles<M, E>(lane);
    const auto inv = fft_twiddles<M, E, true>(lane);
    // All iterations. ONE: the bins are one chunk, whose columns stay in registers; otherwise every
    // iteration reads the columns of each chunk. In a loop of their own the reads are issued together: 256
    // pulses with 512 bins take 6.4 ms (7.7 with both cases in one loop), 384 with 64 bins 2.14 (2.31). At 64
    // pulses a loop over the one chunk stays: without it 9 registers are spilled instead of 5, and a
    // frame takes 0.97 instead of 0.93 ms.
    float2 s[E];
    auto iterate = [&]<bool ONE>() {
        for (int it = 0; it < J.iterations; ++it) {
            float2 acc[RPT];
#pragma unroll
            for (int i = 0; i < RPT; ++i) acc[i] = make_float2(0.0f, 0.0f);
            for (int c0 = 0; c0 < (ONE && M > 64 ? 1 : U); c0 += CF) {
                const float2* col = su + static_cast<size_t>(c0 + g) * M;
                if constexpr (!ONE) {   // U and CF are powers of two: every column is one of the U
#pragma unroll
                    for (int e = 0; e < E; ++e) s[e] = col[C::in(lane, e)];
                }
                float2 x[E];
#pragma unroll
                for (int e = 0; e < E; ++e) x[e] = cmul(phi[C::in(lane, e)], s[e]);
                fft<M, E, -1, true>(x, buf, lane, fwd);
#pragma unroll
                for (int e = 0; e < E; ++e) x[e] = cscale(x[e], cabs_hw(x[e]));
                fft<M, E, +1, true, true>(x, buf, lane, inv);   // back to the layout of s
#pragma unroll
                for (int e = 0; e < E; ++e) buf[C::in(lane, e)] = af_term<M>(s[e], x[e], invM);
                __syncthreads();
                const int ncol = min(CF, U - c0);
                if constexpr (Q > 1) {
                    // Q lanes per row: lane q sums sub-chunk q column by column, then every lane adds
                    // the Q sub-chunk sums in order
                    const int m = tid / Q, q = tid % Q;
                    float2 t = make_float2(0.0f, 0.0f);
                    if (m < M) {
                        const int k1 = min((q + 1) * A::SUB, ncol);
                        for (int k = q * A::SUB; k < k1; ++k) t = cadd(t, bufs[k * lds_padded_size(M) + m]);
                    }
#pragma unroll
                    for (int j = 0; j < Q; ++j) acc[0] = cadd(acc[0], make_float2(__shfl(t.x, j, Q), __shfl(t.y, j, Q)));
                } else {
#pragma unroll
                    for (int i = 0; i < RPT; ++i) {
                        const int m = tid + i * NT;
                        if (m < M) {
                            float2 t = make_float2(0.0f, 0.0f);
                            for (int k = 0; k < ncol; ++k) t = cadd(t, bufs[k * lds_padded_size(M) + m]);
                            acc[i] = cadd(acc[i], t);
                        }
                    }
                }
                __syncthreads();
            }
            if constexpr (Q > 1) {
                const int m = tid / Q;
                if (m < M && tid % Q == 0) {
                    const float a = cabsf_(acc[0]);
                    phi[m] = a > 0.0f ? cscale(acc[0], 1.0f / a) : make_float2(0.0f, 0.0f);
                }
            } else {
#pragma unroll
                for (int i = 0; i < RPT; ++i) {
                    const int m = tid + i * NT;
                    if (m < M) {
                        const float a = cabsf_(acc[i]);
                        phi[m] = a > 0.0f ? cscale(acc[i], 1.0f / a) : make_float2(0.0f, 0.0f);
                    }
                }
            }
            __syncthreads();
        }
    };
    if (J.iterations == 0) {
        // the starting phase as it is
    } else if (U <= CF) {
        const float2* col = su + static_cast<size_t>(g < U ? g : 0) * M;
#pragma unroll
        for (int e = 0; e < E; ++e) s[e] = g < U ? col[C::in(lane, e)] : make_float2(0.0f, 0.0f);
        iterate.template operator()<true>();
    } else {
        iterate.template operator()<false>();
    }
    for (int m = tid; m < M; m += NT) J.phi[static_cast<size_t>(f) * M + m] = phi[m];
    if (J.af_redo && tid == 0) J.dec[f].status &= ~2;
}

// Start of the split and resident forms with the frame's work spread over many workgroups (a
// batch of a few frames leaves most CUs idle under one workgroup per frame): k_af_gather copies
// the selected bins into su as k_autofocus does (same scale exponent, same values), kAfGatherGroups
// workgroups per frame each taking a contiguous share of the (pulse, bin) elements; then
// k_af_bin_doppler forms each pulse's Doppler product of the selected bins (:282) with the
// products added in bin order as k_autofocus adds them, into rowdop, which is free once the bins
// are selected; k_af_start then forms the start phase from it. For the resident form
// k_af_gather also empties the frame's exchange words.
constexpr int kAfGatherGroups = 32;

// The exchange words of frame f in the resident form (xwg_word): for iterations 0, 1, 2 modulo 3,
// sub-chunk q < W/SUB and pulse m, the sub-chunk's per-pulse sum. Frame f owns 4 (W/8) M words of
// af_part, the buffer being sized for it.
template <int M>
__device__ __forceinline__ uint64_t* af_words_of(const Job& J, int f, int it) {
    const size_t nq = static_cast<size_t>(J.W / AfCfg<M>::SUB);
    uint64_t* frame = reinterpret_cast<uint64_t*>(J.af_part) + static_cast<size_t>(f) * 4 * (J.W / 8) * M;
    return frame + static_cast<size_t>(it % 3) * nq * M;
}

template <int M>
__global__ __launch_bounds__(256) void k_af_gather(Job J, int resident) {
    HIP_DYNAMIC_SHARED(int, lsel);                                 // W
    float* red = reinterpret_cast<float*>(lsel + J.W);             // 32
    const int f = blockIdx.y, tid = threadIdx.x;
    const int W = J.W;
    const int U = J.dec[f].unit2_num;
    const int* sel = J.sel + static_cast<size_t>(f) * W;
    float cm = 0.0f;
    for (int u = tid; u < U; u += 256) cm = fmaxf(cm, J.colmax[static_cast<size_t>(f) * W + sel[u]]);
    cm = block_max<256>(cm, red);
    const int e = af_scale_exponent(cm);
    for (int u = tid; u < U; u += 256) lsel[u] = sel[u];
    __syncthreads();
    if (resident) {   // the words of the ceil(U / SUB) sub-chunks
        const int words = (U + AfCfg<M>::SUB - 1) / AfCfg<M>::SUB * M;
        for (int i = blockIdx.x * 256 + tid; i < words; i += gridDim.x * 256)
            for (int it = 0; it < 3; ++it) xwg_store(af_words_of<M>(J, f, it) + i, kXwgEmpty);
    }
    const float2* X = J.x + static_cast<size_t>(f) * M * W;
    float2* su = J.su + static_cast<size_t>(f) * W * M;
    const int total = U * M, share = (total + gridDim.x - 1) / gridDim.x;
    const int i0 = blockIdx.x * share, i1 = min(i0 + share, total);
    for (int idx0 = i0 + tid; idx0 < i1; idx0 += 8 * 256) {
        float2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = idx0 + i * 256;
            if (idx < i1) v[i] = X[static_cast<size_t>(idx / U) * W + lsel[idx % U]];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = idx0 + i * 256;
            if (idx < i1) su[static_cast<size_t>(idx % U) * M + idx / U] = make_float2(ldexpf(v[i].x, -e), ldexpf(v[i].y, -e));
        }
    }
}

template <int M>
__global__ __launch_bounds__(256) void k_af_bin_doppler(Job J) {
    const int f = blockIdx.y, m = blockIdx.x * 256 + threadIdx.x;
    if (m >= M - 1) return;
    const int U = J.dec[f].unit2_num;
    const float2* su = J.su + static_cast<size_t>(f) * J.W * M;
    float2 acc = make_float2(0.0f, 0.0f);
    for (int u0 = 0; u0 < U; u0 += 8) {
        float2 a[8], b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (u0 + i < U) {
                a[i] = su[static_cast<size_t>(u0 + i) * M + m];
                b[i] = su[static_cast<size_t>(u0 + i) * M + m + 1];
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (u0 + i < U) acc = cadd(acc, cconjmul(a[i], b[i]));
    }
    J.rowdop[static_cast<size_t>(f) * M + m] = acc;
}

template <int M>
__global__ __launch_bounds__(256) void k_af_start(Job J) {
    HIP_DYNAMIC_SHARED(double, scr);   // M (scan) + 32 (its partial sums), the phase (M float2)
    const int f = blockIdx.x, tid = threadIdx.x;
    float2* phi = reinterpret_cast<float2*>(scr + M + 32);
    if (tid == 0) J.dec[f].status &= ~2;   // of an earlier run's autofocus
    if (J.phi0_given) {
        for (int m = tid; m < M; m += 256) phi[m] = J.phi0_in[static_cast<size_t>(f) * M + m];
        __syncthreads();
    } else {
        doppler_phase<256>(J.rowdop + static_cast<size_t>(f) * M, M, phi, scr, scr + M);
    }
    for (int m = tid; m < M; m += 256) {
        J.phi0[static_cast<size_t>(f) * M + m] = phi[m];
        J.phi[static_cast<size_t>(f) * M + m] = phi[m];
    }
}

// The same fixed-point update with a frame spread over several workgroups, for batches too small
// to fill the GPU with one workgroup per frame. The start kernels gather the selected bins and form
// the starting phase; then iteration `it` is a launch of k_af_cols:
// workgroup (j, f) takes the frame's current phase, transforms sub-chunk j of the selected bins
// and writes its per-pulse sums of conj(S) IFFT(G |G|) (/ M unless M is a power of two, af_term)
// into the iteration's half of af_part.
// The current phase is either formed by every workgroup alike from the previous iteration's sums
// (FOLD: one launch per iteration) or read from J.phi, which k_af_phase writes after each
// iteration (two launches per iteration, no repeated work). The transforms and the summation
// order are those of k_autofocus, so the phases agree bit for bit.
// Unit phasor of pulse m's sum over the nsub sub-chunk sums part[q M + m], added in order.
template <int M>
__device__ __forceinline__ float2 af_phase_from(const float2* part, int nsub, int m) {
    float2 acc = make_float2(0.0f, 0.0f);
    for (int q = 0; q < nsub; q += 8) {   // up to eight loads in flight, added in order
        float2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (q + i < nsub) v[i] = part[static_cast<size_t>(q + i) * M + m];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (q + i < nsub) acc = cadd(acc, v[i]);
    }
    const float a = cabsf_(acc);
    return a > 0.0f ? cscale(acc, 1.0f / a) : make_float2(0.0f, 0.0f);
}

// the half of af_part that iteration `it` writes; frame f's sub-chunk sums in it
template <int M>
__device__ __forceinline__ float2* af_part_of(const Job& J, int f, int it) {
    const size_t per_frame = static_cast<size_t>(J.W / AfCfg<M>::SUB) * M;
    return J.af_part + (static_cast<size_t>(it & 1) * J.K + f) * per_frame;
}

// Twiddle constants of a column's forward and reversed inverse transform.
template <int M>
struct AfTwiddles {
    decltype(fft_twiddles<M, AfCfg<M>::E>(0)) fwd;
    decltype(fft_twiddles<M, AfCfg<M>::E, true>(0)) inv;
    __device__ explicit AfTwiddles(int lane) : fwd(fft_twiddles<M, AfCfg<M>::E>(lane)), inv(fft_twiddles<M, AfCfg<M>::E, true>(lane)) {}
};

// One iteration's work on one sub-chunk of a frame's selected bins: the SUB columns (column
// c0 + tid / TPF in s, first-pass layout, zero where invalid) are multiplied by the phase phi
// (M values), transformed, scaled by |G|, transformed back, multiplied by conj(S) (af_term) and
// left in bufs; then the per-pulse sums over the sub-chunk's ncol columns, each added column by
// column, are handed to put(m, sum). Every thread of the workgroup calls it.
template <int M, typename Put>
__device__ __forceinline__ void af_subchunk(const float2 (&s)[AfCfg<M>::E], const float2* phi,
                                            int ncol, float2* bufs, int tid, const AfTwiddles<M>& tw, Put put) {
    using A = AfCfg<M>;
    using C = ColCfg<M>;
    constexpr int E = A::E, TPF = A::TPF, NTS = A::SUB * TPF;
    const int g = tid / TPF, lane = tid % TPF;
    float2* buf = bufs + g * lds_padded_size(M);
    const float invM = 1.0f / static_cast<float>(M);
    float2 x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = cmul(phi[C::in(lane, e)], s[e]);
    fft<M, E, -1, true>(x, buf, lane, tw.fwd);
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = cscale(x[e], cabs_hw(x[e]));
    fft<M, E, +1, true, true>(x, buf, lane, tw.inv);   // back to the layout of s
#pragma unroll
    for (int e = 0; e < E; ++e) buf[C::in(lane, e)] = af_term<M>(s[e], x[e], invM);
    __syncthreads();
    for (int m = tid; m < M; m += NTS) {
        float2 t = make_float2(0.0f, 0.0f);
        if (ncol == A::SUB) {
#pragma unroll
            for (int k = 0; k < A::SUB; ++k) t = cadd(t, bufs[k * lds_padded_size(M) + m]);
        } else {
            for (int k = 0; k < ncol; ++k) t = cadd(t, bufs[k * lds_padded_size(M) + m]);
        }
        put(m, t);
    }
}

// The sub-chunk of workgroup blockIdx.x of frame f. Only nsub of a frame's gridDim.x (a multiple of 8)
// workgroups have one, and consecutive workgroups go to the eight XCDs in turn, so the first nsub of
// every frame would share the first XCDs: frame f's sub-chunks start f nsub workgroups on.
__device__ __forceinline__ int af_subchunk_of(int f, int nsub) {
    const unsigned G = gridDim.x;
    return static_cast<int>((blockIdx.x + G - (static_cast<unsigned>(f) * static_cast<unsigned>(nsub)) % G) % G);
}

template <int M, bool FOLD>
__global__ __launch_bounds__(AfCfg<M>::SUB * AfCfg<M>::TPF) void k_af_cols(Job J, int it) {
    using A = AfCfg<M>;
    using C = ColCfg<M>;
    constexpr int E = A::E, TPF = A::TPF, SUB = A::SUB, NTS = SUB * TPF;
    HIP_DYNAMIC_SHARED(float2, bufs);   // SUB * lds_padded_size(M), then (FOLD) the phase (M)
    const int f = blockIdx.y, tid = threadIdx.x;
    const int U = J.dec[f].unit2_num;
    const int nsub = (U + SUB - 1) / SUB;
    const int j = af_subchunk_of(f, nsub);
    if (j >= nsub) return;   // the whole workgroup leaves before any barrier
    const int c0 = j * SUB;
    const int W = J.W;
    const float2* phi = J.phi + static_cast<size_t>(f) * M;
    if (FOLD && it > 0) {
        float2* formed = bufs + SUB * lds_padded_size(M);
        const float2* prev = af_part_of<M>(J, f, it - 1);
        for (int m = tid; m < M; m += NTS) formed[m] = af_phase_from<M>(prev, nsub, m);
        __syncthreads();
        phi = formed;
    }
    const int u = c0 + tid / TPF, lane = tid % TPF;
    const bool valid = u < U;
    const float2* col = J.su + static_cast<size_t>(f) * W * M + static_cast<size_t>(valid ? u : 0) * M;
    const AfTwiddles<M> tw(lane);
    float2 s[E];
#pragma unroll
    for (int e = 0; e < E; ++e) s[e] = valid ? col[C::in(lane, e)] : make_float2(0.0f, 0.0f);
    float2* part = af_part_of<M>(J, f, it) + static_cast<size_t>(j) * M;
    af_subchunk<M>(s, phi, min(SUB, U - c0), bufs, tid, tw, [&](int m, float2 t) { part[m] = t; });
}

// Adds n sub-chunk sums of pulse m to acc in order, from exchange words M apart. They are loaded
// together, and all again until none is empty. A thread that has polled more than `limit` times in a
// row gives up (waiting = false) and sets status bit 2; one that waits looks for that bit every
// kAfStatusPolls polls and gives up as well.
constexpr int kAfStatusPolls = 64;
template <int M, int n>
__device__ __forceinline__ void af_add_words(float2& acc, const uint64_t* w, int limit, bool& waiting, int32_t& status) {
    uint64_t v[n];
    for (int polls = 0;; ++polls) {
        bool all = true;
#pragma unroll
        for (int i = 0; i < n; ++i) v[i] = xwg_load(w + i * M);
#pragma unroll
        for (int i = 0; i < n; ++i) all = all && v[i] != kXwgEmpty;
        if (all || !waiting) break;
        if (polls >= limit) {
            waiting = false;
            atomicOr(&status, 2);
            break;
        }
        if (polls % kAfStatusPolls == kAfStatusPolls - 1 && (xwg_load(&status) & 2)) {
            waiting = false;
            break;
        }
        xwg_pause();
    }
#pragma unroll
    for (int i = 0; i < n; ++i) acc = cadd(acc, xwg_value(v[i]));
}

// af_phase_from over exchange words, bit for bit. nsub is a power of two, or 1 (the selected bins are
// a power of two of them).
template <int M>
__device__ __forceinline__ float2 af_phase_from_words(const uint64_t* words, int nsub, int m, int limit, bool& waiting,
                                                      int32_t& status) {
    float2 acc = make_float2(0.0f, 0.0f);
    const uint64_t* w = words + m;
    int q = 0;
    // the other workgroups' sums come about now: a first round that is too early costs its whole latency
    // (with several workgroups on a CU 3 to 8 percent of an iteration)
    xwg_pause();
    xwg_pause();
    for (; q + 4 <= nsub; q += 4) af_add_words<M, 4>(acc, w + static_cast<size_t>(q) * M, limit, waiting, status);
    if (q + 2 <= nsub) {
        af_add_words<M, 2>(acc, w + static_cast<size_t>(q) * M, limit, waiting, status);
        q += 2;
    }
    if (q < nsub) af_add_words<M, 1>(acc, w + static_cast<size_t>(q) * M, limit, waiting, status);
    const float a = cabsf_(acc);
    return a > 0.0f ? cscale(acc, 1.0f / a) : make_float2(0.0f, 0.0f);
}

// The fixed-point iterations of k_af_cols (FOLD) in one launch: workgroup (j, f) keeps sub-chunk
// j of frame f's selected bins in registers for every iteration and hands its per-pulse sums to
// the frame's other workgroups; every workgroup then forms the next phase from all nsub sums, in
// sub-chunk order. The transforms, sums and phases are those of k_af_cols bit for bit.
// The sums travel as 64-bit words that are empty (kXwgEmpty) until they are written, in three buffers
// by iteration modulo 3, all empty at the start (k_af_gather). The thread of pulse m, having read all
// of iteration it, empties its workgroup's word of iteration it - 1, which it + 2 takes next:
// - every reader is done with it: a workgroup writes iteration it only after its barrier behind all
//   reads of it - 1;
// - every reader of it + 2 finds it emptied: it reads there only after this thread's word of it + 1,
//   before whose store the thread has waited for the emptying to be acknowledged (a transform
//   later, so that wait costs nothing).
// All of a frame's workgroups must be resident together; every XCD takes its share of a grid's
// workgroups in order, so where the first incomplete frame lacks one, only complete frames are
// ahead of it, and it completes as those finish. That holds for one such grid on the GPU; two at once can
// each hold what the other's frames lack. So a wait that exceeds J.af_wait_polls polls (a quarter
// of a second by default; a negative bound gives up at once) sets status bit 2 of the frame, which
// k_af_start cleared, and ends its workgroup. Once the bit is set the frame's other workgroups leave too:
// those that wait within kAfStatusPolls polls, those placed later before their first transform. (The words
// they would read are those of an iteration that the leavers never finished: each would wait its own
// bound.) The frame's phase stays the starting phase, and the default form does the frame over with
// k_autofocus. Otherwise workgroup 0 of each frame writes the final phase to J.phi.
// Bound by the latency of an iteration (two transforms by one wave per SIMD, the sums, the
// exchange): 3.6 us at 256 pulses, 6.1 at 512, whether the frames are 1 or 40, as long as every
// workgroup has a CU for itself and the XCDs share the work (af_subchunk_of). At 256 pulses the
// transforms and products take 5500 cycles, the sums 700 and the exchange, which the number of load
// instructions decides, 1700; with a tag in every word, so twice as many loads, 2500.
template <int M>
__global__ __launch_bounds__(AfCfg<M>::SUB * AfCfg<M>::TPF) void k_af_resident(Job J, int least, int most) {
    using A = AfCfg<M>;
    using C = ColCfg<M>;
    constexpr int E = A::E, TPF = A::TPF, SUB = A::SUB, NTS = SUB * TPF;
    HIP_DYNAMIC_SHARED(float2, bufs);   // SUB * lds_padded_size(M), then the phase (M) and a flag
    float2* phi = bufs + SUB * lds_padded_size(M);
    int* const gone = reinterpret_cast<int*>(phi + M);   // the workgroup leaves
    const int f = blockIdx.y, tid = threadIdx.x;
    const int U = J.dec[f].unit2_num;
    const int nsub = (U + SUB - 1) / SUB;
    if (nsub < least || nsub > most) return;   // another launch's frame
    const int j = af_subchunk_of(f, nsub);
    if (j >= nsub) return;   // the whole workgroup leaves before any barrier
    const int c0 = j * SUB;
    const int W = J.W;
    const int u = c0 + tid / TPF, lane = tid % TPF;
    const bool valid = u < U;
    const float2* col = J.su + static_cast<size_t>(f) * W * M + static_cast<size_t>(valid ? u : 0) * M;
    int32_t& status = J.dec[f].status;
    if (tid == 0) {
        if (J.af_wait_polls < 0) atomicOr(&status, 2);   // a negative bound: every wait gives up
        *gone = (xwg_load(&status) & 2) != 0;
    }
    const AfTwiddles<M> tw(lane);
    float2 s[E];
#pragma unroll
    for (int e = 0; e < E; ++e) s[e] = valid ? col[C::in(lane, e)] : make_float2(0.0f, 0.0f);
    for (int m = tid; m < M; m += NTS) phi[m] = J.phi[static_cast<size_t>(f) * M + m];
    __syncthreads();
    if (*gone) return;       // the whole workgroup
    bool waiting = true;     // false once this thread has given up
    for (int it = 0; it < J.iterations; ++it) {
        uint64_t* const words = af_words_of<M>(J, f, it);
        uint64_t* const old = af_words_of<M>(J, f, it + 2) + static_cast<size_t>(j) * M;   // iteration it - 1
        af_subchunk<M>(s, phi, min(SUB, U - c0), bufs, tid, tw, [&](int m, float2 t) {
            if (m == tid) xwg_stores_done();   // the words emptied an iteration ago
            xwg_store(words + static_cast<size_t>(j) * M + m, xwg_word(t));
        });
        for (int m = tid; m < M; m += NTS) {
            phi[m] = af_phase_from_words<M>(words, nsub, m, J.af_wait_polls, waiting, status);
            xwg_store(old + m, kXwgEmpty);
        }
        if (!waiting) *gone = 1;
        __syncthreads();
        if (*gone) return;   // the next write is behind af_subchunk's barrier
    }
    if (j == 0)
        for (int m = tid; m < M; m += NTS) J.phi[static_cast<size_t>(f) * M + m] = phi[m];
}

template <int M>
__global__ __launch_bounds__(256) void k_af_phase(Job J, int it) {
    using A = AfCfg<M>;
    const int f = blockIdx.y, m = blockIdx.x * 256 + threadIdx.x;
    if (m >= M) return;
    const int nsub = (J.dec[f].unit2_num + A::SUB - 1) / A::SUB;
    J.phi[static_cast<size_t>(f) * M + m] = af_phase_from<M>(af_part_of<M>(J, f, it), nsub, m);
}

// ------------------------------------------------------------------------------------------
namespace {
template <int M>
size_t af_cols_lds(bool fold) {
    return (static_cast<size_t>(AfCfg<M>::SUB) * lds_padded_size(M) + (fold ? M : 0)) * sizeof(float2);
}
template <int M>
constexpr size_t kAfResidentNeed = (static_cast<size_t>(AfCfg<M>::SUB) * lds_padded_size(M) + M) * sizeof(float2) + sizeof(int);
// Resident workgroups that a CU can hold: 16 waves of at most 128 vector registers (384 pulses take 134: 12
// waves), and their LDS.
template <int M>
constexpr int kAfResidentFit = std::min((M == 384 ? 12 : 16) / ((AfCfg<M>::SUB * AfCfg<M>::TPF + 63) / 64),
                                        static_cast<int>(kLdsBytes / kAfResidentNeed<M>));
template <int M>
size_t colfft_lds() {
    using C = ColCfg<M>;
    const size_t work = std::max(static_cast<size_t>(M) * (C::CT + 1), static_cast<size_t>(C::CT) * lds_padded_size(M));
    return work * sizeof(float2);
}
template <int M>
size_t autofocus_lds() {
    using A = AfCfg<M>;
    return 2 * M * sizeof(float2) + (M + A::NT) * sizeof(double) + static_cast<size_t>(A::CF) * lds_padded_size(M) * sizeof(float2);
}
size_t select_lds(int W) { return (3 * W + 32) * sizeof(int); }
}  // namespace

#define ISAR_PULSE_SWITCH(M, BODY)                       \
    switch (M) {                                         \
    case 64: { constexpr int MM = 64; BODY; } break;     \
    case 128: { constexpr int MM = 128; BODY; } break;   \
    case 192: { constexpr int MM = 192; BODY; } break;   \
    case 256: { constexpr int MM = 256; BODY; } break;   \
    case 384: { constexpr int MM = 384; BODY; } break;   \
    case 512: { constexpr int MM = 512; BODY; } break;   \
    case 1024: { constexpr int MM = 1024; BODY; } break; \
    default: break;                                      \
    }

bool pulse_count_supported(int M) {
    return M == 64 || M == 128 || M == 192 || M == 256 || M == 384 || M == 512 || M == 1024;
}

hipError_t configure_pa_kernels() {
    hipError_t err = hipSuccess;
#ifndef ISAR_EMU
    auto set = [&](const void* fn, size_t bytes) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        if (e != hipSuccess) {
            err = e;
            report_config_error(__FILE__, bytes);
        }
    };
#define ISAR_SET_PA(MM)                                                          \
    set(reinterpret_cast<const void*>(&k_pa_colfft<MM>), colfft_lds<MM>());      \
    set(reinterpret_cast<const void*>(&k_autofocus<MM>), autofocus_lds<MM>());   \
    set(reinterpret_cast<const void*>(&k_af_cols<MM, true>), af_cols_lds<MM>(true));   \
    set(reinterpret_cast<const void*>(&k_af_cols<MM, false>), af_cols_lds<MM>(false));   \
    set(reinterpret_cast<const void*>(&k_af_resident<MM>), std::max(kAfResidentNeed<MM>, kLdsBytes / 2 + 1024));
    ISAR_SET_PA(64) ISAR_SET_PA(128) ISAR_SET_PA(192) ISAR_SET_PA(256) ISAR_SET_PA(384) ISAR_SET_PA(512)
    ISAR_SET_PA(1024)
#undef ISAR_SET_PA
#endif
    return err;
}

void launch_pa_colfft(const Job& J, hipStream_t s) {
    ISAR_PULSE_SWITCH(J.M, ISAR_LAUNCH(k_pa_doppler<MM>, dim3(J.K), dim3(256), (MM + 32) * sizeof(double), s, J));
    ISAR_PULSE_SWITCH(J.M, ISAR_LAUNCH(k_pa_colfft<MM>, dim3(J.W / ColCfg<MM>::CT, J.K), dim3(ColCfg<MM>::NT),
                                       colfft_lds<MM>(), s, J));
}
void launch_pa_select(const Job& J, hipStream_t s) {
    if (J.W == kRangeCut) ISAR_LAUNCH(k_pa_select<kRangeCut>, dim3(J.K), dim3(kRangeCut), select_lds(J.W), s, J);
}
void launch_autofocus(const Job& J, hipStream_t s) {
    ISAR_PULSE_SWITCH(J.M, ISAR_LAUNCH(k_autofocus<MM>, dim3(J.K), dim3(AfCfg<MM>::NT), autofocus_lds<MM>(), s, J));
}
namespace {
// The start phase and the gathered bins of the split and resident forms (k_af_gather,
// k_af_bin_doppler, k_af_start).
template <int MM>
void autofocus_start_spread(const Job& J, bool resident, hipStream_t s) {
    ISAR_LAUNCH(k_af_gather<MM>, dim3(kAfGatherGroups, J.K), dim3(256), J.W * sizeof(int) + 32 * sizeof(float), s, J,
                resident ? 1 : 0);
    if (!J.phi0_given) ISAR_LAUNCH(k_af_bin_doppler<MM>, dim3((MM - 1 + 255) / 256, J.K), dim3(256), 0, s, J);
    ISAR_LAUNCH(k_af_start<MM>, dim3(J.K), dim3(256), (MM + 32) * sizeof(double) + MM * sizeof(float2), s, J);
}

template <int MM>
void autofocus_split(const Job& J, bool fold, hipStream_t s) {
    autofocus_start_spread<MM>(J, false, s);
    constexpr int SUB = AfCfg<MM>::SUB;
    const dim3 cols_grid(J.W / SUB, J.K);
    const dim3 cols_block(SUB * AfCfg<MM>::TPF);
    const dim3 phase_grid((MM + 255) / 256, J.K);
    for (int it = 0; it < J.iterations; ++it) {
        if (fold) {
            ISAR_LAUNCH((k_af_cols<MM, true>), cols_grid, cols_block, af_cols_lds<MM>(true), s, J, it);
        } else {
            ISAR_LAUNCH((k_af_cols<MM, false>), cols_grid, cols_block, af_cols_lds<MM>(false), s, J, it);
            ISAR_LAUNCH(k_af_phase<MM>, phase_grid, dim3(256), 0, s, J, it);
        }
    }
    if (fold && J.iterations > 0) ISAR_LAUNCH(k_af_phase<MM>, phase_grid, dim3(256), 0, s, J, J.iterations - 1);
}
}  // namespace

void launch_autofocus_split(const Job& J, bool fold, hipStream_t s) {
    ISAR_PULSE_SWITCH(J.M, autofocus_split<MM>(J, fold, s));
}

namespace {
template <int MM>
void autofocus_resident(const Job& J, bool guarded, hipStream_t s) {
    autofocus_start_spread<MM>(J, true, s);
    if (J.iterations > 0) {
        constexpr int SUB = AfCfg<MM>::SUB;
        const AfResidentShapes shapes = af_resident_shapes(J.K, SUB, kAfResidentNeed<MM>, kAfResidentFit<MM>);
        for (int i = 0; i < shapes.n; ++i)
            ISAR_LAUNCH_RESIDENT(k_af_resident<MM>, dim3(J.W / SUB, J.K), dim3(SUB * AfCfg<MM>::TPF), shapes.shape[i].lds, s,
                                 J, i ? shapes.shape[0].sub_chunks + 1 : 1, shapes.shape[i].sub_chunks);
        if (guarded) {
            Job redo = J;
            redo.af_redo = 1;
            ISAR_LAUNCH(k_autofocus<MM>, dim3(J.K), dim3(AfCfg<MM>::NT), autofocus_lds<MM>(), s, redo);
        }
    }
}
}  // namespace

void launch_autofocus_resident(const Job& J, bool guarded, hipStream_t s) {
    ISAR_PULSE_SWITCH(J.M, autofocus_resident<MM>(J, guarded, s));
}

}  // namespace isar
