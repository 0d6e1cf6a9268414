// nn.hip — kernels of the learned autofocus warm start: a small multilayer perceptron with BF16
// weights and FP32 accumulation on the matrix cores (gfx950's v_mfma_f32_16x16x32_bf16), its backward
// pass and Adam update, and the per-pulse phase features it reads and writes.
//
// There is no counterpart in the reference: the network seeds fast-entropy autofocus
// (phase_adjustment.cu:282-324) with a predicted per-pulse phase; the plain iteration still runs
// from that start and remains the judge of the result.
#include "../dev_common.hpp"
#include "../launchers.hpp"

namespace isar {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bfloat16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ short to_bf16(float f) {
    unsigned u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return static_cast<short>(u >> 16);
}
__device__ __forceinline__ __bf16 bits_bf16(short s) { return __builtin_bit_cast(__bf16, s); }
__device__ __forceinline__ short as_bf16(float f) { return to_bf16(f); }
__device__ __forceinline__ short as_bf16(uint16_t b) { return static_cast<short>(b); }

// D = A B + C for one 16 x 16 x 32 tile. Lane l holds A[l % 16][8 (l / 16) + t] and
// B[8 (l / 16) + t][l % 16] for t < 8, and D[4 (l / 16) + t][l % 16] for t < 4.
__device__ __forceinline__ f32x4 mfma16x32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Eight consecutive k of one row (or column) of an operand as they are in memory. VEC: they are
// consecutive there and aligned to their size (16 bytes at most a load), and k is a multiple of 8.
// Nothing outside the operand is read: where line >= lines or kk >= k the last one inside is, and the
// values of kk >= k become zeros.
template <typename T, bool VEC>
struct Frag {
    static constexpr int kWords = VEC ? static_cast<int>(8 * sizeof(T) / 16) : 8;
    typename std::conditional<VEC, uint4, T>::type v[kWords];
    __device__ __forceinline__ void load(const T* p, int line, int lines, long s_line, int kk, int k, long s_k) {
        p += min(line, lines - 1) * s_line;
        if constexpr (VEC) {
            const uint4* q = reinterpret_cast<const uint4*>(p + min(kk, k - 8));
#pragma unroll
            for (int i = 0; i < kWords; ++i) v[i] = q[i];
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = p[min(kk + t, k - 1) * s_k];
        }
    }
    // the eight added in order, those of kk >= k left out
    __device__ __forceinline__ float sum(int kk, int k) const {
        static_assert(!VEC, "single loads");
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) s += kk + t < k ? v[t] : 0.0f;
        return s;
    }
    __device__ __forceinline__ bf16x8 get(int kk, int k) const {
        T e[8];
        if constexpr (VEC) __builtin_memcpy(e, v, sizeof e);
        else {
#pragma unroll
            for (int t = 0; t < 8; ++t) e[t] = v[t];
        }
        bf16x8 r;
#pragma unroll
        for (int t = 0; t < 8; ++t) r[t] = bits_bf16(kk + t < k ? as_bf16(e[t]) : static_cast<short>(0));
        return r;
    }
};

template <typename TA, typename TB>
struct GemmArgs {
    int m, n, k;
    const TA* a;
    long sam, sak;
    const TB* b;
    long sbk, sbn;
    float* c;
    long scm;
    const float* bias;
    const float* mask;
    long smm;
    float* colsum;
};

// C[m][n] = sum_k A(m, k) B(k, n) with A(m, k) = a[m sam + k sak], B(k, n) = b[k sbk + n sbn],
// operands rounded to BF16, products accumulated in FP32 in the order of k. One wave per block of
// 16 T x 16 T of C. Epilogue: 0 store; 1 + bias[n], then max(0, .); 2 + bias[n]; 3 times (mask[m][n] > 0).
// With EPI = 0 the waves of the first row of blocks also add B's columns before rounding, colsum[n] =
// sum_k B(k, n): of the weight gradient's operand dZ that is the bias gradient, which took a launch of
// its own and another pass over dZ (14 of a training step's 159 us).
// AV, BV: the operand's k are consecutive and aligned (Frag).
//
// Bound by the latency of its loads: the matrix work of a layer is under a microsecond, its
// operands are in the L2, and the sums follow k, so that a wave has a serial chain over k. So the
// loads of four steps of 32 k (two for T = 2) are issued together, 16 bytes each where the layout allows,
// and small products take T = 1, four times as many waves (use_small_tiles). The first layer of the
// 256-pulse network, 256 x 128 x 1024, takes 15 us (95 with a step's loads waited for one by one and 32 x 32 tiles),
// the training step's products 61 instead of 406.
template <typename TA, typename TB, int EPI, int T, bool AV, bool BV>
__device__ __forceinline__ void gemm_block(const GemmArgs<TA, TB>& G, int bx, int by) {
    const int m = G.m, n = G.n, k = G.k;
    constexpr int kTile = 16 * T, kSteps = T == 1 ? 4 : 2;
    const int l = threadIdx.x;
    const int bm = by * kTile, bn = bx * kTile;
    const int li = l % 16, lk = 8 * (l / 16), lr = 4 * (l / 16);
    f32x4 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float cs[T];
#pragma unroll
    for (int i = 0; i < T; ++i) cs[i] = 0.0f;
    for (int k0 = 0; k0 < k; k0 += 32 * kSteps) {
        Frag<TA, AV> fa[kSteps][T];
        Frag<TB, BV> fb[kSteps][T];
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int kk = k0 + 32 * q + lk;
#pragma unroll
            for (int i = 0; i < T; ++i) {
                fa[q][i].load(G.a, bm + 16 * i + li, m, G.sam, kk, k, G.sak);
                fb[q][i].load(G.b, bn + 16 * i + li, n, G.sbn, kk, k, G.sbk);
            }
        }
        issue_point();
#pragma unroll
        for (int q = 0; q < kSteps; ++q) {
            const int kk = k0 + 32 * q + lk;
            if (k0 + 32 * q >= k) break;
            bf16x8 va[T], vb[T];
#pragma unroll
            for (int i = 0; i < T; ++i) {
                va[i] = fa[q][i].get(kk, k);
                vb[i] = fb[q][i].get(kk, k);
                if constexpr (EPI == 0) cs[i] += fb[q][i].sum(kk, k);
            }
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j) acc[i][j] = mfma16x32(va[i], vb[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const int col = bn + 16 * j + li;
            if (col >= n) continue;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int row = bm + 16 * i + lr + t;
                if (row >= m) continue;
                float v = acc[i][j][t];
                if constexpr (EPI == 1) v = fmaxf(v + G.bias[col], 0.0f);
                if constexpr (EPI == 2) v += G.bias[col];
                if constexpr (EPI == 3) v = G.mask[row * G.smm + col] > 0.0f ? v : 0.0f;
                G.c[row * G.scm + col] = v;
            }
        }
    if constexpr (EPI == 0) {
        if (by == 0) {
#pragma unroll
            for (int i = 0; i < T; ++i) {   // the four groups of 16 lanes hold every fourth eight of k
                cs[i] += lane_xor<32>(cs[i]);
                cs[i] += lane_xor<16>(cs[i]);
                const int col = bn + 16 * i + li;
                if (l < 16 && col < n) G.colsum[col] = cs[i];
            }
        }
    }
}

}  // namespace

template <typename TA, typename TB, int EPI, int T, bool AV, bool BV>
__global__ __launch_bounds__(64) void k_gemm_bf16(GemmArgs<TA, TB> G) {
    gemm_block<TA, TB, EPI, T, AV, BV>(G, blockIdx.x, blockIdx.y);
}

// The two products of a layer's backward pass that read dZ and do not depend on each other, in one
// launch: the first `first` workgroups form the weight (and bias) gradient, across_dw to a row of
// blocks, the rest dZ W^T.
template <bool VEC>
__global__ __launch_bounds__(64) void k_gemm_backward(GemmArgs<float, float> dw, GemmArgs<float, uint16_t> dx, int first,
                                                      int across_dw, int across_dx) {
    const int b = blockIdx.x;
    if (b < first) gemm_block<float, float, 0, 1, false, false>(dw, b % across_dw, b / across_dw);
    else gemm_block<float, uint16_t, 3, 1, VEC, VEC>(dx, (b - first) % across_dx, (b - first) / across_dx);
}

// Adam (bias-corrected) on FP32 master parameters; the BF16 copy of each weight follows.
__global__ void k_adam(int n, float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, uint16_t* __restrict__ pb, const int* __restrict__ bf_index,
                       float lr, float beta1, float beta2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = beta1 * m1[i] + (1.0f - beta1) * gi;
    const float b = beta2 * m2[i] + (1.0f - beta2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float v = p[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    p[i] = v;
    const int bi = bf_index[i];
    if (bi >= 0) pb[bi] = static_cast<uint16_t>(to_bf16(v));
}

// BF16 copies of the weights from the FP32 master parameters
__global__ void k_to_bf16(int n, const float* __restrict__ p, uint16_t* __restrict__ pb,
                          const int* __restrict__ bf_index) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int bi = bf_index[i];
    if (bi >= 0) pb[bi] = static_cast<uint16_t>(to_bf16(p[i]));
}

// mean squared error over rows x cols and its gradient 2 (pred - target) / (rows cols)
__global__ void k_mse(int rows, int cols, const float* __restrict__ pred, const float* __restrict__ target,
                      float* __restrict__ grad, double* __restrict__ loss) {
    __shared__ double red[256];
    const int r = blockIdx.x, tid = threadIdx.x;
    const float scale = 2.0f / (static_cast<float>(rows) * static_cast<float>(cols));
    double s = 0.0;
    for (int j = tid; j < cols; j += blockDim.x) {
        const size_t i = static_cast<size_t>(r) * cols + j;
        const float d = pred[i] - target[i];
        if (grad) grad[i] = scale * d;
        s += static_cast<double>(d) * d;
    }
    red[tid] = s;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    if (tid == 0) loss[r] = red[0] / (static_cast<double>(rows) * cols);
}

// Per-pulse phase change between two autofocus phases: out[f stride + 2m] + j out[f stride + 2m+1]
// = phi_b[f][m] conj(phi_a[f][m]).
__global__ void k_phase_change(int frames, int M, const float2* __restrict__ phi_a, const float2* __restrict__ phi_b,
                               float* __restrict__ out, int stride) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= frames * M) return;
    const int f = i / M, m = i % M;
    const float2 v = cmulc(phi_b[i], phi_a[i]);
    float* o = out + static_cast<size_t>(f) * stride + 2 * m;
    o[0] = v.x;
    o[1] = v.y;
}

// Warm start phi_w = phi_b * unit(pred); a zero prediction keeps phi_b.
__global__ void k_compose_phase(int frames, int M, const float2* __restrict__ phi_b, const float* __restrict__ pred,
                                float2* __restrict__ phi_w) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= frames * M) return;
    const float2 q = make_float2(pred[2 * static_cast<size_t>(i)], pred[2 * static_cast<size_t>(i) + 1]);
    const float a = cabsf_(q);
    phi_w[i] = a > 0.0f ? cmul(phi_b[i], cscale(q, 1.0f / a)) : phi_b[i];
}

// Per frame, the starting phase whose image entropy is lower: out = ent_b < ent_a ? phi_b : phi_a
// (ties keep phi_a); ent_out (optional) receives the entropy of the phase kept.
__global__ void k_select_phase(int frames, int M, const float2* __restrict__ phi_a, const double* __restrict__ ent_a,
                               const float2* __restrict__ phi_b, const double* __restrict__ ent_b,
                               float2* __restrict__ out, double* __restrict__ ent_out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= frames * M) return;
    const int f = i / M;
    const bool take_b = ent_b[f] < ent_a[f];
    out[i] = take_b ? phi_b[i] : phi_a[i];
    if (ent_out && i % M == 0) ent_out[f] = take_b ? ent_b[f] : ent_a[f];
}

// The final judgement of a learned result: per frame, out = img_b (the learned image) when its
// entropy is no worse than img_a's (the plain result) within rel_tol, else img_a; accepted[f]
// records the choice. out may alias either input.
__global__ void k_accept_image(int frames, int n, const float* __restrict__ img_a, const double* __restrict__ ent_a,
                               const float* img_b, const double* __restrict__ ent_b, double rel_tol, float* out,
                               int32_t* __restrict__ accepted) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<long long>(frames) * n) return;
    const int f = static_cast<int>(i / n);
    const bool take_b = ent_b[f] <= ent_a[f] * (1.0 + rel_tol);
    out[i] = take_b ? img_b[i] : img_a[i];
    if (accepted && i % n == 0) accepted[f] = take_b ? 1 : 0;
}

// Half step from phi_a toward phi_b: out = phi_a * sqrt(unit(phi_b conj(phi_a))), the square root
// taken on the shorter arc (unit(1 + c)); an exactly opposite pair turns by +pi/2.
__global__ void k_half_phase(int frames, int M, const float2* __restrict__ phi_a, const float2* __restrict__ phi_b,
                             float2* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= frames * M) return;
    const float2 a = phi_a[i];
    float2 c = cconjmul(a, phi_b[i]);                  // phi_b conj(phi_a)
    const float cm = cabsf_(c);
    c = cm > 0.0f ? cscale(c, 1.0f / cm) : make_float2(1.0f, 0.0f);
    float2 h = make_float2(1.0f + c.x, c.y);
    const float hm = cabsf_(h);
    h = hm > 1e-20f ? cscale(h, 1.0f / hm) : make_float2(0.0f, 1.0f);
    out[i] = cmul(a, h);
}

// ln(q / 2^(k - 1023)) of a positive normal double to about 2e-16 (absolute, beside the rounding of the
// result) by table and series: with the mantissa in [1, 2) cut into 128 intervals, c_j about the
// reciprocal of interval j's centre and r = mantissa c_j - 1, at most 1/256 in magnitude,
// ln q = e ln 2 - ln c_j + ln(1 + r). (P. T. P. Tang, "Table-driven implementation of the logarithm
// function in IEEE floating-point arithmetic", 1990.)
struct LogRow {
    double c, ln_c;   // c_j and -ln c_j
};
struct LogTable {
    LogRow row[128];
    constexpr LogTable() : row() {
        for (int j = 0; j < 128; ++j) {
            const double c = 1.0 / (1.0 + (j + 0.5) / 128.0);
            // -ln c = 2 artanh(z), z = (1 - c) / (1 + c) <= 1/3
            const double z = (1.0 - c) / (1.0 + c), z2 = z * z;
            double term = z, sum = 0.0;
            for (int i = 1; i < 40; i += 2) {
                sum += term / i;
                term *= z2;
            }
            row[j] = LogRow{c, 2.0 * sum};
        }
    }
};
__constant__ const LogTable kLogTable{};

constexpr double kLn2 = 0.69314718055994530942;
__device__ __forceinline__ int biased_exponent(double q) {   // q >= 0
    return static_cast<int>(__builtin_bit_cast(uint64_t, q) >> 52);
}
__device__ __forceinline__ double log_by_table(double q, int k, const LogRow* rows) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, q);
    const unsigned hi = static_cast<unsigned>(bits >> 32);
    const LogRow t = rows[(hi >> 13) & 127];
    const uint64_t mb = (static_cast<uint64_t>((hi & 0x000fffffu) | 0x3ff00000u) << 32) | (bits & 0xffffffffu);
    const double r = fma(__builtin_bit_cast(double, mb), t.c, -1.0);
    const double e = static_cast<double>(static_cast<int>(hi >> 20) - k);
    double y = fma(r, -1.0 / 6.0, 1.0 / 5.0);   // the next term is below 2e-18
    y = fma(y, r, -1.0 / 4.0);
    y = fma(y, r, 1.0 / 3.0);
    y = fma(y, r, -0.5);
    y = fma(y * r, r, r);
    return fma(e, kLn2, t.ln_c) + y;
}

// Image entropy -sum p ln p, p = q / T, q = img^2, T = sum q, one workgroup per image, FP64 sums, one pass
// over the image: (T ln(T / r) - sum q ln(q / r)) / T for any r. With r = 1 both terms grow with ln T and
// nearly cancel (amplitudes of 1e4: off by 7e-15, where -sum p ln p is off by 6e-16). So r is the power
// of two of the largest q so far, per thread and then for all: raising it by 2^d takes T d ln 2 from the
// second sum, and the terms that count have q near r. Off by as much as -sum p ln p or less
// (131072 cells, amplitudes 1e-15 to 1e15), and the same bits for an image scaled by a power of two.
// A single bright cell gives 0 exactly, as both terms are then the same product. Bound by the loads'
// latency and FP64 issue: 256 images of 256 x 512 take 33 us (4.1 TB/s), 1024 of them 116; 32 and 113
// with r = 1; the 1024 132 with the registers left free, as a CU then holds one workgroup; 390 the 256 in
// two passes with the library's logarithm.
struct EntropySums {
    double total, s;
    int k;   // biased exponent of r; 0: no q yet
    __device__ __forceinline__ void raise(int to) {
        if (to <= k) return;
        s = fma(total, static_cast<double>(k - to) * kLn2, s);
        k = to;
    }
    __device__ __forceinline__ void add(double q, const LogRow* rows) {   // q is a float's square: normal or 0
        total += q;
        s = fma(q, log_by_table(q, k, rows), s);   // 0 where q = 0: the logarithm is finite there
    }
};
template <int NT>
__global__ __launch_bounds__(NT, 8) void k_image_entropy(int n, const float* __restrict__ img, double* __restrict__ out) {
    constexpr int WAVES = NT / 64;
    __shared__ LogRow rows[128];
    __shared__ EntropySums red[WAVES];
    const int f = blockIdx.x, tid = threadIdx.x;
    const float* x = img + static_cast<size_t>(f) * n;
    if (tid < 128) rows[tid] = kLogTable.row[tid];
    __syncthreads();
    EntropySums a{0.0, 0.0, 0};
    auto square = [](float v) { return static_cast<double>(v) * v; };
    constexpr int kLoads = 8;
    int i = tid;
    for (; i + (kLoads - 1) * NT < n; i += kLoads * NT) {
        float v[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) v[u] = x[i + u * NT];
        issue_point();
        float top = 0.0f;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) top = fmaxf(top, fabsf(v[u]));
        a.raise(biased_exponent(square(top)));
#pragma unroll
        for (int u = 0; u < kLoads; ++u) a.add(square(v[u]), rows);
    }
    for (; i < n; i += NT) {
        const double q = square(x[i]);
        a.raise(biased_exponent(q));
        a.add(q, rows);
    }
    auto combine = [&]<int WIDTH>() {
        a.raise(group_combine<WIDTH>(a.k, [](int p, int q) { return max(p, q); }));
        a.total = group_combine<WIDTH>(a.total, [](double p, double q) { return p + q; });
        a.s = group_combine<WIDTH>(a.s, [](double p, double q) { return p + q; });
    };
    combine.template operator()<64>();
    if (tid % 64 == 0) red[tid / 64] = a;
    __syncthreads();
    if (tid >= 64) return;
    a = red[tid % WAVES];
    combine.template operator()<WAVES>();
    if (tid == 0) {
        // no entropy where the image is all zero, or its energy infinite or NaN; the difference's
        // rounding may leave a hair below 0
        const bool any = a.total > 0.0 && a.total <= 1.7976931348623157e308;
        const double tl = opaque(a.total * log_by_table(a.total, a.k, rows));   // rounded by itself, as s is
        out[f] = any ? fmax((tl - a.s) / a.total, 0.0) : 0.0;
    }
}

// ------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------
namespace {
// 16 x 16 tiles until 32 x 32 tiles give every SIMD a wave; above, the larger tiles read each operand
// half as often. 1024 x 2048 x 128 (2048 tiles of 32 x 32) takes 9.9 us in the larger and 14.5 in the
// smaller tiles, 2048 x 128 x 512 (256) 17.5 and 13.3, 1024 x 128 x 4096 (128) 84 and 52; at 512 tiles
// it depends on k (31 and 36 us at k = 1024, 7.0 and 6.0 at 128).
bool use_small_tiles(int m, int n) {
    return static_cast<long long>((m + 31) / 32) * ((n + 31) / 32) < 4 * kComputeUnits;
}

// Whether the eight k of a fragment can be read as 16-byte words.
template <typename T>
bool vector_k(const T* p, long s_k, long s_line, int k) {
    constexpr long per = 16 / static_cast<long>(sizeof(T));
    return s_k == 1 && s_line % per == 0 && k % 8 == 0 && reinterpret_cast<uintptr_t>(p) % 16 == 0;
}

// AK, BK: the callers' layouts have consecutive k in that operand; both must be readable so, or
// neither is.
template <bool AK, bool BK, typename TA, typename TB>
bool vector_both(const GemmArgs<TA, TB>& G) {
    return (AK || BK) && (!AK || vector_k(G.a, G.sak, G.sam, G.k)) && (!BK || vector_k(G.b, G.sbk, G.sbn, G.k));
}
template <typename TA, typename TB, int EPI, bool AK, bool BK>
void gemm_bf16(const GemmArgs<TA, TB>& G, hipStream_t s) {
    const bool small = use_small_tiles(G.m, G.n), vec = vector_both<AK, BK>(G);
    const int tile = small ? 16 : 32;
    const dim3 grid((G.n + tile - 1) / tile, (G.m + tile - 1) / tile);
#define ISAR_GEMM(T, AV, BV) ISAR_LAUNCH((k_gemm_bf16<TA, TB, EPI, T, AV, BV>), grid, dim3(64), 0, s, G)
    if (vec) {
        if (small) ISAR_GEMM(1, AK, BK);
        else ISAR_GEMM(2, AK, BK);
    } else {
        if (small) ISAR_GEMM(1, false, false);
        else ISAR_GEMM(2, false, false);
    }
#undef ISAR_GEMM
}
}  // namespace

void launch_dense_forward(int batch, int in, int out, const float* a, const uint16_t* w, const float* bias, float* z,
                          int relu, hipStream_t s) {
    const GemmArgs<float, uint16_t> G{batch, out, in, a, in, 1, w, out, 1, z, out, bias, nullptr, 0, nullptr};
    if (relu) gemm_bf16<float, uint16_t, 1, true, false>(G, s);
    else gemm_bf16<float, uint16_t, 2, true, false>(G, s);
}
void launch_dense_backward(int batch, int in, int out, const float* a, const float* dz, const uint16_t* w, float* dw,
                           float* db, float* da, hipStream_t s) {
    // dW = A^T dZ (in x out), db = column sums of dZ; dA = dZ W^T where A > 0
    const GemmArgs<float, float> W{in, out, batch, a, 1, in, dz, out, 1, dw, out, nullptr, nullptr, 0, db};
    if (!da) {
        gemm_bf16<float, float, 0, false, false>(W, s);
        return;
    }
    const GemmArgs<float, uint16_t> A{batch, in, out, dz, out, 1, w, 1, out, da, in, nullptr, a, in, nullptr};
    // One launch while both take 16 x 16 tiles: a layer of the 256-pulse network at batch 256 takes 6.5 us, two
    // launches took 10.5.
    if (use_small_tiles(W.m, W.n) && use_small_tiles(A.m, A.n)) {
        const int xw = (W.n + 15) / 16, xa = (A.n + 15) / 16;
        const int first = xw * ((W.m + 15) / 16), rest = xa * ((A.m + 15) / 16);
        if (vector_both<true, true>(A))
            ISAR_LAUNCH(k_gemm_backward<true>, dim3(first + rest), dim3(64), 0, s, W, A, first, xw, xa);
        else
            ISAR_LAUNCH(k_gemm_backward<false>, dim3(first + rest), dim3(64), 0, s, W, A, first, xw, xa);
        return;
    }
    gemm_bf16<float, float, 0, false, false>(W, s);
    gemm_bf16<float, uint16_t, 3, true, true>(A, s);
}
void launch_adam(int n, float* p, const float* g, float* m1, float* m2, uint16_t* pb, const int* bf_index, float lr,
                 float beta1, float beta2, float eps, float c1, float c2, hipStream_t s) {
    ISAR_LAUNCH(k_adam, dim3((n + 255) / 256), dim3(256), 0, s, n, p, g, m1, m2, pb, bf_index, lr, beta1, beta2, eps,
                c1, c2);
}
void launch_to_bf16(int n, const float* p, uint16_t* pb, const int* bf_index, hipStream_t s) {
    ISAR_LAUNCH(k_to_bf16, dim3((n + 255) / 256), dim3(256), 0, s, n, p, pb, bf_index);
}
void launch_mse(int rows, int cols, const float* pred, const float* target, float* grad, double* loss, hipStream_t s) {
    ISAR_LAUNCH(k_mse, dim3(rows), dim3(256), 0, s, rows, cols, pred, target, grad, loss);
}
void launch_phase_change(int frames, int M, const float2* a, const float2* b, float* out, int stride, hipStream_t s) {
    ISAR_LAUNCH(k_phase_change, dim3((frames * M + 255) / 256), dim3(256), 0, s, frames, M, a, b, out, stride);
}
void launch_compose_phase(int frames, int M, const float2* phi_b, const float* pred, float2* phi_w, hipStream_t s) {
    ISAR_LAUNCH(k_compose_phase, dim3((frames * M + 255) / 256), dim3(256), 0, s, frames, M, phi_b, pred, phi_w);
}
void launch_select_phase(int frames, int M, const float2* phi_a, const double* ent_a, const float2* phi_b,
                         const double* ent_b, float2* out, double* ent_out, hipStream_t s) {
    ISAR_LAUNCH(k_select_phase, dim3((frames * M + 255) / 256), dim3(256), 0, s, frames, M, phi_a, ent_a, phi_b, ent_b,
                out, ent_out);
}
void launch_half_phase(int frames, int M, const float2* phi_a, const float2* phi_b, float2* out, hipStream_t s) {
    ISAR_LAUNCH(k_half_phase, dim3((frames * M + 255) / 256), dim3(256), 0, s, frames, M, phi_a, phi_b, out);
}
void launch_accept_image(int frames, int n, const float* img_a, const double* ent_a, const float* img_b,
                         const double* ent_b, double rel_tol, float* out, int32_t* accepted, hipStream_t s) {
    const long long total = static_cast<long long>(frames) * n;
    ISAR_LAUNCH(k_accept_image, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, s, frames, n, img_a,
                ent_a, img_b, ent_b, rel_tol, out, accepted);
}
// 1024 threads an image from 8192 cells on, where every thread has a whole group of loads, 256 below:
// 2000 images of 100 cells take 4.5 us (10.4 with 1024 threads), 1024 of 1000 cells 4.4 (6.1), of 8192
// cells 10.1 (11.3); but one image of 16384 cells 7.0 (5.5), 256 of 32768 14 (10).
constexpr int kEntropyWideCells = 8192;
void launch_image_entropy(int frames, int n, const float* img, double* out, hipStream_t s) {
    if (n < kEntropyWideCells) ISAR_LAUNCH(k_image_entropy<256>, dim3(frames), dim3(256), 0, s, n, img, out);
    else ISAR_LAUNCH(k_image_entropy<1024>, dim3(frames), dim3(1024), 0, s, n, img, out);
}

}  // namespace isar
