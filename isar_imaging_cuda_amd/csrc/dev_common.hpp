// dev_common.hpp — device primitives for the gfx950 imaging kernels: complex arithmetic,
// wave64/workgroup reductions, exact phase generation and an LDS-resident Stockham FFT.
#pragma once

#include "pipeline_types.hpp"

namespace isar {

// ------------------------------------------------------------------------------------------
// complex float helpers (float2 = re, im)
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {
    return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
// conj(a) * b
__device__ __forceinline__ float2 cconjmul(float2 a, float2 b) {
    return make_float2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float cabs2(float2 a) { return a.x * a.x + a.y * a.y; }
__device__ __forceinline__ float cabsf_(float2 a) { return sqrtf(a.x * a.x + a.y * a.y); }
// Square root by the hardware instruction alone (within 1 ulp). sqrtf compiles to that
// instruction plus about 15 more for correct rounding; where a square root is taken per element
// inside FP32 transforms, that expansion costs more issue slots than it buys accuracy.
__device__ __forceinline__ float sqrt_hw(float v) {
#ifdef ISAR_EMU
    return sqrtf(v);
#else
    return __builtin_amdgcn_sqrtf(v);
#endif
}
__device__ __forceinline__ float cabs_hw(float2 a) { return sqrt_hw(a.x * a.x + a.y * a.y); }
// float -> int as a CUDA device conversion performs it: truncation toward zero, clamped to the int
// range, NaN -> 0 (the reference relies on it where Thrust accumulates floats as ints)
__device__ __forceinline__ int trunc_sat_i32(float v) {
    if (!(v == v)) return 0;
    if (v >= 2147483648.0f) return 2147483647;
    if (v <= -2147483648.0f) return -2147483647 - 1;
    return static_cast<int>(v);
}
// multiply by (dir * i): dir = -1 -> -i, dir = +1 -> +i
template <int DIR>
__device__ __forceinline__ float2 cmul_i(float2 a) {
    return DIR < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

__device__ __forceinline__ float2 expjpi_twiddle(float t);

// exp(j pi t) for a phase given in half-turns; t is reduced to [-1, 1] in FP64 before the FP32
// evaluation, so arguments carrying n^2 or k*s growth keep their digits.
__device__ __forceinline__ float2 expjpi_reduced(double t) {
    t -= 2.0 * rint(0.5 * t);
    return expjpi_twiddle(static_cast<float>(t));
}
// exp(j pi t) for t in [-2, 2] given exactly in FP32 (FFT twiddle arguments): octant reduction
// t = q/4 + r, |r| <= 1/8, then Taylor polynomials of sin(pi r) (degree 9) and cos(pi r)
// (degree 10), whose truncation errors (< 3e-11) are far below FP32 rounding, and a rotation by
// exp(j pi q / 4).
__device__ __forceinline__ float2 expjpi_twiddle(float t) {
    const float qf = rintf(4.0f * t);
    const int q = static_cast<int>(qf) & 7;
    const float r = t - 0.25f * qf;   // exact for dyadic t
    const float x = 3.14159265358979323846f * r;
    const float x2 = x * x;
    const float sn = x * (1.0f + x2 * (-1.6666667163e-1f + x2 * (8.3333337680e-3f + x2 * (-1.9841270114e-4f + x2 * 2.7557319224e-6f))));
    const float cs = 1.0f + x2 * (-0.5f + x2 * (4.1666667908e-2f + x2 * (-1.3888889225e-3f + x2 * (2.4801587642e-5f - x2 * 2.7557319224e-7f))));
    // rotation by exp(j pi q / 4) with selects only: the odd octant first (times (1 + j)/sqrt 2),
    // then the quadrant (times j^(q/2))
    constexpr float h = 0.70710678118654752440f;
    const bool odd = q & 1;
    float c = odd ? h * (cs - sn) : cs;
    float s = odd ? h * (cs + sn) : sn;
    const bool q1 = q & 2, q2 = q & 4;
    const float c1 = q1 ? -s : c, s1 = q1 ? c : s;
    c = q2 ? -c1 : c1;
    s = q2 ? -s1 : s1;
    return make_float2(c, s);
}

// ------------------------------------------------------------------------------------------
// exchange between the lanes of a wave
// ------------------------------------------------------------------------------------------
// v of lane (lane ^ MASK), a power of two below 64: by DPP moves within a row of 16 lanes and by the
// swap instructions between rows, so no trip through the LDS crossbar (about 100 cycles a step in
// the one-workgroup kernels, whose chains of such steps nothing else covers).
template <int MASK>
__device__ __forceinline__ unsigned lane_xor_bits(unsigned v) {
#ifdef ISAR_EMU
    return __shfl_xor(v, MASK, 64);
#else
    static_assert(MASK == 1 || MASK == 2 || MASK == 4 || MASK == 8 || MASK == 16 || MASK == 32, "one bit of the lane");
    const int b = static_cast<int>(v);
    if constexpr (MASK == 1) return __builtin_amdgcn_mov_dpp(b, 0xB1, 0xf, 0xf, true);        // quad_perm 1 0 3 2
    else if constexpr (MASK == 2) return __builtin_amdgcn_mov_dpp(b, 0x4E, 0xf, 0xf, true);   // quad_perm 2 3 0 1
    else if constexpr (MASK == 4)   // half-row mirror (lane ^ 7), then quad_perm 3 2 1 0 (lane ^ 3)
        return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(b, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
    else if constexpr (MASK == 8) return __builtin_amdgcn_mov_dpp(b, 0x128, 0xf, 0xf, true);  // row rotate by 8
    else if constexpr (MASK == 16) {   // odd rows of the first with even rows of the second
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (threadIdx.x & 16) ? r[0] : r[1];
    } else {                           // upper half of the first with lower half of the second
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (threadIdx.x & 32) ? r[0] : r[1];
    }
#endif
}
template <int MASK>
__device__ __forceinline__ int lane_xor(int v) { return static_cast<int>(lane_xor_bits<MASK>(static_cast<unsigned>(v))); }
template <int MASK>
__device__ __forceinline__ float lane_xor(float v) { return __uint_as_float(lane_xor_bits<MASK>(__float_as_uint(v))); }
template <int MASK, typename T>
__device__ __forceinline__ T lane_xor_64(T v) {
    uint64_t b;
    __builtin_memcpy(&b, &v, sizeof b);
    b = (static_cast<uint64_t>(lane_xor_bits<MASK>(static_cast<unsigned>(b >> 32))) << 32) |
        lane_xor_bits<MASK>(static_cast<unsigned>(b));
    __builtin_memcpy(&v, &b, sizeof b);
    return v;
}
template <int MASK>
__device__ __forceinline__ double lane_xor(double v) { return lane_xor_64<MASK>(v); }
template <int MASK>
__device__ __forceinline__ long long lane_xor(long long v) { return lane_xor_64<MASK>(v); }
template <int MASK>
__device__ __forceinline__ float2 lane_xor(float2 v) { return make_float2(lane_xor<MASK>(v.x), lane_xor<MASK>(v.y)); }

// v combined over groups of WIDTH lanes (a power of two up to 64) by steps v = step(v, v of lane ^ WIDTH / 2,
// ... ^ 1)
template <int WIDTH, typename T, typename F>
__device__ __forceinline__ T group_combine(T v, F step) {
    if constexpr (WIDTH >= 64) v = step(v, lane_xor<32>(v));
    if constexpr (WIDTH >= 32) v = step(v, lane_xor<16>(v));
    if constexpr (WIDTH >= 16) v = step(v, lane_xor<8>(v));
    if constexpr (WIDTH >= 8) v = step(v, lane_xor<4>(v));
    if constexpr (WIDTH >= 4) v = step(v, lane_xor<2>(v));
    if constexpr (WIDTH >= 2) v = step(v, lane_xor<1>(v));
    return v;
}

// ------------------------------------------------------------------------------------------
// reductions
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum_d(double v) {
    return group_combine<64>(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return group_combine<64>(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float2 wave_sum2(float2 v) {
    return group_combine<64>(v, [](float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); });
}
// (value, index) argmax and argmin with the lowest index on ties: LESS = true takes the smaller value
template <bool LESS, int MASK>
__device__ __forceinline__ void wave_arg_step(float& v, int& i) {
    const float ov = lane_xor<MASK>(v);
    const int oi = lane_xor<MASK>(i);
    const bool take = (LESS ? ov < v : ov > v) | ((ov == v) & (oi < i));
    v = take ? ov : v;
    i = take ? oi : i;
}
template <bool LESS>
__device__ __forceinline__ void wave_arg(float& v, int& i) {
    wave_arg_step<LESS, 32>(v, i);
    wave_arg_step<LESS, 16>(v, i);
    wave_arg_step<LESS, 8>(v, i);
    wave_arg_step<LESS, 4>(v, i);
    wave_arg_step<LESS, 2>(v, i);
    wave_arg_step<LESS, 1>(v, i);
}

// Workgroup-wide reductions through a small LDS scratch (>= 16 slots). All threads get the
// result. Must be called by every thread of the workgroup.
template <int NT>
__device__ __forceinline__ long long block_sum_i64(long long v, long long* red) {
    v = group_combine<64>(v, [](long long a, long long b) { return a + b; });
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) red[w] = v;
    __syncthreads();
    long long r = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) r += red[i];
    return r;
}
template <int NT>
__device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) red[w] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) r = fmaxf(r, red[i]);
    return r;
}
template <int NT>
__device__ __forceinline__ void block_argmax(float& v, int& i, float* redv, int* redi) {
    wave_arg<false>(v, i);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) { redv[w] = v; redi[w] = i; }
    __syncthreads();
    v = redv[0];
    i = redi[0];
#pragma unroll
    for (int k = 1; k < NT / 64; ++k) {
        const float ov = redv[k];
        const int oi = redi[k];
        const bool take = (ov > v) | ((ov == v) & (oi < i));
        v = take ? ov : v;
        i = take ? oi : i;
    }
}
template <int NT>
__device__ __forceinline__ void block_argmin(float& v, int& i, float* redv, int* redi) {
    wave_arg<true>(v, i);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) { redv[w] = v; redi[w] = i; }
    __syncthreads();
    v = redv[0];
    i = redi[0];
#pragma unroll
    for (int k = 1; k < NT / 64; ++k) {
        const float ov = redv[k];
        const int oi = redi[k];
        const bool take = (ov < v) | ((ov == v) & (oi < i));
        v = take ? ov : v;
        i = take ? oi : i;
    }
}
// Exclusive prefix sum of integers over the workgroup; returns the exclusive prefix, total in
// *tot. With T = unsigned the sums wrap modulo 2^32.
template <int NT, typename T = int>
__device__ __forceinline__ T block_exclusive_scan(T v, T* red, T* tot) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    T x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        T y = __shfl_up(x, o, 64);
        if (l >= o) x += y;
    }
    __syncthreads();
    if (l == 63) red[w] = x;
    __syncthreads();
    T base = 0, all = 0;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) {
        T r = red[k];
        if (k < w) base += r;
        all += r;
    }
    *tot = all;
    return base + x - v;
}

// ------------------------------------------------------------------------------------------
// register and address helpers
// ------------------------------------------------------------------------------------------
// A copy of v that the compiler cannot see through. Index and address arithmetic derived from it
// is recomputed where it is used instead of being kept live in registers across transforms.
__device__ __forceinline__ int opaque(int v) {
#ifndef ISAR_EMU
    asm volatile("" : "+v"(v));
#endif
    return v;
}
// Keeps the compiler from moving instructions across: placed after a batch of loads, so that they
// are issued together instead of each just before its use (which it prefers where that saves registers).
__device__ __forceinline__ void issue_point() {
#ifndef ISAR_EMU
    __builtin_amdgcn_sched_barrier(0);
#endif
}
// Element i of p for 0 <= i < 2^28 / sizeof(T) (p typically wave-uniform): the byte offset is
// formed in 32 bits, so the access can take the base in scalar registers and a 32-bit per-lane
// offset instead of a 64-bit address per lane.
template <typename T>
__device__ __forceinline__ T& elem_u32(T* p, unsigned i) {
    using B = std::conditional_t<std::is_const_v<T>, const char, char>;
    return *reinterpret_cast<T*>(reinterpret_cast<B*>(p) + i * static_cast<unsigned>(sizeof(T)));
}

// Value of v held by lane `lane` (a compile-time constant in practice) of the calling wave.
__device__ __forceinline__ float wave_read_lane(float v, int lane) {
#ifdef ISAR_EMU
    return __shfl(v, lane, 64);
#else
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
#endif
}

// v, equal in every lane of the wave, in scalar registers
__device__ __forceinline__ double uniform(double v) {
#ifdef ISAR_EMU
    return v;
#else
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
#endif
}

// 1 / v to about 1 ulp (v_rcp_f32), without the correctly rounded division sequence.
__device__ __forceinline__ float rcp_hw(float v) {
#ifdef ISAR_EMU
    return 1.0f / v;
#else
    return __builtin_amdgcn_rcpf(v);
#endif
}

__device__ __forceinline__ float opaque(float v) {
#ifndef ISAR_EMU
    asm volatile("" : "+v"(v));
#endif
    return v;
}

__device__ __forceinline__ double opaque(double v) {
#ifndef ISAR_EMU
    asm volatile("" : "+v"(v));
#endif
    return v;
}

__device__ __forceinline__ float2 opaque(float2 v) {
#ifndef ISAR_EMU
    asm volatile("" : "+v"(v.x), "+v"(v.y));
#endif
    return v;
}

// Column tile of workgroup b among the `tiles` tiles (gridDim.x) of a frame, ordered so that one
// XCD runs adjacent tiles. Workgroups go to the 8 XCDs round-robin by linear id (b + tiles f), so
// with tiles % 8 == 0 XCD x takes tiles [x tiles/8, (x+1) tiles/8) of every frame: tiles narrower
// than a 128-byte line then share its fetch in one L2 instead of each XCD fetching it.
__device__ __forceinline__ int xcd_tile(int b, int tiles) {
    return (tiles & 7) ? b : (b & 7) * (tiles >> 3) + (b >> 3);
}

}  // namespace isar

#include "fft.hpp"

namespace isar {

// Hamming window 0.54 - 0.46 cos(2 pi n / (len - 1))  (genHammingVec, common.cu:260-266)
__device__ __forceinline__ float hamming(int n, int len) {
    return 0.54f - 0.46f * cospif(2.0f * static_cast<float>(n) / static_cast<float>(len - 1));
}

}  // namespace isar

namespace isar {

// Sum over aligned groups of WIDTH lanes (WIDTH a power of two <= 64).
template <int WIDTH>
__device__ __forceinline__ float group_sum(float v) {
    static_assert(WIDTH <= 64, "shuffle groups cannot span waves");
    return group_combine<WIDTH>(v, [](float a, float b) { return a + b; });
}
template <int WIDTH>
__device__ __forceinline__ float2 group_sum2(float2 v) {
    static_assert(WIDTH <= 64, "shuffle groups cannot span waves");
    return group_combine<WIDTH>(v, [](float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); });
}

// Inclusive prefix sum in FP64 of n values held as v[i] (i < n) in LDS, in place, by the whole
// workgroup (NT threads): every 64 consecutive values are scanned by a wave, then the sums of the
// 64s before are added in their order, so that the result does not depend on NT. red: n / 64 slots.
// (A serial pass over 1024 threads' partial sums took 11 us of a kernel's 16.)
template <int NT>
__device__ __forceinline__ void block_inclusive_scan_d(double* v, int n, double* red) {
    const int lane = threadIdx.x & 63;
    for (int i0 = 0; i0 < n; i0 += NT) {   // every thread takes part in the shuffles
        const int i = i0 + threadIdx.x;
        double x = i < n ? v[i] : 0.0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double y = __shfl_up(x, o, 64);
            x = lane >= o ? x + y : x;
        }
        if (i < n) v[i] = x;
        if (lane == 63 && i - 63 < n) red[i >> 6] = x;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += NT) {
        double base = 0.0;
        for (int k = 0; k < (i >> 6); ++k) base += red[k];
        v[i] += base;
    }
    __syncthreads();
}

// Column-transform configuration for M-point slow-time transforms inside a 256-thread block. A forward
// transform takes the layout in() to out(), a reversed one (fft<..., true>) back.
template <int M>
struct ColCfg {
    static constexpr int E = (M == 192 || M == 384 || M == 768) ? 12 : 16;
    static constexpr int TPF = M / E;                  // threads per transform
    static constexpr int NT = 256;
    static constexpr int CT = NT / TPF;                // transforms (columns) per block
    __device__ static int in(int lane, int e) { return fft_in_pos<M, E>(lane, e); }
    __device__ static int out(int lane, int e) { return fft_out_pos<M, E>(lane, e); }
};

// Copies columns n0 ... n0 + CT - 1 of rows 0 ... M - 1 of a row-major matrix of W columns into LDS,
// element (m, c) at sm[m (CT + 1) + c], by NT threads with eight loads of a thread in flight: the
// column kernels wait for this tile before anything else, and with a load at a time that wait was
// most of their time.
template <int NT, int CT>
__device__ __forceinline__ void load_column_tile(const float2* src, int W, int n0, int M, float2* sm, int tid) {
    const int total = M * CT;
    for (int i0 = tid; i0 < total; i0 += 8 * NT) {
        float2 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = min(i0 + q * NT, total - 1);
            v[q] = elem_u32(src, static_cast<unsigned>((i / CT) * W + n0 + i % CT));
        }
        issue_point();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int i = i0 + q * NT;
            if (i < total) sm[(i / CT) * (CT + 1) + i % CT] = v[q];
        }
    }
}

// ------------------------------------------------------------------------------------------
// Hand-off between the workgroups of one launch (the resident autofocus). Values pass through
// memory as 64-bit words stored and loaded as agent-scope relaxed atomics: global accesses with
// sc1 set, which are written through to the device's point of coherence and read from it, never
// from a stale line of another XCD's L2. A word is empty until its value is stored, and a reader
// polls it until it is not, so nothing but the value itself has to arrive; a word that is used again
// is emptied first, and that store waited for (s_waitcnt 0). No fence, L2 write-back or invalidation
// is involved.
// ------------------------------------------------------------------------------------------
constexpr uint64_t kXwgEmpty = ~0ull;   // two NaNs
__device__ __forceinline__ uint64_t xwg_word(float2 v) {
    uint64_t w;
    __builtin_memcpy(&w, &v, sizeof w);
    return w == kXwgEmpty ? w - 1 : w;   // NaNs as well
}
__device__ __forceinline__ float2 xwg_value(uint64_t w) {
    float2 v;
    __builtin_memcpy(&v, &w, sizeof v);
    return v;
}
__device__ __forceinline__ void xwg_store(uint64_t* p, uint64_t w) {
#ifdef ISAR_EMU
    __atomic_store_n(p, w, __ATOMIC_RELAXED);
#else
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}
__device__ __forceinline__ uint64_t xwg_load(const uint64_t* p) {
#ifdef ISAR_EMU
    return __atomic_load_n(p, __ATOMIC_RELAXED);
#else
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}
// Waits until this thread's stores are acknowledged.
__device__ __forceinline__ int32_t xwg_load(const int32_t* p) {
#ifdef ISAR_EMU
    return __atomic_load_n(p, __ATOMIC_SEQ_CST);
#else
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}
__device__ __forceinline__ void xwg_stores_done() {
#ifdef ISAR_EMU
    __atomic_thread_fence(__ATOMIC_SEQ_CST);
#else
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
#endif
}
__device__ __forceinline__ void xwg_pause() {
#ifdef ISAR_EMU
    ++isar_emu::pauses;
    std::this_thread::yield();
#else
    __builtin_amdgcn_s_sleep(2);
#endif
}

}  // namespace isar
