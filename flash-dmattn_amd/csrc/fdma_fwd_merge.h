// Shares of split keys, forward: what a share leaves -- O in fp32, divided by its sum, and its log2-sum-exp -- and how they are added up.
// With arrival counters the workgroup of a row block that finishes last does it: the shares lie in the order in which the lanes hold
// them, 1 KB per store.  Without, a launch of its own does, and they lie row by row.  The arithmetic is the same, and so are the bits.
#pragma once

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

// Written and read by workgroups of one launch, possibly behind different L2s: device-scope accesses, which go where every XCD sees them
// (no fence: it would walk the whole L2, in every workgroup).  Whole lines, the wave's first 8 bytes of four numbers in front of its second:
// 8 bytes of each of 64 rows per store, which no cache gathers, made the launch twice as long as without shares.
// `at`: a piece of 256 floats and 2 * lane.
__device__ __forceinline__ void share_store4(float *at, f32x4_t v) {
    union { f32x2_t f; uint64_t u; } a, b;
    a.f = f32x2_t{v[0], v[1]};
    b.f = f32x2_t{v[2], v[3]};
    __hip_atomic_store((uint64_t *)at, a.u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store((uint64_t *)(at + 128), b.u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void share_store(float *dst, float v) {
    __hip_atomic_store((uint32_t *)dst, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x4_t share_load4(const float *at) {
    union { f32x2_t f; uint64_t u; } a, b;
    a.u = __hip_atomic_load((const uint64_t *)at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    b.u = __hip_atomic_load((const uint64_t *)(at + 128), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return f32x4_t{a.f[0], a.f[1], b.f[0], b.f[1]};
}
__device__ __forceinline__ float share_load(const float *src) {
    return __uint_as_float(__hip_atomic_load((const uint32_t *)src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Weights of a row's shares, 2^(l_s - l) with l = log2 sum_s 2^l_s, from their l_s (-inf beyond the last).  Only a share without a visible
// key, l_s = -inf, is left out: an l_s that is no number (a NaN among its keys or in the query) has a weight that is none either,
// which makes the row what the call with whole keys makes it.  No share with a visible key: 0 and +inf.
struct ShareWeights {
    float w[MAX_KEY_SPLITS], inv, lse;
};
__device__ __forceinline__ ShareWeights share_weights(const float (&l)[MAX_KEY_SPLITS]) {
    ShareWeights r;
    float top = l[0], sum = 0.f;
#pragma unroll
    for (int s = 1; s < MAX_KEY_SPLITS; s++) top = fmaxf(top, l[s]);
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) {
        r.w[s] = l[s] != -INFINITY ? fast_exp2(l[s] - top) : 0.f;
        sum += r.w[s];
    }
    r.inv = sum > 0.f ? 1.f / sum : 0.f;
    r.lse = sum > 0.f ? (top + __builtin_amdgcn_logf(sum)) * kLn2 : INFINITY;
    return r;
}
// Eight elements of O in 16 bits, from the shares' weighted sum
template <typename T> __device__ __forceinline__ u32x4_t merged8(float inv, const f32x4_t (&a)[2]) {
    u32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = Elem<T>::pack2(a[e >> 1][2 * (e & 1)] * inv, a[e >> 1][2 * (e & 1) + 1] * inv);
    return w;
}
__device__ __forceinline__ void add_share(f32x4_t (&a)[2], float w, const f32x4_t (&v)[2]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        a[0][e] = fmaf(w, v[0][e], a[0][e]);
        a[1][e] = fmaf(w, v[1][e], a[1][e]);
    }
}
// Weights of one lane's row, its l_s `l_step` apart; and eight of its elements, two pieces of four, at `first` and 256 floats on, of shares
// `step` apart
__device__ __forceinline__ ShareWeights lane_share_weights(const float *l, int64_t l_step, int n, bool (&on)[MAX_KEY_SPLITS]) {
    float x[MAX_KEY_SPLITS];
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) x[s] = s < n ? share_load(l + s * l_step) : -INFINITY;
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) on[s] = x[s] != -INFINITY;
    return share_weights(x);
}
// ... of N units of eight, 512 floats apart: the shares four at a time, all their loads in flight together (one unit after the other was a trip
// to memory each).
template <typename T, int N>
__device__ __forceinline__ void lane_merged(const ShareWeights &r, const float *first, int64_t step, int n, const bool (&on)[MAX_KEY_SPLITS], u32x4_t (&out)[N]) {
    f32x4_t a[N][2];
#pragma unroll
    for (int u = 0; u < N; u++) a[u][0] = a[u][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto four = [&](auto s0_c) {
        constexpr int s0 = decltype(s0_c)::value;
        f32x4_t v[4][N][2];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const float *at = first + (s0 + s < n ? s0 + s : n - 1) * step;  // (beyond the last: it again, dropped)
#pragma unroll
            for (int u = 0; u < N; u++) {
                v[s][u][0] = share_load4(at + u * 512);
                v[s][u][1] = share_load4(at + u * 512 + 256);
            }
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int u = 0; u < N; u++) {
#pragma unroll
                for (int e = 0; e < 4; e++) {  // (what a share without a visible key left need not be a number)
                    v[s][u][0][e] = on[s0 + s] ? v[s][u][0][e] : 0.f;
                    v[s][u][1][e] = on[s0 + s] ? v[s][u][1][e] : 0.f;
                }
                add_share(a[u], r.w[s0 + s], v[s][u]);
            }
    };
    static_assert(MAX_KEY_SPLITS == 8, "two rounds");
    four(std::integral_constant<int, 0>());
    if (n > 4) four(std::integral_constant<int, 4>());
#pragma unroll
    for (int u = 0; u < N; u++) out[u] = merged8<T>(r.inv, a[u]);
}

// Counts this workgroup, whose share is stored, in at counter `at` (zero at the start, left zero): whether it is the last of `n`.  Called by
// all its threads together; `flag`: a word of LDS that is free.  Nothing waits for another workgroup: one that is not last just ends.
__device__ __forceinline__ bool last_share(int32_t *at, int n, int *flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave until its own stores are acknowledged ...
    __syncthreads();                                   // ... and all of them
    if (threadIdx.x == 0) {
        const int last = __hip_atomic_fetch_add(at, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
        if (last) __hip_atomic_store(at, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    return *flag != 0;
}

}  // namespace fdma
