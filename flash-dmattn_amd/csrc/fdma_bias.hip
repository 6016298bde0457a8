// Producer of the dynamic-mask attention bias, fused: bias[b, j, 0, l] = A[j] * softplus(dt[b, l, j]) with
// dt = V_flat[b, l, :] . W[j, :] (+ pb[j]), V_flat the value states of all kv heads of a token side by side -- the
// `A * softplus(dt_proj(V))` of the reference's Doge caller (examples/modeling/modeling_doge.py:217-222), which there is a
// linear layer, a softplus, a multiply, a transpose and a cast through the tensor library in front of every attention
// call, and the same again backwards.  The column-summed dBias that the attention backward returns in the bias's own
// [B, Hkv, 1, Lk] shape is consumed here directly.
//
// Forward: bound by reading V once.  A wave owns 32 tokens and a range of the columns of V_flat; 128 columns at a time (8 KB)
// go from global memory straight into one of the wave's two pieces of LDS -- whole 256-byte runs of a row per 16 lanes, no
// barrier, the next piece in flight while one is worked on -- and from there into the A operand of MFMA 32x32x16; W rows, the B
// operand, come from the caches.  The accumulator column of lane j < Hkv holds dt of 16 of the tokens; it goes through LDS so that
// softplus is computed by all lanes and the bias rows leave in runs.  (Every lane fetching 16 bytes of its own row per step asked
// for 32 lines per instruction.  8 x 4093 tokens of 8 x 128, 67 MB, bf16: 23 us that way, 16.7 with one piece of 256 columns that is
// waited for whole, 14.4 now; 4 x 2304 of 16 x 256, 288 workgroups of eight pieces in a row: 24.7 -> 20.0; 4 x 2048 of 8 x 64
// 8.0 -> 5.6.)
// Backward: a workgroup owns a run of tokens; d_dt = dBias * A * sigmoid(dt) goes to LDS, then a thread owns four
// columns of V_flat and walks the tokens: dV = d_dt W and the workgroup's share of dW = d_dt^T V_flat, dA and dpb, which
// go to fp32 partials that a second kernel folds in a fixed order (bit-reproducible).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {
namespace {

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(__expf(x)); }  // torch: beta 1, threshold 20
__device__ __forceinline__ float sigmoid_f(float x) { return x > 20.f ? 1.f : 1.f / (1.f + __expf(-x)); }  // d softplus / dx, same threshold

// SPLITK: the four waves of a workgroup share 32 tokens, a quarter of the columns each (few tokens: more waves in
// flight); otherwise every wave owns 32 tokens of its own and reads whole rows.
constexpr int PC = 128;                       // columns of V_flat per piece
constexpr int PIECE_BYTES = 32 * PC * 2;      // of 32 tokens
constexpr int PIECE_LOADS = PIECE_BYTES / 1024;
constexpr int WAVE_LDS = 2 * PIECE_BYTES;     // a wave's two pieces
constexpr int OFF_OUT = 8192;                 // ... reused: accumulators (4 KB), and from here the 16-bit results [head][token]
constexpr int OUT_PITCH = 34;

template <typename T, bool SPLITK>
__global__ void __launch_bounds__(256) dyn_bias_fwd_kernel(const DynBiasParams p) {
    using E = Elem<T>;
    __shared__ __attribute__((aligned(256))) char smem[4 * WAVE_LDS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, g = lane >> 5;
    const int64_t n_rows = (int64_t)p.B * p.L;
    const int64_t row0 = SPLITK ? (int64_t)blockIdx.x * 32 : ((int64_t)blockIdx.x * 4 + wave) * 32;
    if (!SPLITK && row0 >= n_rows) return;  // (no barrier on this path)
    const int K = p.Hk * p.d;
    const int b0 = (int)(row0 / p.L), l0 = (int)(row0 - (int64_t)b0 * p.L);
    const int n_tok = n_rows - row0 < 32 ? (int)(n_rows - row0) : 32;
    // batch entry and position of token row0 + t
    auto place = [&](int t, int &b, int &l) {
        b = b0;
        l = l0 + t;
        while (l >= p.L) { l -= p.L; b++; }
    };
    char *piece = smem + wave * WAVE_LDS;
    const uint16_t *wrow = (const uint16_t *)p.w + (int64_t)(r < p.Hk ? r : 0) * K;
    const uint32_t wmask = r < p.Hk ? 0xffffffffu : 0u;  // output columns beyond Hkv: zero operand (no branch around the load)
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.f;
    constexpr int KU = PC / 16;
    const int n_ks = K / 16, per_wave = SPLITK ? ((n_ks + 3) / 4 + KU - 1) / KU * KU : n_ks;
    const int ks_begin = SPLITK ? wave * per_wave : 0;
    const int ks_end = ks_begin + per_wave < n_ks ? ks_begin + per_wave : n_ks;
    // direct load i of a piece: tokens 4 i .. 4 i + 3 (clamped duplicates beyond the last), lane l the chunk POSITION l % 16 of row
    // t = 4 i + l / 16, which holds chunk position ^ (t % 16): reads of one chunk by 16 tokens then fall into 16 different chunks
    const int cpos = lane & 15, tq = lane >> 4;
    const uint16_t *vrow[PIECE_LOADS];
#pragma unroll
    for (int i = 0; i < PIECE_LOADS; i++) {
        int b, l;
        place(4 * i + tq < n_tok ? 4 * i + tq : n_tok - 1, b, l);
        vrow[i] = (const uint16_t *)p.v + b * p.v_b + (int64_t)l * p.v_r;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(piece));
    // requests piece n of this wave: W's rows first, so that the youngest PIECE_LOADS requests are those of the columns
    auto fetch = [&](int n, u32x4_t (&bw)[KU]) {
        const int ks0 = ks_begin + n * KU;
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int ks = ks0 + u < ks_end ? ks0 + u : ks_end - 1;  // (a short last piece re-reads the last step and drops it)
            bw[u] = *(const u32x4_t *)(wrow + ks * 16 + 8 * g);
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < PIECE_LOADS; i++) {
            int kk = ks0 * 16 + ((cpos ^ ((4 * i + tq) & 15)) * 8);
            kk = kk < ks_end * 16 ? kk : ks_begin * 16;  // (past this wave's columns: any of its chunks, never read)
            const int head = p.v_h == p.d ? 0 : kk / p.d;
            const uint16_t *src = vrow[i] + (int64_t)head * p.v_h + (kk - head * p.d);
            load_lds16_at(src, lds0 + (n & 1) * PIECE_BYTES + i * 1024);
        }
    };
    // piece n, which has landed
    auto work = [&](int n, u32x4_t (&bw)[KU]) {
        const int ks0 = ks_begin + n * KU;
        const char *base = piece + (n & 1) * PIECE_BYTES + r * (PC * 2);
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const uint32_t m = (ks0 + u < ks_end) ? wmask : 0u;
            u32x4_t a = *(const u32x4_t *)(base + (((2 * u + g) ^ (r & 15)) << 4));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                bw[u][e] &= m;
                a[e] = (ks0 + u < ks_end) ? a[e] : 0u;  // (what an unused part of the piece holds need not be a number)
            }
            acc = E::mfma(a, bw[u], acc);
        }
    };
    const int n_pieces = ks_begin < ks_end ? (ks_end - ks_begin + KU - 1) / KU : 0;
    u32x4_t bw0[KU], bw1[KU];
    // (a piece's successor is requested before it is worked on.  Where the two ways to a wait differ in what is in flight, the compiler
    // waits for everything: hence no branch inside)
    auto reads_done = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };  // (of the piece that is overwritten next)
    auto landed = [&](auto younger) { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(decltype(younger)::value) : "memory"); };
    constexpr auto one_more = std::integral_constant<int, PIECE_LOADS>();
    constexpr auto none = std::integral_constant<int, 0>();
    if (n_pieces > 0) {
        int n = 0;
        fetch(0, bw0);
#pragma unroll 1
        for (; n + 2 < n_pieces; n += 2) {
            reads_done();
            fetch(n + 1, bw1);
            landed(one_more);
            work(n, bw0);
            reads_done();
            fetch(n + 2, bw0);
            landed(one_more);
            work(n + 1, bw1);
        }
        if (n + 1 < n_pieces) {
            reads_done();
            fetch(n + 1, bw1);
            landed(one_more);
            work(n, bw0);
            landed(none);
            work(n + 1, bw1);
        } else {
            landed(none);
            work(n, bw0);
        }
    }
    __builtin_amdgcn_wave_barrier();
    // ---- dt of (token, head) = the waves' sums in wave order; bias rows through LDS
    if (r < p.Hk) {
#pragma unroll
        for (int i = 0; i < 16; i++) ((float *)piece)[i * 64 + lane] = acc[i];
    }
    if (SPLITK) __syncthreads();
    const char *part = SPLITK ? smem : piece;
    uint16_t *s_out = (uint16_t *)(part + OFF_OUT);
    const int step = SPLITK ? 256 : 64, t0 = SPLITK ? (int)threadIdx.x : lane;
    const int n_out = n_tok * p.Hk;
    for (int idx = t0; idx < n_out; idx += step) {
        const int t = idx / p.Hk, j = idx - t * p.Hk;
        const int at = ((t >> 3) * 4 + (t & 3)) * 64 + ((t >> 2) & 1) * 32 + j;  // token t = 8 (i / 4) + 4 g + i % 4
        float dt = ((const float *)part)[at];
        if (SPLITK) {
#pragma unroll
            for (int w = 1; w < 4; w++) dt += ((const float *)(part + w * WAVE_LDS))[at];
        }
        dt += p.pb ? E::lo((uint32_t)((const uint16_t *)p.pb)[j]) : 0.f;
        if (p.dt) p.dt[row0 * p.Hk + idx] = dt;
        s_out[j * OUT_PITCH + t] = (uint16_t)(E::pack2(E::lo((uint32_t)((const uint16_t *)p.a)[j]) * softplus_f(dt), 0.f) & 0xffffu);
    }
    if (SPLITK) __syncthreads();
    else __builtin_amdgcn_wave_barrier();  // (the LDS operations of one wave execute in order)
    for (int idx = t0; idx < 32 * p.Hk; idx += step) {
        const int j = idx >> 5, t = idx & 31;
        if (t < n_tok) {
            int b, l;
            place(t, b, l);
            ((uint16_t *)p.bias)[b * p.bias_b + (int64_t)j * p.bias_h + l] = s_out[j * OUT_PITCH + t];
        }
    }
}

// Backward, first stage.  Latency: a workgroup's tokens are one trip to memory when their loads are issued together, ahead of
// d_dt (eight trips of four tokens each before), and the two halves of a workgroup take half of a pass's tokens each: 4 x 2048
// tokens of 8 x 64 took 18 us, now 12.  Workgroup `c` owns token rows [c * rows_per_wg, ...).  HM = Hkv rounded up to 8, 16 or 32:
// thread t works on output head t % HM for the per-head sums, so each sum is built in a fixed order; in the main part
// a thread owns CPT adjacent columns of V_flat (4; 2 when 32 heads' worth of accumulators must fit the registers or
// when V_flat has too few columns to give every thread four).
template <typename T, int HM, int CPT>
__global__ void __launch_bounds__(512) dyn_bias_bwd_kernel(const DynBiasParams p) {
    using E = Elem<T>;
    constexpr int RB = 64;                   // tokens per pass through LDS
    constexpr int TB = 16;                   // tokens whose loads are in flight together (registers)
    constexpr int NT = 512, HC = 16 / CPT < HM ? 16 / CPT : HM;  // HC: heads whose sums the halves exchange at a time
    __shared__ float s_ddt[RB * HM];
    __shared__ float s_red[2][NT / 64][HM];
    __shared__ float s_x[HC * CPT * 256];
    const int tid = threadIdx.x, half = __builtin_amdgcn_readfirstlane(tid >> 8), ctid = tid & 255;  // (columns are owned by a thread of each half)
    const int Hk = p.Hk, K = Hk * p.d;
    const int64_t wg_row0 = (int64_t)blockIdx.x * p.rows_per_wg;
    const int64_t n_rows = (int64_t)p.B * p.L;
    const int64_t wg_row1 = wg_row0 + p.rows_per_wg < n_rows ? wg_row0 + p.rows_per_wg : n_rows;
    const int j_mine = tid % HM, rgroup = tid / HM;
    constexpr int RSTEP = NT / HM;
    const float a_mine = j_mine < Hk ? E::lo((uint32_t)((const uint16_t *)p.a)[j_mine]) : 0.f;
    float sum_a = 0.f, sum_pb = 0.f;  // this thread's share of dA[j_mine], dpb[j_mine]
    float *part_w = p.part + (int64_t)blockIdx.x * p.part_stride;
    const int n_groups = (K + 256 * CPT - 1) / (256 * CPT);  // column groups: the same trip count for every thread

    for (int grp = blockIdx.y; grp < n_groups; grp += gridDim.y) {
        const int k0 = grp * 256 * CPT + ctid * CPT;
        const bool has_cols = k0 < K;
        const int head = has_cols ? k0 / p.d : 0, dd = has_cols ? k0 - head * p.d : 0;
        // (raw, unconditional loads: the pass below requests its own before anything looks at these)
        uint32_t wraw[HM][CPT / 2];
        float wj[HM][CPT], dw[HM][CPT];
#pragma unroll
        for (int j = 0; j < HM; j++) {
#pragma unroll
            for (int e = 0; e < CPT; e += 2) {
                wraw[j][e / 2] = *(const uint32_t *)((const uint16_t *)p.w + (int64_t)(j < Hk ? j : 0) * K + (has_cols ? k0 : 0) + e);
                dw[j][e] = dw[j][e + 1] = 0.f;
            }
        }
        for (int64_t base = wg_row0; base < wg_row1; base += RB) {
            // the first TB tokens' values are requested in front of everything else of the pass
            const int n = (int)(wg_row1 - base < RB ? wg_row1 - base : RB);
            uint32_t vraw[TB][CPT / 2];
            const int b0 = (int)((uint32_t)base / (uint32_t)p.L), l0 = (int)base - b0 * p.L;  // (fewer than 2^31 tokens: their values fill the memory)
            auto place = [&](int t, int &b, int &l) {  // batch entry and position of token base + t
                b = b0;
                l = l0 + t;
                while (l >= p.L) { l -= p.L; b++; }
            };
            // (rows are walked by adding strides, not by a product per token and matrix in scalar arithmetic)
            const int64_t col_v = (int64_t)head * p.v_h + dd, col_dv = (int64_t)head * p.dv_h + dd;
            auto load_v = [&](int rr0) {
                int b, l;
                place(rr0 < n ? rr0 : n - 1, b, l);
                const uint16_t *row = (const uint16_t *)p.v + b * p.v_b + (int64_t)l * p.v_r;
#pragma unroll
                for (int u = 0; u < TB; u++) {
#pragma unroll
                    for (int e = 0; e < CPT / 2; e++) vraw[u][e] = *(const uint32_t *)(row + col_v + 2 * e);
                    if (rr0 + u + 1 < n) {  // (past the last token: it again)
                        row += p.v_r;
                        if (++l == p.L) { l = 0; row += p.v_b - p.L * p.v_r; }
                    }
                }
            };
            const int nh = (n + 1) / 2, h_lo = half ? nh : 0, h_hi = half ? n : nh;  // this half's tokens
            load_v(h_lo);
            uint16_t gb_raw[RB / RSTEP];
            float dt_raw[RB / RSTEP];
#pragma unroll
            for (int i = 0; i < RB / RSTEP; i++) {
                const int rr = rgroup + i * RSTEP;
                int b, l;
                place(rr < n ? rr : n - 1, b, l);
                const int j = j_mine < Hk ? j_mine : 0;
                gb_raw[i] = ((const uint16_t *)p.dbias)[b * p.dbias_b + (int64_t)j * p.dbias_h + l];
                dt_raw[i] = p.dt[(base + (rr < n ? rr : n - 1)) * Hk + j];
            }
            __syncthreads();
            if (base == wg_row0) {
#pragma unroll
                for (int j = 0; j < HM; j++)
#pragma unroll
                    for (int e = 0; e < CPT; e += 2) {
                        wj[j][e] = j < Hk ? E::lo(wraw[j][e / 2]) : 0.f;
                        wj[j][e + 1] = j < Hk ? E::hi(wraw[j][e / 2]) : 0.f;
                    }
            }
            // d_dt of the RB tokens of this pass -> LDS; the per-head sums are taken on the first column group
#pragma unroll
            for (int i = 0; i < RB / RSTEP; i++) {
                const int rr = rgroup + i * RSTEP;
                float ddt = 0.f;
                if (j_mine < Hk && rr < n) {
                    const float gb = E::lo((uint32_t)gb_raw[i]), dt = dt_raw[i];
                    ddt = gb * a_mine * sigmoid_f(dt);
                    if (grp == 0) {
                        sum_a += gb * softplus_f(dt);
                        sum_pb += ddt;
                    }
                }
                s_ddt[rr * HM + j_mine] = ddt;
            }
            __syncthreads();
            for (int rr0 = h_lo; rr0 < h_hi; rr0 += TB) {
                if (rr0 > h_lo) load_v(rr0);
                int b, l;
                place(rr0, b, l);
                uint16_t *orow = (uint16_t *)p.dv + b * p.dv_b + (int64_t)l * p.dv_r;
#pragma unroll
                for (int u = 0; u < TB; u++) {
                    if (rr0 + u < h_hi && has_cols) {
                        float v4[CPT], dv[CPT];
#pragma unroll
                        for (int e = 0; e < CPT; e += 2) {
                            v4[e] = E::lo(vraw[u][e / 2]);
                            v4[e + 1] = E::hi(vraw[u][e / 2]);
                            dv[e] = dv[e + 1] = 0.f;
                        }
#pragma unroll
                        for (int j = 0; j < HM; j++) {
                            const float ddt = s_ddt[(rr0 + u) * HM + j];  // same address for the whole wave: a broadcast read; 0 beyond Hkv
#pragma unroll
                            for (int e = 0; e < CPT; e++) {
                                dw[j][e] += ddt * v4[e];
                                dv[e] += ddt * wj[j][e];
                            }
                        }
#pragma unroll
                        for (int e = 0; e < CPT; e += 2) *(uint32_t *)(orow + col_dv + e) = E::pack2(dv[e], dv[e + 1]);
                    }
                    orow += p.dv_r;
                    if (++l == p.L) { l = 0; orow += p.dv_b - p.L * p.dv_r; }
                }
            }
        }
        // the halves' sums, in order, HC heads at a time
#pragma unroll
        for (int j0 = 0; j0 < HM; j0 += HC) {
            __syncthreads();
            if (half) {
#pragma unroll
                for (int j = 0; j < HC; j++)
#pragma unroll
                    for (int e = 0; e < CPT; e++) s_x[(j * CPT + e) * 256 + ctid] = dw[j0 + j][e];
            }
            __syncthreads();
            if (!half && has_cols) {
#pragma unroll
                for (int j = 0; j < HC; j++)
                    if (j0 + j < Hk) {
#pragma unroll
                        for (int e = 0; e < CPT; e++) part_w[(int64_t)(j0 + j) * K + k0 + e] = dw[j0 + j][e] + s_x[(j * CPT + e) * 256 + ctid];
                    }
            }
        }
    }
    // per-head sums: a head's threads in a wave, by lane swaps, then the waves in order.  (All of a head's NT / HM through LDS by one
    // thread were a chain of 64 reads.)
    if (blockIdx.y) return;
    auto fold = [&](float x) -> float {
        const uint32_t u = __float_as_uint(x);
        const auto r32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        x = __uint_as_float((uint32_t)r32[0]) + __uint_as_float((uint32_t)r32[1]);
        if (HM <= 16) {
            const uint32_t w = __float_as_uint(x);
            const auto r16 = __builtin_amdgcn_permlane16_swap(w, w, false, false);
            x = __uint_as_float((uint32_t)r16[0]) + __uint_as_float((uint32_t)r16[1]);
        }
        if (HM <= 8) x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x128, 0xf, 0xf, false));  // row_ror:8
        return x;
    };
    sum_a = fold(sum_a);
    sum_pb = fold(sum_pb);
    if ((tid & 63) < HM) {
        s_red[0][tid >> 6][tid & 63] = sum_a;
        s_red[1][tid >> 6][tid & 63] = sum_pb;
    }
    __syncthreads();
    if (tid < Hk) {
        float sa = 0.f, sb = 0.f;
#pragma unroll
        for (int w = 0; w < NT / 64; w++) {
            sa += s_red[0][w][tid];
            sb += s_red[1][w][tid];
        }
        part_w[(int64_t)Hk * K + tid] = sa;
        part_w[(int64_t)Hk * K + Hk + tid] = sb;
    }
}

// Backward, second stage: dW, dA, dpb = sum of the workgroups' partials.  A workgroup owns 64 elements; wave w adds every
// eighth partial (all loads of 16 of them in flight), and the eight sums are added in wave order: a fixed order.  (A thread
// per element left 17 workgroups, each a chain of 256 loads: 12.7 us for 4 MB, now 4.7.)
constexpr int RED_WAVES = 8;
template <typename T>
__global__ void __launch_bounds__(64 * RED_WAVES) dyn_bias_reduce_kernel(const DynBiasParams p) {
    using E = Elem<T>;
    __shared__ float s_sum[RED_WAVES][64];
    const int Hk = p.Hk, K = Hk * p.d, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t per = (int64_t)Hk * K + 2 * Hk;
    const int64_t e = (int64_t)blockIdx.x * 64 + lane, ec = e < per ? e : per - 1;
    float s = 0.f;
    for (int c0 = wave; c0 < p.n_wg; c0 += 16 * RED_WAVES) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int c = c0 + u * RED_WAVES;
            v[u] = p.part[(int64_t)(c < p.n_wg ? c : wave) * p.part_stride + ec];
        }
#pragma unroll
        for (int u = 0; u < 16; u++) s += c0 + u * RED_WAVES < p.n_wg ? v[u] : 0.f;
    }
    s_sum[wave][lane] = s;
    __syncthreads();
    if (wave > 0 || e >= per) return;
#pragma unroll
    for (int w = 1; w < RED_WAVES; w++) s += s_sum[w][lane];
    const uint16_t out = (uint16_t)(E::pack2(s, 0.f) & 0xffffu);
    if (e < (int64_t)Hk * K) ((uint16_t *)p.dw)[e] = out;
    else if (e < (int64_t)Hk * K + Hk) ((uint16_t *)p.da)[e - (int64_t)Hk * K] = out;
    else if (p.dpb) ((uint16_t *)p.dpb)[e - (int64_t)Hk * K - Hk] = out;
}

}  // namespace

hipError_t launch_dyn_bias_fwd(const DynBiasParams &p, int dtype, hipStream_t stream) {
    const int64_t n_rows = (int64_t)p.B * p.L;
    if (n_rows <= 0) return hipSuccess;
    if (n_rows < 131072) {  // fewer than 4096 token tiles: split the columns over the waves as well
        const dim3 grid((unsigned)((n_rows + 31) / 32));
        if (dtype == 0) hipLaunchKernelGGL((dyn_bias_fwd_kernel<bf16_tag, true>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((dyn_bias_fwd_kernel<fp16_tag, true>), grid, dim3(256), 0, stream, p);
    } else {
        const dim3 grid((unsigned)((n_rows + 127) / 128));
        if (dtype == 0) hipLaunchKernelGGL((dyn_bias_fwd_kernel<bf16_tag, false>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((dyn_bias_fwd_kernel<fp16_tag, false>), grid, dim3(256), 0, stream, p);
    }
    return hipGetLastError();
}

// columns of V_flat per thread: four, where there are enough of them and the sums for them fit the registers
static bool four_columns(int Hk, int d) { return Hk <= 16 && Hk * d >= 1024; }

int dyn_bias_bwd_workgroups(int64_t n_rows, int Hk, int d, int *rows_per_wg) {
    // Runs of 32 tokens while the device holds all workgroups at a time (the partials are Hkv * Hkv * d floats each), else runs as long
    // as that takes, in whole eights.  A CU holds two workgroups of up to 8 heads with two columns a thread (105 registers) and one of
    // all others (161 to 256): with twice as many as that a second round starts, mostly empty.  us, kernel and fold, 512 / 256 workgroups:
    // 9000 tokens of 8 x 128 31.0 / 23.8, 16 x 256 140 / 92, 24 x 64 98.6 / 64.7; 16385 39.2 / 32.4, 183 / 136, 120 / 93; 33000 55.1 / 49.0, 280 / 233, 181 / 153;
    // 131072 155 / 149, 802 / 736, 553 / 534; 8 x 64, which fits twice: 33000 33.2 / 38.3, 98304 61 / 80.  (Runs of whole passes of 64 tokens
    // instead of whole eights: 33000 of 8 x 64 39.8.)
    const int most = (Hk <= 8 && !four_columns(Hk, d) ? 2 : 1) * device_cus();
    int64_t rows = 32;
    if ((n_rows + 31) / 32 > most) rows = ((n_rows + most - 1) / most + 7) / 8 * 8;
    *rows_per_wg = (int)rows;
    return (int)((n_rows + rows - 1) / rows);
}

hipError_t launch_dyn_bias_bwd(const DynBiasParams &p, int dtype, hipStream_t stream) {
    const int64_t n_rows = (int64_t)p.B * p.L;
    if (n_rows <= 0) return hipSuccess;
    const bool wide = four_columns(p.Hk, p.d);
    const int groups = (p.Hk * p.d + (wide ? 1023 : 511)) / (wide ? 1024 : 512);  // column groups of the kernel
    // (side by side where all of them run at once: a workgroup's time is its groups one behind the other.  us, before / now, the lane swaps of
    // the per-head sums among them: 500 tokens of 16 x 256 52.9 / 17.8, 122 of 16 x 96 28.2 / 15.6, 2396 of 8 x 96 18.4 / 10.4, 2048 of 16 x 128
    // 32.8 / 20.2; the sums alone: 4 x 2048 of 8 x 64 15.0 / 12.3, 83 of 4 x 128 11.5 / 8.5)
    const dim3 grid(p.n_wg, p.n_wg * groups <= device_cus() ? groups : 1);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(512), 0, stream, p); };
    if (dtype == 0) {
        if (p.Hk <= 8) wide ? go(dyn_bias_bwd_kernel<bf16_tag, 8, 4>) : go(dyn_bias_bwd_kernel<bf16_tag, 8, 2>);
        else if (p.Hk <= 16) wide ? go(dyn_bias_bwd_kernel<bf16_tag, 16, 4>) : go(dyn_bias_bwd_kernel<bf16_tag, 16, 2>);
        else go(dyn_bias_bwd_kernel<bf16_tag, 32, 2>);
    } else {
        if (p.Hk <= 8) wide ? go(dyn_bias_bwd_kernel<fp16_tag, 8, 4>) : go(dyn_bias_bwd_kernel<fp16_tag, 8, 2>);
        else if (p.Hk <= 16) wide ? go(dyn_bias_bwd_kernel<fp16_tag, 16, 4>) : go(dyn_bias_bwd_kernel<fp16_tag, 16, 2>);
        else go(dyn_bias_bwd_kernel<fp16_tag, 32, 2>);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t per = (int64_t)p.Hk * p.Hk * p.d + 2 * p.Hk;
    const dim3 fold((unsigned)((per + 63) / 64));
    if (dtype == 0) hipLaunchKernelGGL(dyn_bias_reduce_kernel<bf16_tag>, fold, dim3(64 * RED_WAVES), 0, stream, p);
    else hipLaunchKernelGGL(dyn_bias_reduce_kernel<fp16_tag>, fold, dim3(64 * RED_WAVES), 0, stream, p);
    return hipGetLastError();
}

}  // namespace fdma
