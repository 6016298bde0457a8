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
// Backward: a workgroup owns a run of tokens: d_dt = dBias * A * sigmoid(dt), dV = d_dt W and the run's share of dW = d_dt^T V_flat, dA and
// dpb, which go to fp32 partials that a second kernel folds in a fixed order (bit-reproducible).
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

// Backward, first stage: two contractions, dV = d_dt W over the heads and dW = d_dt^T V_flat over the tokens, on MFMA 16x16x4 in fp32
// (operands and sums stay 32 bits; twice the rate of the vector unit, which the products were bound by, and its registers spilled).
// A wave owns 128 columns of V_flat and 16 tokens at a time, workgroup (x, y) the tokens [x * rows_per_wg, ...) and col_waves such
// column ranges; what is left of its eight waves takes tiles of tokens in turn, and their dW meet in LDS at the end, in order.
//   * dW: lane (c, g) holds columns 8 c .. 8 c + 7 of tokens 4 q + g -- 16-byte loads, a row of 256 bytes per 16 lanes -- and step e takes
//     the e-th of them.  The sum of head j lies in lanes j, 16 + j, ..: 32 columns each.
//   * dV: the step's rows are columns 32 m + 8 (rho / 4) + 2 (rho % 4) + h of W, so a lane ends with eight columns of its token.
//   * d_dt of (token, head) is made in the lane that dV wants it in; dW wants it transposed: through a KB of LDS of the wave's own.
// HM = Hkv rounded up to 8, 16 or 32.  Bound by memory where there are many tokens (4 x 17701 of 16 x 64, 290 MB: 56 of the 92 at the rate of a
// copy), else by a chain of one trip to memory, three barriers and the fold.  us, kernel and fold, products on the vector unit by columns of
// one thread / now: 4 x 2048 of 8 x 64 14.6 / 11.3, 122 of 16 x 96 17.8 / 11.8, 2 x 8566 of 2 x 128 20.9 / 13.8, 4000 of 16 x 256 65.3 / 29.6,
// 33000 of 8 x 128 45.2 / 37.5, of 1 x 64 25.4 / 13.0, 4 x 17701 of 16 x 64 117 / 92, 131072 of 8 x 128 156 / 127.
constexpr int BWD_COLS = 128, BWD_TOK = 16, BWD_WAVES = 8;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_a8_t __attribute__((aligned(8)));

template <typename T, int HM>
__global__ void __launch_bounds__(64 * BWD_WAVES) __attribute__((amdgpu_waves_per_eu(HM <= 16 ? 4 : 2))) dyn_bias_bwd_kernel(const DynBiasParams p) {
    using E = Elem<T>;
    constexpr int NS = HM / 4, NB = (HM + 15) / 16;  // steps of dV over the heads; sixteens of heads
    constexpr int PITCH = 16 * NB + 4;
    __shared__ __attribute__((aligned(256))) char smem[BWD_WAVES * 8192 + 2 * BWD_WAVES * HM * 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
    const int Hk = p.Hk, K = Hk * p.d;
    const int col_waves = p.col_waves, tok_waves = BWD_WAVES / col_waves, cw = wave % col_waves, tw = wave / col_waves;
    const int k0 = ((int)blockIdx.y * col_waves + cw) * BWD_COLS;
    const int64_t row0 = (int64_t)blockIdx.x * p.rows_per_wg, n_rows = (int64_t)p.B * p.L;  // (fewer than 2^31 tokens: their values fill the memory)
    const int n_tok = (int)(row0 + p.rows_per_wg < n_rows ? p.rows_per_wg : n_rows - row0);
    const bool per_head = blockIdx.y == 0 && cw == 0;  // these waves make the sums of dA and dpb as well
    float *part_w = p.part + (int64_t)blockIdx.x * p.part_stride;
    float *s_wave = (float *)(smem + wave * 8192), *s_red = (float *)(smem + BWD_WAVES * 8192);

    // batch entry and position of token t of the tile whose first one is (b0, l0)
    auto place = [&](int b0, int l0, int t, int &b, int &l) {
        b = b0;
        l = l0 + t;
        while (l >= p.L) { l -= p.L; b++; }
    };
    u32x4_t vraw[4];
    uint16_t gb_raw[NS];
    float dt_raw[NS];
    const int kv = k0 + 8 * c < K ? k0 + 8 * c : 0, kv_head = kv / p.d;  // (columns beyond the last: any, their results go nowhere)
    const int64_t col_v = (int64_t)kv_head * p.v_h + (kv - kv_head * p.d);
    // requests tile i (tokens past the last one: it again)
    auto fetch = [&](int i) {
        const int at = 16 * i < n_tok ? 16 * i : n_tok - 1, left = n_tok - 1 - at;
        const uint32_t base = (uint32_t)row0 + (uint32_t)at;
        const int b0 = (int)(base / (uint32_t)p.L), l0 = (int)(base - (uint32_t)b0 * (uint32_t)p.L);
        int b, l;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            place(b0, l0, 4 * q + g < left ? 4 * q + g : left, b, l);
            vraw[q] = *(const u32x4_t *)((const uint16_t *)p.v + b * p.v_b + (int64_t)l * p.v_r + col_v);
        }
        const int t = c < left ? c : left;
        place(b0, l0, t, b, l);
        int g_mine = g;
        asm volatile("" : "+v"(g_mine));  // (where the heads' rows begin is not kept over the tiles: registers)
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int j = 4 * s + g_mine < Hk ? 4 * s + g_mine : 0;
            gb_raw[s] = ((const uint16_t *)p.dbias)[b * p.dbias_b + (int64_t)j * p.dbias_h + l];
            dt_raw[s] = p.dt[(int64_t)(base + (uint32_t)t) * Hk + j];
        }
    };

    f32x4_t dw[NB][8];
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int e = 0; e < 8; e++) dw[nb][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float sum_a[NS], sum_pb[NS], a_mine[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) sum_a[s] = sum_pb[s] = 0.f;

    if (k0 < K && 16 * tw < n_tok) {
        fetch(tw);
        uint32_t wraw[4][NS];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int j = 4 * s + g < Hk ? 4 * s + g : 0;
            const uint32_t keep = 4 * s + g < Hk ? 0xffffffffu : 0u;
            a_mine[s] = E::lo((uint32_t)((const uint16_t *)p.a)[j] & keep);
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const int col = k0 + 32 * m + 8 * (c >> 2) + 2 * (c & 3);
                wraw[m][s] = *(const uint32_t *)((const uint16_t *)p.w + (int64_t)j * K + (col < K ? col : 0)) & keep;
            }
        }
        uint32_t heads = 0;  // a byte each: the heads that this lane's four pieces of a dV row lie in
#pragma unroll
        for (int m = 0; m < 4; m++) heads |= (uint32_t)((k0 + 32 * m + 8 * g) / p.d & 0xff) << (8 * m);
        for (int i = tw; 16 * i < n_tok; i += tok_waves) {
            const int left = n_tok - 16 * i;
            // d_dt, where dV wants it and in LDS
            float ddt[NS];
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const float gb = E::lo((uint32_t)gb_raw[s]), dt = dt_raw[s];
                const bool ok = c < left && 4 * s + g < Hk;
                ddt[s] = ok ? gb * a_mine[s] * sigmoid_f(dt) : 0.f;
                if (per_head) {
                    sum_a[s] += ok ? gb * softplus_f(dt) : 0.f;
                    sum_pb[s] += ddt[s];
                }
                s_wave[c * PITCH + 4 * s + g] = ddt[s];
            }
            __builtin_amdgcn_wave_barrier();  // (the LDS operations of one wave execute in order)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t keep = 4 * q + g < left ? 0xffffffffu : 0u;  // (an infinity past the last token is not multiplied by its zero)
                float dd[NB];
#pragma unroll
                for (int nb = 0; nb < NB; nb++) dd[nb] = s_wave[(4 * q + g) * PITCH + 16 * nb + (HM < 16 ? c & (HM - 1) : c)];
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const uint32_t x = vraw[q][e / 2] & keep;
#pragma unroll
                    for (int nb = 0; nb < NB; nb++) {
                        dw[nb][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(E::lo(x), dd[nb], dw[nb][e], 0, 0, 0);
                        dw[nb][e + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(E::hi(x), dd[nb], dw[nb][e + 1], 0, 0, 0);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
            if (16 * (i + tok_waves) < n_tok) fetch(i + tok_waves);  // (on its way while dV is made)
            int b, l;
            {
                const uint32_t base = (uint32_t)row0 + (uint32_t)(16 * i);
                const int b0 = (int)(base / (uint32_t)p.L);
                place(b0, (int)(base - (uint32_t)b0 * (uint32_t)p.L), c < left ? c : 0, b, l);
            }
            asm volatile("" : "+v"(heads));  // (the places themselves, computed in front of the loop, are eight registers)
            uint16_t *orow = (uint16_t *)p.dv + b * p.dv_b + (int64_t)l * p.dv_r;
#pragma unroll
            for (int m = 0; m < 4; m++) {
                if (k0 + 32 * m < K) {
                    f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < NS; s++) {
                        asm volatile("" : "+v"(wraw[m][s]));  // (kept packed: unpacked in front of the loop it is twice the registers)
                        lo = __builtin_amdgcn_mfma_f32_16x16x4f32(E::lo(wraw[m][s]), ddt[s], lo, 0, 0, 0);
                        hi = __builtin_amdgcn_mfma_f32_16x16x4f32(E::hi(wraw[m][s]), ddt[s], hi, 0, 0, 0);
                    }
                    u32x4_t out;
#pragma unroll
                    for (int x = 0; x < 4; x++) out[x] = E::pack2(lo[x], hi[x]);
                    const int kd = k0 + 32 * m + 8 * g, head = (int)(heads >> (8 * m) & 0xffu);
                    if (c < left && kd < K) *(u32x4_a8_t *)(orow + head * p.dv_h + (kd - head * p.d)) = out;
                }
            }
        }
    }
    // dW: lane (j, g) has columns 32 g + 4 r .. of head j in piece r = 2 i + e / 4 of eight; a wave adds up its share of the pieces
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        auto store = [&](int r, f32x4_t x) {
            const int j = 16 * nb + c, col = k0 + 32 * g + 4 * r;
            if (j < Hk && col < K) *(f32x4_t *)(part_w + (int64_t)j * K + col) = x;
        };
        auto piece = [&](int r) {
            const int i = r >> 1, e = (r & 1) * 4;
            return f32x4_t{dw[nb][e][i], dw[nb][e + 1][i], dw[nb][e + 2][i], dw[nb][e + 3][i]};
        };
        if (tok_waves == 1) {
#pragma unroll
            for (int r = 0; r < 8; r++) store(r, piece(r));
            continue;
        }
        if (nb) __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; r++) *(f32x4_t *)(s_wave + (r * 64 + lane) * 4) = piece(r);
        __syncthreads();
        for (int r = tw * (8 / tok_waves); r < (tw + 1) * (8 / tok_waves); r++) {
            const float *src = (const float *)(smem + cw * 8192) + (r * 64 + lane) * 4;
            f32x4_t x = *(const f32x4_t *)src;
            for (int w = 1; w < tok_waves; w++) x += *(const f32x4_t *)(src + w * col_waves * 2048);
            store(r, x);
        }
    }
    // dA and dpb: the sixteen tokens' lanes by swaps, then the waves in order
    if (blockIdx.y) return;
    auto fold = [&](float x) -> float {
        auto ror = [&](auto ctrl) { x += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), decltype(ctrl)::value, 0xf, 0xf, false)); };
        ror(std::integral_constant<int, 0x128>{});  // row_ror: 8, 4, 2, 1
        ror(std::integral_constant<int, 0x124>{});
        ror(std::integral_constant<int, 0x122>{});
        ror(std::integral_constant<int, 0x121>{});
        return x;
    };
    if (cw == 0) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float sa = fold(sum_a[s]), sb = fold(sum_pb[s]);
            if (c == 0) {
                s_red[tw * HM + 4 * s + g] = sa;
                s_red[(BWD_WAVES + tw) * HM + 4 * s + g] = sb;
            }
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < Hk) {
        float sa = 0.f, sb = 0.f;
        for (int w = 0; w < tok_waves; w++) {
            sa += s_red[w * HM + threadIdx.x];
            sb += s_red[(BWD_WAVES + w) * HM + threadIdx.x];
        }
        part_w[(int64_t)Hk * K + threadIdx.x] = sa;
        part_w[(int64_t)Hk * K + Hk + threadIdx.x] = sb;
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

// runs of tokens at most (their partial results, Hkv * Hkv * d floats each, cost what a run does)
static int most_runs(int Hk, int d) { return (Hk <= 8 && Hk * d < 1024 ? 2 : 1) * device_cus(); }

// The size of the workspace: a partial result for every 32 tokens or, where those are more than the most, for runs of whole eights.
int dyn_bias_bwd_parts(int64_t n_rows, int Hk, int d) {
    const int most = most_runs(Hk, d);
    int64_t rows = 32;
    if ((n_rows + rows - 1) / rows > most) rows = ((n_rows + most - 1) / most + 7) / 8 * 8;
    return (int)((n_rows + rows - 1) / rows);
}

// Runs of tokens (what it returns: as many as dyn_bias_bwd_parts or fewer), their length, and the column ranges that a workgroup takes.
int dyn_bias_bwd_workgroups(int64_t n_rows, int Hk, int d, int *rows_per_wg, int *col_waves) {
    const int groups = (Hk * d + BWD_COLS - 1) / BWD_COLS, cus = device_cus(), most = most_runs(Hk, d);
    // Few tokens: a tile each for the eight waves of a workgroup of one column range; fewest partial results.  Up to two rounds of the two
    // workgroups that a CU holds: us, up to one / two: 9000 tokens of 16 x 64 26.5 / 23.0, 4000 of 16 x 256 34.4 / 29.6, 9000 of 8 x 128
    // 19.5 / 18.7, 30000 of 8 x 64 25.5 / 26.4.
    if ((n_rows + 127) / 128 * groups <= 4 * cus && n_rows <= 64 * most) {
        *rows_per_wg = BWD_WAVES * BWD_TOK;
        *col_waves = 1;
        return (int)((n_rows + 127) / 128);
    }
    // Else up to four column ranges to a workgroup, two waves each; eight, one each, where the registers of more than 16 heads leave room
    // for one workgroup on a CU, or more than 16 ranges are rounds of their own (us, two / four / eight: 4 x 17701 of 16 x 64 92 / 92 / 101,
    // 33000 of 8 x 128 39.7 / 37.5 / 39.4, of 32 x 64 196 / 175 / 167, 9000 of 16 x 256 66.7 / 60.8 / 55.6).
    const int side = Hk > 16 || groups > 16 ? BWD_WAVES : BWD_WAVES / 2, in_turn = (groups + side - 1) / side;
    *col_waves = (groups + in_turn - 1) / in_turn;
    int64_t rows = 2 * BWD_TOK;
    if ((n_rows + rows - 1) / rows > most) rows = ((n_rows + most - 1) / most + BWD_TOK - 1) / BWD_TOK * BWD_TOK;
    *rows_per_wg = (int)rows;
    return (int)((n_rows + rows - 1) / rows);
}

hipError_t launch_dyn_bias_bwd(const DynBiasParams &p, int dtype, hipStream_t stream) {
    const int64_t n_rows = (int64_t)p.B * p.L;
    if (n_rows <= 0) return hipSuccess;
    const int groups = (p.Hk * p.d + BWD_COLS - 1) / BWD_COLS, waves = p.col_waves * (BWD_WAVES / p.col_waves);
    const dim3 grid(p.n_wg, (groups + p.col_waves - 1) / p.col_waves);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64 * waves), 0, stream, p); };
    if (dtype == 0) {
        if (p.Hk <= 8) go(dyn_bias_bwd_kernel<bf16_tag, 8>);
        else if (p.Hk <= 16) go(dyn_bias_bwd_kernel<bf16_tag, 16>);
        else go(dyn_bias_bwd_kernel<bf16_tag, 32>);
    } else {
        if (p.Hk <= 8) go(dyn_bias_bwd_kernel<fp16_tag, 8>);
        else if (p.Hk <= 16) go(dyn_bias_bwd_kernel<fp16_tag, 16>);
        else go(dyn_bias_bwd_kernel<fp16_tag, 32>);
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
