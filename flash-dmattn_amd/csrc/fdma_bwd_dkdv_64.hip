// Backward dynamic-mask attention for gfx950, general form (mask and / or bias vary per query row), head dims up to 64, rows of
// whole aligned chunks: the dK / dV / dBias kernel.
//
// Same math, work items and outputs as bwd_dkdv_kernel (fdma_bwd.hip; compute_dq_dk_dv_1colblock,
// csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the reference).  That kernel brings mask and bias through registers into a
// fused tile: at two workgroups per CU its staging registers spill, and every step waits for its own loads and its own stores.
//
// Here a workgroup is 4 waves over 128 keys (32 per wave), two on a CU, and a step is 32 query rows of one head:
//   * Everything comes straight into LDS (global_load_lds), requested two steps ahead into three stages: Q, dO and the row statistics
//     for all waves; bias and mask of a wave's own 32 keys, by the wave and for itself alone.  A wave waits for its loads by count and
//     meets the others once per step, where Q and dO change hands.
//   * A lane owns a key.  Its bias values and mask bytes of eight rows are columns of row-major tiles: transposing reads.
//   * dS takes the place of the wave's bias elements and leaves in 64-byte pieces of rows, by the wave that made it.
//   * The part of a per-query dBias above the causal diagonal, which no step visits, is written between the steps, by the workgroup
//     of the mirrored key block: the fewer steps a block has, the more of it there is to clear.  (Nobody reads it soon: stores
//     that stay out of the caches, 510 -> 473 us below.)
// A bias that heads share (BIAS_SUM) is summed over the group in registers; the group's heads follow each other.
// Bound by memory where every head has rows of its own: a kernel that only reads mask and bias and writes dBias in this order takes
// 440-450 us of the 473 at B = 2, L = 4096, H = 16 (300 with everything in L2).  Two workgroups of 190 registers and 61 KB: three of
// 168 spill (670 us).  bwd_dkdv_kernel / now, causal, bf16 (us): that shape 640 / 473; B = 2, L = 2048, H = 16, Hk = 4, heads sharing
// rows 201 / 102; L = 2048, H = 8, one bias value per key 39.7 / 27.4.
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int D = 64;
constexpr int NT = 256;
constexpr int BM = 32;    // query rows per step
constexpr int BN = 128;   // keys per workgroup
constexpr int KS = D / 16, DB = D / 32;
constexpr int ROW = D * 2;
constexpr int TILE = BM * ROW;

// what the bias is: none, one value per key, a row per query (whose dBias is dS), one that the heads of a group share (dS summed)
enum { BIAS_NONE, BIAS_COL, BIAS_ROWS, BIAS_SUM };

template <int BIAS> struct Smem {
    static constexpr bool ROWS = BIAS >= BIAS_ROWS;
    static constexpr int OFF_STAT = 2 * TILE;               // LSE, D: 64 floats each (what a direct load of a wave fills)
    static constexpr int OFF_WAVE = OFF_STAT + 512;         // per wave: bias rows of 64 bytes, mask rows of 32
    static constexpr int WB = ROWS ? BM * 64 : 0, WAVE = WB + BM * 32;
    static constexpr int STAGE = OFF_WAVE + 4 * WAVE;
    static constexpr int NST = 3;
    static constexpr int TOTAL = NST * STAGE;
    static_assert(STAGE % 256 == 0, "stages keep the bank alignment the swizzle is made for");
    static_assert(2 * TOTAL <= 160 * 1024, "two workgroups per CU");
};


typedef int v2i32_t __attribute__((ext_vector_type(2)));
// sixteen lanes read an 8 x 16 tile of bytes: lane i passes the address of bytes 8 (i & 1) .. of row i / 2 and gets column i
__device__ __forceinline__ u32x2_t lds_ld_tr8(uint32_t addr) {
    return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i32_t *)(uintptr_t)addr));
}

template <typename T, bool CAUSAL, bool BITS, int BIAS>
__global__ void __launch_bounds__(NT, 2) bwd_dkdv_64_kernel(const BwdParams p) {
    using E = Elem<T>;
    using SM = Smem<BIAS>;
    constexpr bool ROWS = SM::ROWS;
    constexpr int STAGE = SM::STAGE, NST = SM::NST;
    constexpr int N_DMA = 4 + (ROWS ? 2 : 0);  // direct loads of a wave per step: Q, dO, statistics, mask, bias
    constexpr int N_ST = BIAS == BIAS_ROWS ? 2 : 0;  // stores of a wave per step
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    // linear workgroup id -> (key block, segment, kv head, batch), key block OUTERMOST and ascending: under causal masking
    // the low key blocks are seen by the most queries, so the heaviest workgroups of every head start first
    const int hb_count = f.Hk * f.B, segs = p.kv_segs, part_id = (int)blockIdx.x;
    const int n_block = part_id / (hb_count * segs), seg = (part_id / hb_count) % segs, hk = (part_id % hb_count) % f.Hk, b = (part_id % hb_count) / f.Hk;
    const int G = f.H / f.Hk;
    const int n0 = n_block * BN, nw = n0 + wave * 32;
    const int key = nw + r;  // the key column this lane owns
    const int shift = f.Lk - f.Lq;

    const int M_blocks = (f.Lq + BM - 1) / BM;
    auto first_block = [&](int n) -> int {  // of the query blocks that see keys n ..
        const int first_q = n - shift, m = first_q > 0 ? first_q / BM : 0;
        return !CAUSAL ? 0 : (m > M_blocks ? M_blocks : m);
    };
    const int m_start = first_block(n0);
    // this workgroup's segment of the query blocks that see its keys (general_kv_segments), from the last one down.  Heads innermost
    // where they share the dBias rows; outermost where a column sum per bias head is kept.
    const int m_lo = (M_blocks - m_start) * seg / segs, n_m = (M_blocks - m_start) * (seg + 1) / segs - m_lo;
    const int n_steps = n_m * G;

    // ---- dBias above the diagonal: rows 0 .. z_rows - 1 of the mirrored key block, 16 rows x 128 keys at a time, one store of every
    // wave each (rows and keys beyond the ends clear a valid piece once more: the number of stores is fixed)
    const bool per_head = f.Hb == f.H;
    int z_left = 0, z_head = 0, z_row = 0, z_rows = 0;
    const int z_key = ((int)gridDim.x / (hb_count * segs) - 1 - n_block) * BN;
    char *z_base = nullptr;
    const uint32_t db_r2 = ROWS ? (uint32_t)(p.db_r * 2) : 0;
    const int64_t db_h2 = ROWS && per_head ? p.db_h * 2 : 0;  // bytes from one head of the group to the next
    const int64_t db_off = ROWS ? b * p.db_b + (f.Hb == 1 ? 0 : per_head ? hk * G : hk) * p.db_h : 0;
    uint32_t z_col = 0;
    if (ROWS && CAUSAL) {
        z_rows = first_block(z_key) * BM;
        z_rows = z_rows < f.Lq ? z_rows : f.Lq;
        const int per = (z_rows + 15) / 16, all = per * (per_head ? G : 1);
        const int z0 = (int)((int64_t)all * seg / segs);
        z_left = (int)((int64_t)all * (seg + 1) / segs) - z0;
        z_head = per > 0 ? z0 / per : 0;
        z_row = (z0 - z_head * per) * 16;
        z_base = (char *)((uint16_t *)p.dbias + db_off + z_key) + z_head * db_h2;
        z_col = (uint32_t)(z_key + 8 * (tid & 15) < f.Lk ? 16 * (tid & 15) : 0);
    }
    auto clear_one = [&]() {
        const RowPiece at = row_piece(z_row, z_rows, tid >> 4, db_r2);
        __builtin_nontemporal_store(u32x4_t{0, 0, 0, 0}, (u32x4_t *)(z_base + at.base + (at.off + z_col)));
        z_left--;
        z_row += 16;
        if (z_row >= z_rows) {
            z_row = 0;
            z_base += db_h2;
        }
    };

    // ---- stationary K / V fragments (B operands)
    u32x4_t kf[KS], vf[KS];
    {
        const int key_c = key < f.Lk ? key : f.Lk - 1;
        const uint16_t *kp = (const uint16_t *)f.k + b * f.k_b + (int64_t)key_c * f.k_r + hk * f.k_h;
        const uint16_t *vp = (const uint16_t *)f.v + b * f.v_b + (int64_t)key_c * f.v_r + hk * f.v_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            kf[ks] = vf[ks] = u32x4_t{0, 0, 0, 0};
            if (c < f.d) {
                kf[ks] = *(const u32x4_t *)(kp + c);
                vf[ks] = *(const u32x4_t *)(vp + c);
            }
        }
    }
    const bool has_mask = f.mask != nullptr;
    const uint32_t no_mask = has_mask ? 0u : 0x80808080u;
    auto column_bias = [&](int h) -> float {
        if (BIAS != BIAS_COL) return 0.f;
        const int hb = f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk);
        return E::lo((uint32_t)((const uint16_t *)f.bias)[b * f.bi_b + hb * f.bi_h + (key < f.Lk ? key : f.Lk - 1)]);
    };

    // ---- direct loads of a step.  Q, dO: wave w fetches rows 8 w .. 8 w + 7; a lane fills chunk position lane % 8 of its row, which
    // holds chunk position ^ chunk_swz(row) of the global row.  Rows beyond the queries repeat the last one, and chunks beyond the keys a
    // valid one (masked where used); chunks beyond d repeat chunk 0 (they meet zeros).
    auto load16 = [](uint32_t off, gptr_t base, uint32_t dst) {
        load_lds16(off, base, __builtin_amdgcn_readfirstlane(dst));
    };
    auto load4 = [](uint32_t off, gptr_t base, uint32_t dst) {
        load_lds4(off, base, __builtin_amdgcn_readfirstlane(dst));
    };
    const int prow = 8 * wave + (lane >> 3);
    const int pchunk = (lane & 7) ^ (int)chunk_swz<64>(prow);
    const uint32_t pcol = pchunk * 8 < f.d ? pchunk * 16 : 0;
    const uint32_t q_r2 = (uint32_t)(f.q_r * 2), do_r2 = (uint32_t)(p.do_r * 2);
    const uint32_t bi_r2 = ROWS ? (uint32_t)(f.bi_r * 2) : 0, m_r1 = BITS ? (uint32_t)f.mb_r : (has_mask ? (uint32_t)f.m_r : 0);
    const bool w_live = nw < f.Lk;                            // this wave has keys (rows of 8 of them)
    const int bchunk = nw + 8 * (lane & 3) < f.Lk ? lane & 3 : 0;
    const uint32_t bcol = w_live ? (uint32_t)(nw + 8 * bchunk) * 2 : 0;
    const uint32_t mcol = !has_mask || !w_live ? 0 : BITS ? (uint32_t)nw / 8 : (uint32_t)(nw + (nw + 16 * (lane & 1) < f.Lk ? 16 * (lane & 1) : 0));
    // bases of the group's first head, and bytes from one head, and one row, to the next
    const int h0 = hk * G;
    const int64_t q_h2 = f.q_h * 2, do_h2 = p.do_h * 2;
    const char *q_base = (const char *)((const uint16_t *)f.q + b * f.q_b + h0 * f.q_h), *do_base = (const char *)((const uint16_t *)p.dout + b * p.do_b + h0 * p.do_h);
    // (even waves fetch the LSE values, odd ones D, all the same)
    const int st_h = wave & 1 ? p.Lq_rounded : f.Lq;
    const float *st_base = (wave & 1 ? p.softmax_d : f.lse) + ((int64_t)b * f.H + h0) * st_h;
    const int hm = f.Hm == 1 ? 0 : f.Hm == f.H ? h0 : hk;
    const int64_t m_h1 = has_mask && f.Hm == f.H ? (BITS ? f.mb_h : f.m_h) : 0;
    const uint8_t *m_base = !has_mask ? (const uint8_t *)f.k : BITS ? f.mbits + b * f.mb_b + hm * f.mb_h : f.mask + b * f.m_b + hm * f.m_h;
    const int64_t bi_h2 = ROWS && per_head ? f.bi_h * 2 : 0;
    const char *bi_base = ROWS ? (const char *)((const uint16_t *)f.bias + b * f.bi_b + (f.Hb == 1 ? 0 : per_head ? h0 : hk) * f.bi_h) : nullptr;
    // offsets of this lane's pieces: its row (clamped per step: offsets grow with the row), its column
    const uint32_t q_row = prow * q_r2, do_row = prow * do_r2, m_row = (uint32_t)(BITS ? r : lane >> 1) * m_r1, bi_row = (uint32_t)(lane >> 2) * bi_r2;
    auto least = [](uint32_t x, uint32_t y) { return x < y ? x : y; };

    int dma_gi = 0, dma_mi = M_blocks - 1 - m_lo, dma_stage = 0;  // the step being fetched
    const int mi_last = M_blocks - m_lo - n_m;
    auto advance = [&](int &gi, int &mi) {
        if (ROWS) {
            if (++gi == G) { gi = 0; mi--; }
        } else if (mi-- == mi_last) {
            mi = M_blocks - 1 - m_lo;
            gi++;
        }
    };
    auto dma_step = [&](bool more) {  // all loads of that step; then on to the following one (past the last it is fetched again)
        const int m0 = dma_mi * BM;
        const int left = f.Lq - 1 - m0;
        const uint32_t rows = (uint32_t)(left < BM - 1 ? left : BM - 1);
        const uint32_t st = lds0 + (uint32_t)(dma_stage * STAGE), sw = st + SM::OFF_WAVE + wave * SM::WAVE;
        load16(least(q_row, rows * q_r2) + pcol, uniform_ptr(q_base + dma_gi * q_h2 + (int64_t)m0 * q_r2), st + wave * 1024);
        load16(least(do_row, rows * do_r2) + pcol, uniform_ptr(do_base + dma_gi * do_h2 + (int64_t)m0 * do_r2), st + TILE + wave * 1024);
        load4(least((uint32_t)r, rows) * 4, uniform_ptr(st_base + dma_gi * st_h + m0), st + SM::OFF_STAT + (wave & 1) * 256);
        const gptr_t mb = uniform_ptr(m_base + dma_gi * m_h1 + (int64_t)m0 * m_r1);
        if (BITS) load4(least(m_row, rows * m_r1) + mcol, mb, sw + SM::WB);
        else load16(least(m_row, rows * m_r1) + mcol, mb, sw + SM::WB);
        if (ROWS) {
            const gptr_t bb = uniform_ptr(bi_base + dma_gi * bi_h2 + (int64_t)m0 * bi_r2);
#pragma unroll
            for (int i = 0; i < 2; i++) load16(least(bi_row + 16 * i * bi_r2, rows * bi_r2) + bcol, bb, sw + i * 1024);
        }
        dma_stage = dma_stage == NST - 1 ? 0 : dma_stage + 1;
        if (more) advance(dma_gi, dma_mi);
    };

    // fragment addresses (stage 0): rows of Q (dO: + TILE); transposing reads of either, of the wave's bias and of its mask
    const int frow = pi_row(r);
    const uint32_t a_off = lds0 + (uint32_t)frow * ROW + (((uint32_t)g ^ chunk_swz<64>(frow)) << 4);
    const TrLane tr = tr_lane(lane);
    const uint32_t tr_off = lds0 + tr_chunk<64>(g, tr);
    const uint32_t w_off = lds0 + SM::OFF_WAVE + wave * SM::WAVE;
    const uint32_t bt_off = w_off + (8 * g + tr.te) * 64 + 32 * tr.tdh + 8 * tr.tc;
    const uint32_t mt_off = w_off + SM::WB + (BITS ? 32 * g : (8 * g + ((lane & 15) >> 1)) * 32 + 16 * tr.tdh + 8 * (lane & 1));
    const uint32_t ds_off = w_off + (8 * g) * 64 + 2 * r;
    const uint32_t stat_off = lds0 + SM::OFF_STAT + 32 * g;

    f32x16_t dk[DB], dv[DB], dsum;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dk[db][i] = dv[db][i] = dsum[i] = 0.f;
    float colsum = 0.f;  // row-broadcast dbias: sum over queries of dS for this lane's key

    int gi = 0, mi = M_blocks - 1 - m_lo, stage = 0;
    int z_two = 0, z_last = 0;  // clearing stores of the last two steps, of the last one
    float cb = 0.f;
    if (n_steps > 0) {
        cb = column_bias(hk * G);
        dma_step(n_steps > 1);
        dma_step(n_steps > 2);
    }
    for (int step = 0; step < n_steps; step++) {
        const int m0 = mi * BM;
        const uint32_t st = (uint32_t)(stage * STAGE);
        // This step's loads have landed: behind them the wave has issued the next step's and, from the third step on, the stores of
        // two steps.  (Fewer than all of the clearing's are counted where it ends: a wait for more than is needed.)  Everybody has
        // left the stage before this one.
        if (N_ST && w_live && step >= 2) {
            if (z_two == 4) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N_DMA + 2 * N_ST + 4) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N_DMA + 2 * N_ST) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N_DMA) : "memory");
        }
        dma_step(step + 3 < n_steps);
        if (ROWS && CAUSAL) {
            const int two = z_left >= 2 ? 2 : 0;
            if (two) {
                clear_one();
                clear_one();
            }
            z_two = z_last + two;
            z_last = two;
        }

        // ---- S = Q K^T and dP = dO V^T: M = query, N = key
        f32x16_t s, dp;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = dp[i] = 0.f;
        {
            constexpr int NF = 2 * KS, FR = 4;
            u32x4_t a[NF];
            auto frag = [&](int x) { return lds_ld128(((a_off + st) ^ ((uint32_t)(x >> 1) << 5)) + (x & 1) * TILE); };
#pragma unroll
            for (int x = 0; x < FR; x++) a[x] = frag(x);
#pragma unroll
            for (int x = 0; x < NF; x++) {
                if (x + FR < NF) a[x + FR] = frag(x + FR);
                if (x & 1) dp = E::mfma(a[x], vf[x >> 1], dp);
                else s = E::mfma(a[x], kf[x >> 1], s);
            }
        }
        // ---- P = exp2((S * scale + bias - LSE) * log2e) where the mask keeps; dS = P * (dP - D)
        const bool edge = (CAUSAL && nw + 31 > m0 + shift) || m0 + BM > f.Lq || nw + 32 > f.Lk;
        uint32_t ppk[8], dpk[8];
        float part = 0.f;
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {  // registers 8 blk + e <-> row 16 blk + 8 g + e
            f32x4_t l[2], dd[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                l[q] = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + st + 64 * blk + 16 * q));
                dd[q] = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + st + 256 + 64 * blk + 16 * q));
            }
            u32x2_t bv[2];
            if (ROWS) {
#pragma unroll
                for (int q = 0; q < 2; q++) bv[q] = lds_ld_tr16(bt_off + st + blk * 1024 + q * 256);
            }
            uint32_t mw[BITS ? 8 : 2];
            if (BITS) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const u32x4_t x = lds_ld128(mt_off + st + 64 * blk + 16 * q);
#pragma unroll
                    for (int e = 0; e < 4; e++) mw[(4 * q + e) % (BITS ? 8 : 2)] = x[e];
                }
            } else {
                const u32x2_t x = lds_ld_tr8(mt_off + st + blk * 512);
#pragma unroll
                for (int q = 0; q < 2; q++) mw[q] = (((x[q] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x[q]) | no_mask;  // bit 7 of a byte: it is not zero
            }
            float pv[8], dsv[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float fb = ROWS ? ((e & 1) ? E::hi(bv[e >> 2][(e >> 1) & 1]) : E::lo(bv[e >> 2][(e >> 1) & 1])) : cb;
                const float x = (fmaf(s[8 * blk + e], f.scale, fb) - l[e >> 2][e & 3]) * kLog2e;
                const int keep = BITS ? __builtin_amdgcn_sbfe((int)mw[e % (BITS ? 8 : 2)], r, 1) : __builtin_amdgcn_sbfe((int)mw[(e >> 2) % 2], 8 * (e & 3) + 7, 1);
                pv[e] = __uint_as_float(__float_as_uint(fast_exp2(x)) & (uint32_t)keep);
            }
            if (edge) {  // rows above the diagonal or beyond the queries, keys beyond the end
                asm volatile("" ::: "memory");
                const int lim = key >= f.Lk ? BM : (CAUSAL ? key - shift - m0 : 0) - 16 * blk - 8 * g, lim_hi = f.Lq - m0 - 16 * blk - 8 * g;
#pragma unroll
                for (int e = 0; e < 8; e++) pv[e] = (e >= lim && e < lim_hi) ? pv[e] : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                dsv[e] = pv[e] * (dp[8 * blk + e] - dd[e >> 2][e & 3]);
                if (BIAS == BIAS_COL) part += dsv[e];
                if (BIAS == BIAS_SUM) dsum[8 * blk + e] = gi == 0 ? dsv[e] : dsum[8 * blk + e] + dsv[e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ppk[4 * blk + e] = E::pack2(pv[2 * e], pv[2 * e + 1]);
                dpk[4 * blk + e] = E::pack2(dsv[2 * e], dsv[2 * e + 1]);
            }
        }
        // dS over the bias elements it was made from: same rows, this lane's column
        const bool out = BIAS == BIAS_ROWS || (BIAS == BIAS_SUM && gi == G - 1);
        if (out) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t w = BIAS == BIAS_SUM ? E::pack2(dsum[2 * i], dsum[2 * i + 1]) : dpk[i];
                const uint32_t at = ds_off + st + (16 * (i >> 2) + 2 * (i & 3)) * 64;
                *(__attribute__((address_space(3))) uint16_t *)(uintptr_t)at = (uint16_t)w;
                *(__attribute__((address_space(3))) uint16_t *)(uintptr_t)(at + 64) = (uint16_t)(w >> 16);
            }
        }
        // ---- dV^T += dO^T P ; dK^T += Q^T dS
#pragma unroll
        for (int x = 0; x < 2 * DB; x++) {
            const int qb = x / DB, db = x % DB;
            const u32x4_t pb = {ppk[4 * qb], ppk[4 * qb + 1], ppk[4 * qb + 2], ppk[4 * qb + 3]};
            const u32x4_t sb = {dpk[4 * qb], dpk[4 * qb + 1], dpk[4 * qb + 2], dpk[4 * qb + 3]};
            const uint32_t lo = ((tr_off + st) ^ ((uint32_t)db << 6)) + qb * 16 * ROW, hi = ((tr_off + st) ^ (((uint32_t)db << 6) | 16u)) + (qb * 16 + 4) * ROW;
            const u32x2_t l1 = lds_ld_tr16(lo + TILE), h1 = lds_ld_tr16(hi + TILE), l2 = lds_ld_tr16(lo), h2 = lds_ld_tr16(hi);
            dv[db] = E::mfma(u32x4_t{l1[0], l1[1], h1[0], h1[1]}, pb, dv[db]);
            dk[db] = E::mfma(u32x4_t{l2[0], l2[1], h2[0], h2[1]}, sb, dk[db]);
        }
        // ---- dBias
        if (out && w_live) {  // (rows and chunks beyond the ends store a valid one once more: the number of stores is fixed)
            const uint32_t rows = (uint32_t)((f.Lq - m0 < BM ? f.Lq - m0 : BM) - 1);
            char *dbp = (char *)((uint16_t *)p.dbias + db_off + nw) + gi * db_h2 + (int64_t)m0 * db_r2;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t row = least((uint32_t)(16 * i + (lane >> 2)), rows);
                *(u32x4_t *)(dbp + (row * db_r2 + bchunk * 16)) = lds_ld128(w_off + st + row * 64 + bchunk * 16);
            }
        }
        if (BIAS == BIAS_COL) {
            colsum += part;
            if (mi == mi_last && (f.Hb == f.H || gi == G - 1)) {
                const float tot = xhalf_sum(colsum);
                const int hb = f.Hb == f.H ? hk * G + gi : (f.Hb == 1 ? 0 : hk);
                if (g == 0 && segs > 1) {
                    p.db_part[((int64_t)part_id * G + (f.Hb == f.H ? gi : 0)) * BN + wave * 32 + r] = tot;
                } else if (g == 0 && key < f.Lk) {
                    if (p.dbias_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + key, tot);
                    else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + key] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
                }
                colsum = 0.f;
            }
        }
        const int g_was = gi;
        advance(gi, mi);
        if (BIAS == BIAS_COL && gi != g_was && step + 1 < n_steps) cb = column_bias(hk * G + gi);
        stage = stage == NST - 1 ? 0 : stage + 1;
    }
    // (direct loads still in flight must not land in LDS that belongs to the next workgroup by then)
    __builtin_amdgcn_s_waitcnt(0x0070);
    if (ROWS && CAUSAL)
        while (z_left > 0) clear_one();

    // a key block that no query (of this segment) can see still owns its dbias column
    if (BIAS == BIAS_COL && n_steps == 0 && g == 0) {
        const int ngh = f.Hb == f.H ? G : 1;
        for (int gh = 0; gh < ngh; gh++) {
            const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
            if (segs > 1) p.db_part[((int64_t)part_id * G + gh) * BN + wave * 32 + r] = 0.f;
            else if (!p.dbias_accum && key < f.Lk) ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + key] = 0;
        }
    }
    if (segs > 1) {  // fp32 sums of this segment, in the order the lanes hold them (bwd_dkdv_sum_kernel)
        f32x4_t *dst = (f32x4_t *)p.dkv_part + (int64_t)part_id * 2 * BN * D / 4 + wave * DB * 4 * 64 + lane;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int at = (db * 4 + q) * 64;
                dst[at] = f32x4_t{dk[db][4 * q], dk[db][4 * q + 1], dk[db][4 * q + 2], dk[db][4 * q + 3]};
                dst[at + BN * D / 4] = f32x4_t{dv[db][4 * q], dv[db][4 * q + 1], dv[db][4 * q + 2], dv[db][4 * q + 3]};
            }
        return;
    }
    if (key < f.Lk) {  // dK (scaled) and dV
        uint16_t *dkp = (uint16_t *)p.dk + b * p.dk_b + (int64_t)key * p.dk_r + hk * p.dk_h;
        uint16_t *dvp = (uint16_t *)p.dv + b * p.dv_b + (int64_t)key * p.dv_r + hk * p.dv_h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const int c = 32 * db + 16 * blk + 8 * g;
                if (c < f.d) {
                    u32x4_t wk, wv;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        wk[e] = E::pack2(dk[db][8 * blk + 2 * e] * f.scale, dk[db][8 * blk + 2 * e + 1] * f.scale);
                        wv[e] = E::pack2(dv[db][8 * blk + 2 * e], dv[db][8 * blk + 2 * e + 1]);
                    }
                    *(u32x4_t *)(dkp + c) = wk;
                    *(u32x4_t *)(dvp + c) = wv;
                }
            }
    }
}

template <typename T, bool CAUSAL, bool BITS, int BIAS> hipError_t launch_one(const BwdParams &p, hipStream_t stream) {
    const FwdParams &f = p.f;
    auto kern = bwd_dkdv_64_kernel<T, CAUSAL, BITS, BIAS>;
    static DynSmemLimit smem_limit;
    const hipError_t e = smem_limit.ensure((const void *)kern, Smem<BIAS>::TOTAL);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(((f.Lk + BN - 1) / BN) * f.Hk * f.B * p.kv_segs), dim3(NT), Smem<BIAS>::TOTAL, stream, p);
    return hipGetLastError();
}
template <typename T, bool CAUSAL, bool BITS> hipError_t launch_bias(const BwdParams &p, hipStream_t stream) {
    const FwdParams &f = p.f;
    if (!f.bias) return launch_one<T, CAUSAL, BITS, BIAS_NONE>(p, stream);
    if (f.bi_r == 0) return launch_one<T, CAUSAL, BITS, BIAS_COL>(p, stream);
    return f.Hb == f.H || f.H == f.Hk ? launch_one<T, CAUSAL, BITS, BIAS_ROWS>(p, stream) : launch_one<T, CAUSAL, BITS, BIAS_SUM>(p, stream);
}
template <typename T> hipError_t launch_t(const BwdParams &p, hipStream_t stream) {
    if (p.f.mask && p.f.mbits) return p.f.causal ? launch_bias<T, true, true>(p, stream) : launch_bias<T, false, true>(p, stream);
    return p.f.causal ? launch_bias<T, true, false>(p, stream) : launch_bias<T, false, false>(p, stream);
}

}  // namespace

// Direct loads take aligned 16-byte pieces (bits: 4 bytes) with 32-bit offsets inside the rows of a step (or of a piece to clear); a per-query dBias that several
// workgroups add to goes through fp32 atomics, which bwd_dkdv_kernel has.
bool bwd_dkdv_64_applicable(const BwdParams &p) {
    const FwdParams &f = p.f;
    constexpr int64_t max_stride = (int64_t)1 << 24;
    if (f.d > 64 || f.cu_q || odd_rows(f) || f.Lk % 16 != 0 || f.Lq < 1 || (f.bias && f.bi_r != 0 && p.dbias_accum)) return false;
    if (f.mask && !f.mbits && (((uintptr_t)f.mask | (uintptr_t)f.m_b | (uintptr_t)f.m_h | (uintptr_t)f.m_r) & 15) != 0) return false;
    if (f.bias && f.bi_r != 0 && p.db_r >= max_stride) return false;
    return f.bi_r < max_stride && (f.mask ? (f.mbits ? f.mb_r : f.m_r) < max_stride : true);
}
hipError_t launch_bwd_dkdv_64(const BwdParams &p, int dtype, hipStream_t stream) {
    return dtype == 0 ? launch_t<bf16_tag>(p, stream) : launch_t<fp16_tag>(p, stream);
}

}  // namespace fdma
