// Forward dynamic-mask attention for gfx950, column-mask specialisation with key groups and direct loads: head dims 129 .. 256,
// and below on small grids (takes_key_groups in fdma_fwd_colmask.hip).
//
// Same math, inputs and reference counterparts as fdma_fwd_colmask.hip (compute_attn_1rowblock,
// csrc/flash_sparse_attn/src/flash_fwd_kernel.h:53-804 of the reference; mask and bias absent or broadcast over the query
// dimension).
//
// A workgroup is 8 waves, two to a SIMD: RG groups of 32 query rows times KG = 8 / RG groups of 32 keys, a tile being 32 KG
// keys.  Wave (rw, kg) takes its rows against its keys of every tile, with a softmax of its own; the key groups are merged
// through LDS at the end, each finishing its share of the head dim.
//   * Head dim 256, RG = 4: O alone is 128 registers per lane, Q another 64.  With four waves (one per SIMD, 448 registers,
//     nothing to hide behind) a step of 128 rows x 64 keys took 3.2 us for 0.85 us of matrix work, here 2.0.
//     On small grids RG = 2 (see launch_fwd_wide), with one stage: the next K tile is fetched under the softmax and P V, the next V
//     tile under the scores and the softmax, a barrier more for each.
//   * Head dim 128, RG = 2: 64-row blocks with four key groups are twice as many workgroups with half the chain of tiles.
//     A tile of 128 keys takes 1.4 us where the eight-wave kernel of fdma_fwd_colmask.hip takes 1.6 for 128 rows, on twice
//     the CUs.
//   * Head dim 64, RG = 2: two workgroups to a CU.
//   * K and V tiles go from global memory straight into LDS (global_load_lds, one tile ahead, issued between the MFMAs):
//     no staging registers.  The 16-byte chunks of a 256-byte row, or of the two halves of a 512-byte one, are swizzled as in
//     LdsTile<128>; V is row-major like K, and V^T comes from transposing LDS reads.
//   * The score accumulators start from the fused bias of their keys (fp32, -inf where the mask drops the key), read from an
//     LDS column; the softmax is the online one, with a reference point that moves only when a score exceeds it by 2^8.  Its
//     vector work runs under the MFMAs of the SIMD's other wave.
// LDS: two stages of 64 KB, or one of 128.  Bound by the chain of a tile (scores, softmax, P V, barrier) of two waves per SIMD: without the
// loads it is 0.25 us shorter, without the softmax 0.1.
// Before / now (us): 3001 tokens, 8/4 heads, d = 256, 1024 kept, fp16 57 / 38 (with the bias producer and the mask 75.6 / 56.3);
// 8192 tokens, 8/2 heads, d = 256, 4096 kept 203 / 152; 2300 ragged tokens and others, 16/8 heads, d = 256 152 / 115;
// d = 128: 512 rows x 32 heads against 2048 kept keys of 16384 42.7 / 35.6, 2000 tokens x 4 heads 39.7 / 32.4, 256 x 32 14.8 / 11.0;
// d = 64: 2176 x 16 42.4 / 29.4, 4 x 448 x 8 13.7 / 9.9, 512 x 32 against 2048 kept of 16384 32.9 / 25.9, ragged up to 4928 x 2 74 / 45.
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_fwd_merge.h"

namespace fdma {

namespace {

constexpr int NT = 512;
constexpr int MAX_TILES = 16384;

// RG row groups of 32 query rows, KG = 8 / RG key groups
template <int D_, int RG> struct Cfg {
    static constexpr int D = D_, KG = 8 / RG;
    static constexpr int BM = 32 * RG, BN = 32 * KG;      // query rows per workgroup, keys per tile
    static constexpr int ROW = D * 2, CH = D / 8;         // bytes and 16-byte chunks of a tile row
    static constexpr int TILE = BN * ROW;                 // a K or V tile
    static constexpr int RPP = 64 / CH;                   // rows of a 1 KB piece
    static constexpr int NP = TILE / 1024 / 8;            // pieces per wave of a K or V tile
    static constexpr bool ONE = 4 * TILE > 128 * 1024;    // one stage of K and of V instead of two
    static constexpr int OFF_V = (ONE ? 1 : 2) * TILE;
    static constexpr int OFF_COL = 2 * OFF_V;             // two stages of the fused bias column
    static constexpr int OFF_BITS = OFF_COL + 2 * BN * 4;
    static constexpr int LOOP_BYTES = OFF_BITS + MAX_TILES / 8;
    static constexpr int UPW = D / 16 / KG;               // merge: 16-wide units of O that a wave finishes
    static constexpr int PASSES = KG * (KG - 1) * RG * UPW * 2048 > 128 * 1024 ? 2 : 1, UPP = UPW / PASSES;  // ... in so many passes
    static constexpr int OFF_SUMS = KG * (KG - 1) * RG * UPP * 2048;  // the others' shares of a pass's units, then row sums and references
    static constexpr int MERGE_BYTES = OFF_SUMS + 2 * 8 * 64 * 4;
    static constexpr int SMEM = LOOP_BYTES > MERGE_BYTES + 16 ? LOOP_BYTES : MERGE_BYTES + 16;  // (a word behind the merge: last_share)
    static_assert(SMEM <= 160 * 1024, "one workgroup per CU");
    static_assert(UPW * KG * 16 == D, "every unit of O is finished by one key group");
    static_assert(8 * RPP % 16 == 0, "a wave's pieces lie rows of one swizzle apart");
};

// DC: the head dims that are worked on, 96 of a 128-wide tile for head dims 65 to 96 (the merge takes the others along as zeros).
// LIST (with CMP): the keys are those of a handed-over list, and K, V and bias are read where they lie (see fwd_from_lists).
template <typename T, int D, int DC, int RG, bool CAUSAL, bool CMP, bool LIST>
__device__ __forceinline__ void fwd_wide(const FwdParams &p) {
    using E = Elem<T>;
    using C = Cfg<D, RG>;
    constexpr int KG = C::KG, BM = C::BM, BN = C::BN, ROW = C::ROW, TILE = C::TILE, NP = C::NP, KS = DC / 16, DB = DC / 32;
    constexpr int OFF_V = C::OFF_V, OFF_COL = C::OFF_COL, OFF_BITS = C::OFF_BITS, UPW = C::UPW, UPP = C::UPP;
    static_assert(CMP || !LIST, "a list's keys are counted like compacted ones");
    constexpr bool ONE = C::ONE, SHARES = CMP && !LIST && D <= 128;  // (key_shares cuts nothing above)
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)
    uint32_t *sBits = (uint32_t *)(smem + OFF_BITS);

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int rw = wave % RG, kg = wave / RG;  // 32-row group and key group of this wave

    const RowUnit ru = row_unit(p, blockIdx.x, BM);
    const int part = SHARES ? (int)blockIdx.y : 0;  // (all first shares first: workgroups that turn out to have none come when CUs are free)
    if (ru.block < 0) return;
    const int b = ru.b, hk = ru.hk, h = ru.h;
    const int m0 = ru.block * BM;
    const SeqInfo sq = seq_info(p, b);
    const int LqS = sq.Lq, LkS = sq.Lk;
    const int shift = LkS - LqS;
    const int wrow0 = m0 + rw * 32, qrow = wrow0 + r;

    // ---- staging: a piece is 1 KB, whole rows; wave w fetches pieces w + 8 i of Q, of K and of V.  A lane fills chunk position
    // `lane % CH` of its row, which holds chunk position ^ chunk_swz(row) of the global row; rows 16 apart have the same swizzle.  Rows
    // beyond the keys (queries) are clamped to the last one (their column says -inf; they are not stored), chunks beyond d to chunk 0 (they
    // meet zero Q and columns of O that are not stored).
    int prow = C::RPP * wave + lane / C::CH;
    const int pchunk = lane % C::CH ^ (int)chunk_swz<D>(prow);
    const uint32_t pcol = pchunk * 8 < p.d ? pchunk * 16 : 0;

    // LIST: original columns of the keys of two tiles, the parity of a tile deciding where, held inside [0, Lk) (lists are device data the host
    // cannot check); those of the first tile are requested here and published with Q
    const int lrow = LIST ? (p.m_b == 0 ? 0 : b) * p.Hm + (p.Hm == 1 ? 0 : hk) : 0;
    const int32_t *list = LIST ? p.kept_idx + (int64_t)lrow * p.kept_ld : nullptr;
    auto column_at = [&](int c) { return list[c < LkS ? c : LkS - 1]; };
    const uint32_t idx_off = lds0 + OFF_BITS;
    int32_t list_raw = LIST ? column_at(tid) : 0;

    // ---- Q, requested first of all: through LDS, where the second stage of K (and of V) comes later, or V where there is one stage.
    // As fragments straight from memory every load of a wave touches 32 rows, one cache line after another (2.7 clocks each), and every key
    // group loads them again: of the 8 us that a workgroup of two tiles took at d = 128, 1.7 were spent on the lines of Q.  The kernel
    // before / now, us: 223 tokens x 32/8 heads, d = 128 11.1 / 9.4; 2 x 128 x 32/8, d = 64 7.4 / 6.1; 2 x 256 x 8/4, d = 256 17.6 / 13.8;
    // 2304 ragged tokens and others x 16/8, d = 256 133 / 118; 512 rows x 32/8 against 2048 kept of 16384 37.2 / 34.4.
    static_assert(BM * ROW <= (ONE ? 1 : 2) * TILE, "Q fits there");
    auto q_at = [](uint32_t byte) { return byte + (ONE || byte >= TILE ? OFF_V : TILE); };  // (V's second stage is as far behind V as K's end behind K)
    {
        // (offsets are not negative: rows that lie in descending order are counted from the last one)
        const bool down = p.q_r < 0;
        const int rows = LqS - 1 - m0 < BM - 1 ? LqS - 1 - m0 : BM - 1;
        const gptr_t qb = uniform_ptr((const uint16_t *)p.q + b * p.q_b + (sq.q0 + m0 + (down ? rows : 0)) * p.q_r + h * p.q_h);
        const uint32_t q_r2 = (uint32_t)((down ? -p.q_r : p.q_r) * 2), last = (uint32_t)rows * q_r2;
#pragma unroll
        for (int i = 0; i < BM * ROW / 8192; i++) {
            uint32_t at = (uint32_t)(prow + 8 * C::RPP * i) * q_r2;
            at = at < last ? at : last;
            load_lds16((down ? last - at : at) + pcol, qb, __builtin_amdgcn_readfirstlane(lds0 + q_at(8192 * i) + wave * 1024));
        }
    }

    const int hm = p.mask ? (p.Hm == p.H ? h : (p.Hm == 1 ? 0 : hk)) : 0;
    const int hb = p.bias ? (p.Hb == p.H ? h : (p.Hb == 1 ? 0 : hk)) : 0;
    const uint8_t *mrow = p.mask ? p.mask + b * p.m_b + hm * p.m_h : nullptr;
    const uint16_t *brow = p.bias ? (const uint16_t *)p.bias + b * p.bi_b + hb * p.bi_h : nullptr;
    const uint16_t *kbase = (const uint16_t *)p.k + b * p.k_b + sq.k0 * p.k_r + hk * p.k_h;
    const uint16_t *vbase = (const uint16_t *)p.v + b * p.v_b + sq.k0 * p.v_r + hk * p.v_h;

    // key columns this workgroup iterates over, and the number of them a query row may see
    int Lk = LIST ? p.kept_count[lrow] : CMP ? p.cmp.count[b * p.Hk + hk] : LkS;
    if (LIST) Lk = Lk < 0 ? 0 : (Lk < LkS ? Lk : LkS);
    const int32_t *ccnt = LIST ? p.kept_cnt + (int64_t)lrow * p.kept_ld : CMP ? p.cmp.cnt + (int64_t)(b * p.Hk + hk) * p.cmp.ld : nullptr;
    const float *fbrow = CMP && !LIST ? p.cmp.fb + (int64_t)(b * p.cmp.Hfb + (p.cmp.Hfb == p.H ? h : hk)) * p.cmp.ld : nullptr;
    const int vis_lane = CAUSAL ? visible_columns<CMP>(qrow, LqS, LkS, ccnt) : 0;  // columns below it pass the causal test for this lane's row
    const int vis_wave = CAUSAL ? visible_columns<CMP>(wrow0, LqS, LkS, ccnt) : 0;
    const int vis_block = CAUSAL ? visible_columns<CMP>(m0 + BM - 1, LqS, LkS, ccnt) : 0;
    int n_end = (Lk + BN - 1) / BN;
    if (CAUSAL) {
        const int ne = ((vis_block < 0 ? 0 : vis_block) + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }
    // this workgroup's share of the tiles (see fwd_key_splits)
    int t_first = 0, shares = 1;
    if (SHARES && p.splits > 1) {
        // (no share under 512 keys: the workgroups that are then left over end, and without counters say so)
        const int most = n_end * BN / 512 > 1 ? n_end * BN / 512 : 1;
        shares = p.splits < most ? p.splits : most;
        if (part >= shares) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (Q is not to land in what is another workgroup's LDS by then)
            if (!p.dec_counter && tid < BM && m0 + tid < LqS) p.lse_part[(((int64_t)part * p.B + b) * p.H + h) * p.Lq + m0 + tid] = -INFINITY;
            return;
        }
        t_first = n_end * part / shares;
        n_end = n_end * (part + 1) / shares;
    }

    // ---- active-tile bitmap (compacted keys: every tile is active)
    for (int base = 0; !CMP && base < n_end; base += NT) {
        const int j = base + tid;
        bool act = false;
        if (j < n_end) {
            if (mrow) {
                uint32_t any = 0;
                int col[BN / 16];
                u32x4_t mv[BN / 16];
#pragma unroll
                for (int c = 0; c < BN / 16; c++) col[c] = j * BN + c * 16;
                ld_row16(mrow, col, LkS, mv);
#pragma unroll
                for (int c = 0; c < BN / 16; c++) any |= mv[c][0] | mv[c][1] | mv[c][2] | mv[c][3];
                act = any != 0;
            } else {
                act = true;
            }
        }
        const uint64_t ball = __ballot(act);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (Q: landed with the mask row, which was requested behind it)
        if (lane == 0) {
            const int w0 = (base + wave * 64) >> 5;
            sBits[w0] = (uint32_t)ball;
            sBits[w0 + 1] = (uint32_t)(ball >> 32);
        }
    }
    auto keep_column = [&](int tile) {
        const uint32_t c = (uint32_t)list_raw, last = (uint32_t)LkS - 1;
        lds_st32(idx_off + (uint32_t)((tile & 1) * BN + tid) * 4, c < last ? c : last);
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (Q, which the barrier publishes)
    if (LIST && tid < BN) keep_column(0);
    __syncthreads();
    auto next_active = [&](int j) -> int {  // wave-uniform
        if (CMP) return j < n_end ? j : n_end;
        while (j < n_end) {
            const uint32_t w = __builtin_amdgcn_readfirstlane(lds_ld32(lds0 + OFF_BITS + 4 * (j >> 5))) >> (j & 31);
            if (w) {
                j += __builtin_ctz(w);
                return j < n_end ? j : n_end;
            }
            j = (j | 31) + 1;
        }
        return n_end;
    };

    // K and V of a tile (see above)
    const uint32_t k_r2 = (uint32_t)(p.k_r * 2), v_r2 = (uint32_t)(p.v_r * 2);
    uint32_t k_row = prow * k_r2, v_row = prow * v_r2;  // (offsets grow with the row: clamped by the last row's)
    gptr_t tb_k = nullptr, tb_v = nullptr;
    int t_rows = 0, t_stage = 0, t_tile = 0;  // last row of the tile being fetched, its stage, the tile
    uint32_t braw = 0, mraw = 0;     // first waves: raw bias and mask of key `tid` of that tile
    bool col_ok = false;
    auto set_tile = [&](int j, int stage) {
        tb_k = uniform_ptr(kbase + (LIST ? 0 : (int64_t)j * BN * p.k_r));
        tb_v = uniform_ptr(vbase + (LIST ? 0 : (int64_t)j * BN * p.v_r));
        t_tile = j;
        const int left = Lk - 1 - j * BN;
        t_rows = left < BN - 1 ? left : BN - 1;
        t_stage = stage;
        if (wave < BN / 64) {  // (raw, unconditional loads: an absent mask or bias is the first element of K, ignored)
            const int col = j * BN + tid;
            col_ok = col < Lk;
            const int cc = col_ok ? col : 0;
            if (LIST) {
                braw = (brow ? brow : kbase)[brow ? lds_ld32(idx_off + (uint32_t)((j & 1) * BN + tid) * 4) : 0];
                list_raw = column_at(col + BN);
            } else if (CMP) {
                braw = __float_as_uint(fbrow[cc]);
            } else {
                mraw = (mrow ? mrow : (const uint8_t *)kbase)[mrow ? cc : 0];
                braw = (brow ? brow : kbase)[brow ? cc : 0];
            }
        }
    };
    // (in assembly and waited for by hand: behind the compiler's builtin every LDS read waits for all LDS operations in flight)
    auto dma_piece = [&](int n) {  // NP pieces of K, NP of V
        const int i = n % NP;
        const uint32_t r2 = n < NP ? k_r2 : v_r2;
        uint32_t off;
        if constexpr (LIST) {  // (rows beyond the last kept key: it again)
            const int row = prow + 8 * C::RPP * i;
            off = lds_ld32(idx_off + (uint32_t)((t_tile & 1) * BN + (row < t_rows ? row : t_rows)) * 4) * r2 + pcol;
        } else {
            const uint32_t at = (n < NP ? k_row : v_row) + 8 * C::RPP * i * r2, last = (uint32_t)t_rows * r2;
            off = (at < last ? at : last) + pcol;
        }
        const uint32_t dst = lds0 + (n < NP ? 0 : OFF_V) + (uint32_t)((ONE ? 0 : t_stage * TILE) + (wave + 8 * i) * 1024);
        load_lds16(off, n < NP ? tb_k : tb_v, __builtin_amdgcn_readfirstlane(dst));
    };
    auto publish = [&]() {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's pieces have landed
        if (wave < BN / 64) {
            float v = 0.f;
            bool keep = col_ok;
            if (LIST) {
                if (brow) v = E::lo(braw) * kLog2e;
                keep_column(t_tile + 1);
            } else if (CMP) {
                v = __uint_as_float(braw);
            } else {
                keep = keep && (!mrow || mraw);
                if (brow) v = E::lo(braw) * kLog2e;
            }
            lds_st32(lds0 + OFF_COL + t_stage * BN * 4 + 4 * tid, __float_as_uint(keep ? v : -INFINITY));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    // fragment addresses (stage 0).  K: chunk 2 ks + g of row 32 kg + pi_row(r).  V^T: see LdsTile::tr_base.
    const int frow = 32 * kg + pi_row(r);
    uint32_t a_off = lds0 + (uint32_t)frow * ROW + (((uint32_t)g ^ chunk_swz<D>(frow)) << 4);
    uint32_t tr_off = lds0 + OFF_V + (uint32_t)(32 * kg) * ROW + tr_chunk<D>(g, tr_lane(lane));
    const uint32_t col_off = lds0 + OFF_COL + 128 * kg + 32 * g;

    f32x16_t o[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    float row_sum = 0.f, row_ref = -INFINITY;  // relative to exp2(row_ref); -inf: no visible key met yet

    int jc = next_active(t_first), jn = n_end;
    if (jc < n_end) {
        jn = next_active(jc + 1);
        set_tile(jc, 0);
#pragma unroll
        for (int n = 0; n < (ONE ? NP : 2 * NP); n++) dma_piece(n);
    }
    // ---- Q fragments (B operands): chunk 2 ks + g of row 32 rw + r, scaled by softmax_scale * log2(e) once (the reference also rounds
    // the scaled Q to the input type, flash_fwd_kernel.h:428-439)
    u32x4_t qf[KS];
    {
        const int row = 32 * rw + r;
        const uint32_t at = lds0 + q_at(32 * rw * ROW) + (uint32_t)(r * ROW) + (((uint32_t)g ^ chunk_swz<D>(row)) << 4);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) qf[ks] = lds_ld128((at ^ ((uint32_t)(ks & 7) << 5)) + (uint32_t)(ks >> 3) * 256);
    }
    if constexpr (ONE) {  // everybody has read Q: V takes its place
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (jc < n_end) {
#pragma unroll
            for (int n = NP; n < 2 * NP; n++) dma_piece(n);
        }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = scaled8<T>(qf[ks], p.scale_log2, qrow < LqS && ks * 16 + g * 8 < p.d);
    if (jc < n_end) publish();

    auto one_tile = [&](auto st_c) {
        constexpr int st = decltype(st_c)::value;
        // (the swizzled addresses are these constants XOR a compile-time value, recomputed where used)
        if constexpr (LIST) asm volatile("" : "+v"(a_off), "+v"(tr_off), "+v"(prow));
        else asm volatile("" : "+v"(a_off), "+v"(tr_off), "+v"(k_row), "+v"(v_row));
        const int n0 = jc * BN + 32 * kg;
        set_tile(jn < n_end ? jn : jc, st ^ 1);  // (past the last tile it is fetched again and dropped)
        __builtin_amdgcn_sched_barrier(0);
        // ---- S^T = K Q^T on top of the fused bias of the keys
        f32x16_t s;
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            const f32x4_t b0 = __builtin_bit_cast(f32x4_t, lds_ld128(col_off + st * BN * 4 + 64 * blk));
            const f32x4_t b1 = __builtin_bit_cast(f32x4_t, lds_ld128(col_off + st * BN * 4 + 64 * blk + 16));
#pragma unroll
            for (int e = 0; e < 4; e++) { s[8 * blk + e] = b0[e]; s[8 * blk + 4 + e] = b1[e]; }
        }
        {
            constexpr int FR = 4;
            u32x4_t a[KS];
            auto frag = [&](int ks) { return lds_ld128((a_off ^ ((uint32_t)(ks & 7) << 5)) + (uint32_t)((ONE ? 0 : st * TILE) + (ks >> 3) * 256)); };
#pragma unroll
            for (int ks = 0; ks < FR; ks++) a[ks] = frag(ks);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                if (ks + FR < KS) a[ks + FR] = frag(ks + FR);
                s = E::mfma(a[ks], qf[ks], s);
                if constexpr (!ONE) {
#pragma unroll
                    for (int n = ks * 2 * NP / KS; n < (ks + 1) * 2 * NP / KS; n++) dma_piece(n);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (ONE) {  // everybody has read this K tile: the next one takes its place
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int n = 0; n < NP; n++) dma_piece(n);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (CAUSAL && n0 + 32 > vis_wave) {
            asm volatile("" ::: "memory");  // (a branch: only diagonal tiles pay)
            const int lim = vis_lane - 1 - n0 - 8 * g;  // local columns 16 blk + e <= lim are visible
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = 16 * (i >> 3) + (i & 7) <= lim ? s[i] : -INFINITY;
        }
        // ---- online softmax
        float tmax = s[0];
#pragma unroll
        for (int i = 1; i < 16; i++) tmax = fmaxf(tmax, s[i]);
        tmax = xhalf_max(tmax);
        const bool move = tmax > row_ref + 8.f || (row_ref == -INFINITY && tmax > -INFINITY);
        if (__any(move)) {
            const float alpha = move ? (row_ref == -INFINITY ? 0.f : fast_exp2(row_ref - tmax)) : 1.f;
            row_ref = move ? tmax : row_ref;
            row_sum *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
        }
        const float ref = row_ref == -INFINITY ? 0.f : row_ref;
        uint32_t pk[8];
        float psum0 = 0.f, psum1 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float x0 = fast_exp2(s[2 * i] - ref), x1 = fast_exp2(s[2 * i + 1] - ref);
            psum0 += x0;
            psum1 += x1;
            pk[i] = E::pack2(x0, x1);
        }
        row_sum += psum0 + psum1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ONE) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(NP) : "memory");  // this V tile is there
        // ---- O^T += V^T P^T: V^T through transposing reads, FR2 MFMAs ahead
        {
            constexpr int NG = 2 * DB, FR2 = 3;
            u32x2_t tl[NG], th[NG];
            auto tr_read = [&](int gi) {
                const int kb = gi / DB, db = gi % DB;
                const uint32_t at = (tr_off ^ ((uint32_t)(db & 3) << 6)), hi = (tr_off ^ (((uint32_t)(db & 3) << 6) | 16u));
                const uint32_t c = (uint32_t)((ONE ? 0 : st * TILE) + kb * 16 * ROW + (db >> 2) * 256);
                tl[gi] = lds_ld_tr16(at + c);
                th[gi] = lds_ld_tr16(hi + c + 4 * ROW);
            };
#pragma unroll
            for (int gi = 0; gi < FR2; gi++) tr_read(gi);
#pragma unroll
            for (int gi = 0; gi < NG; gi++) {
                if (gi + FR2 < NG) tr_read(gi + FR2);
                const int kb = gi / DB, db = gi % DB;
                const u32x4_t bop = {pk[4 * kb], pk[4 * kb + 1], pk[4 * kb + 2], pk[4 * kb + 3]};
                const u32x4_t av = {tl[gi][0], tl[gi][1], th[gi][0], th[gi][1]};
                o[db] = E::mfma(av, bop, o[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        publish();
        if constexpr (ONE) {  // ... and everybody has read this V tile (past the last tile nothing is fetched: the merge is next)
            if (jn < n_end) {
#pragma unroll
                for (int n = NP; n < 2 * NP; n++) dma_piece(n);
            }
        }
        jc = jn;
        jn = next_active(jn + 1);
    };
    while (jc < n_end) {
        one_tile(std::integral_constant<int, 0>());
        if (jc >= n_end) break;
        one_tile(std::integral_constant<int, 1>());
    }

    // ---- merge of the key groups: wave (rw, kg) finishes units kg UPW .. + UPW - 1 of its rows, the others hand theirs over
    // (no direct load may be in flight here: it would land in the sums and shares of O that the merge puts where the tiles were.  The
    // compiler does not know of loads issued in assembly, and __syncthreads() does not wait for them.  None is in flight, so the
    // wait is free.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    float total = xhalf_sum(row_sum);
    float *xs = (float *)(smem + C::OFF_SUMS) + lane;
    xs[wave * 64] = total;
    xs[(8 + wave) * 64] = row_ref;
    auto shelf = [&](int dst, int src, int j) -> f32x4_t * {  // unit j of the pass of group dst, from group src
        return (f32x4_t *)smem + (((dst * (KG - 1) + (src + KG - dst - 1) % KG) * RG + rw) * UPP + j) * 2 * 64 + lane;
    };
    auto hand_over = [&](int pass) {
#pragma unroll
        for (int dst = 0; dst < KG; dst++)
            if (dst != kg) {
#pragma unroll
                for (int j = 0; j < UPP; j++)
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const int u = dst * UPW + pass * UPP + j, e = 8 * (u & 1) + 4 * q;
                        const f32x16_t &v = o[u >> 1];
                        shelf(dst, kg, j)[q * 64] = f32x4_t{v[e], v[e + 1], v[e + 2], v[e + 3]};
                    }
            }
        __syncthreads();
    };
    hand_over(0);
    float ref[KG], top = -INFINITY, w[KG];
#pragma unroll
    for (int x = 0; x < KG; x++) {
        ref[x] = xs[(8 + x * RG + rw) * 64];
        top = fmaxf(top, ref[x]);
    }
    const float safe = top == -INFINITY ? 0.f : top;
    total = 0.f;
#pragma unroll
    for (int x = 0; x < KG; x++) {
        w[x] = fast_exp2(ref[x] - safe);
        total += xs[(x * RG + rw) * 64] * w[x];
    }
    const bool row_ok = qrow < LqS;
    const float inv = total > 0.f ? 1.f / total : 0.f;
    // this share's O in fp32 and its log2-sum-exp, which the last workgroup of the row block, or fwd_merge_kernel, adds up
    const bool share = SHARES && (p.dec_counter ? shares > 1 : p.splits > 1);
    const int64_t prow_at = (((int64_t)part * p.B + b) * p.H + h) * p.Lq + qrow;
    // (counters: [unit][share][wave][16-wide unit of O][half][lane] and [unit][share][row])
    float *o_lane = nullptr, *l_lane = nullptr;
    if (SHARES && p.dec_counter) {
        const int64_t first = (int64_t)blockIdx.x * p.splits;
        o_lane = p.o_part + first * (BM * D) + wave * (UPW * 512) + lane * 2;
        l_lane = p.lse_part + first * BM + rw * 32 + r;
    }
    uint16_t *op = (uint16_t *)p.o + b * p.o_b + (sq.q0 + qrow) * p.o_r + h * p.o_h;
#pragma unroll
    for (int pass = 0; pass < C::PASSES; pass++) {
        if (pass > 0) {
            __syncthreads();
            hand_over(pass);
        }
#pragma unroll
        for (int own = 0; own < KG; own++)
            if (own == kg) {
#pragma unroll
                for (int j = 0; j < UPP; j++) {
                    const int u = own * UPW + pass * UPP + j, c = 16 * u + 8 * g;
                    f32x4_t y[2];
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const f32x16_t &v = o[u >> 1];
#pragma unroll
                        for (int e = 0; e < 4; e++) y[q][e] = v[8 * (u & 1) + 4 * q + e] * w[own];
#pragma unroll
                        for (int x = 0; x < KG; x++)
                            if (x != own) {
                                const f32x4_t t = shelf(own, x, j)[q * 64];
#pragma unroll
                                for (int e = 0; e < 4; e++) y[q][e] += t[e] * w[x];
                            }
#pragma unroll
                        for (int e = 0; e < 4; e++) y[q][e] *= inv;
                    }
                    if (share && p.dec_counter) {
                        float *at = o_lane + part * (BM * D) + (pass * UPP + j) * 512;
                        share_store4(at, y[0]);
                        share_store4(at + 256, y[1]);
                    } else if (row_ok && c < p.d) {
                        if (share) {
                            *(f32x4_t *)(p.o_part + prow_at * p.d + c) = y[0];
                            *(f32x4_t *)(p.o_part + prow_at * p.d + c + 4) = y[1];
                        } else {
                            *(u32x4_t *)(op + c) = u32x4_t{E::pack2(y[0][0], y[0][1]), E::pack2(y[0][2], y[0][3]), E::pack2(y[1][0], y[1][1]), E::pack2(y[1][2], y[1][3])};
                        }
                    }
                }
            }
    }
    if (g == 0 && kg == 0 && row_ok) {
        // (a sum that is no number has to reach the result: only an empty share is left out)
        if (share) share_store(p.dec_counter ? l_lane + part * BM : p.lse_part + prow_at, total == 0.f ? -INFINITY : top + __builtin_amdgcn_logf(total));
        else p.lse[b * p.lse_b + h * p.lse_h + sq.q0 + qrow] = total > 0.f ? (top + __builtin_amdgcn_logf(total)) * kLn2 : INFINITY;
    }
    if constexpr (SHARES) {
        if (share && p.dec_counter && last_share(p.dec_counter + blockIdx.x, shares, (int *)(smem + C::MERGE_BYTES)) && row_ok) {
            bool on[MAX_KEY_SPLITS];
            const ShareWeights sw = lane_share_weights(l_lane, BM, shares, on);
            u32x4_t y[UPW];
            lane_merged<T, UPW>(sw, o_lane, BM * D, shares, on, y);
#pragma unroll
            for (int j = 0; j < UPW; j++) {
                const int c = 16 * (kg * UPW + j) + 8 * g;
                if (c < p.d) *(u32x4_t *)(op + c) = y[j];
            }
            if (g == 0 && kg == 0) p.lse[b * p.lse_b + h * p.lse_h + sq.q0 + qrow] = sw.lse;
        }
    }
}

template <typename T, int D, int RG, bool CAUSAL, bool CMP>
__global__ void __launch_bounds__(NT, D == 64 ? 4 : 2) fwd_wide_kernel(const FwdParams p) {
    fwd_wide<T, D, D, RG, CAUSAL, CMP, false>(p);
}
template <typename T, bool CAUSAL, bool CMP>
__global__ void __launch_bounds__(NT, 2) fwd_96_kernel(const FwdParams p) {
    fwd_wide<T, 128, 96, 2, CAUSAL, CMP, false>(p);
}
template <typename T, int D, int DC, int RG, bool CAUSAL>
__global__ void __launch_bounds__(NT, D == 64 ? 4 : 2) fwd_list_kernel(const FwdParams p) {
    fwd_wide<T, D, DC, RG, CAUSAL, true, true>(p);
}

template <typename T, int D, int RG, bool CAUSAL, bool CMP>
hipError_t launch_one(const FwdParams &p, hipStream_t stream) {
    using C = Cfg<D, RG>;
    auto kern = fwd_wide_kernel<T, D, RG, CAUSAL, CMP>;
    const bool less = D == 128 && p.d <= 96;
    if constexpr (D == 128) {
        if (less) kern = fwd_96_kernel<T, CAUSAL, CMP>;
    }
    static DynSmemLimit smem_limit[2];  // one per instantiation
    hipError_t e = smem_limit[less].ensure((const void *)kern, C::SMEM);
    if (e != hipSuccess) return e;
    FwdParams pr = p;
    const int grid = row_grid(pr, C::BM);
    hipLaunchKernelGGL(kern, dim3(grid, CMP && D <= 128 ? p.splits : 1), dim3(NT), C::SMEM, stream, pr);
    return hipGetLastError();
}

template <typename T, int D, int DC, int RG> hipError_t launch_list(const FwdParams &p, hipStream_t stream) {
    auto kern = p.causal ? fwd_list_kernel<T, D, DC, RG, true> : fwd_list_kernel<T, D, DC, RG, false>;
    static DynSmemLimit smem_limit[2];  // one per instantiation
    using C = Cfg<D, RG>;
    hipError_t e = smem_limit[p.causal != 0].ensure((const void *)kern, C::SMEM);
    if (e != hipSuccess) return e;
    FwdParams pr = p;
    const int grid = row_grid(pr, C::BM);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), C::SMEM, stream, pr);
    return hipGetLastError();
}
template <typename T> hipError_t launch_lists(const FwdParams &p, hipStream_t stream) {
    if (p.d > 128) return launch_list<T, 256, 256, 4>(p, stream);
    if (p.d > 96) return launch_list<T, 128, 128, 2>(p, stream);
    return p.d > 64 ? launch_list<T, 128, 96, 2>(p, stream) : launch_list<T, 64, 64, 2>(p, stream);
}

template <typename T, int D, int RG> hipError_t launch_t(const FwdParams &p, hipStream_t stream) {
    if (p.cmp.on) return p.causal ? launch_one<T, D, RG, true, true>(p, stream) : launch_one<T, D, RG, false, true>(p, stream);
    return p.causal ? launch_one<T, D, RG, true, false>(p, stream) : launch_one<T, D, RG, false, false>(p, stream);
}

}  // namespace

// Head dims above 128: 64-row blocks as long as all of them run at once (one to a CU), with half the chain of tiles; then 128-row ones,
// for which K and V are fetched half as often.  128 / 64 rows (us): 8192 tokens x 2 heads, 2048 kept 62.7 / 54.0; 512 rows x 16 heads
// against 2000 kept of 8000 63.8 / 54.8; 1500 x 8, all kept 62.2 / 55.2; 2 x 700 x 4 27.7 / 24.6; 1024 x 2 23.8 / 23.9; beyond a block per
// CU 3001 x 8 (376 blocks) 45.6 / 51.1, 2000 x 16 (512) 34.4 / 45.7.
hipError_t launch_fwd_wide(const FwdParams &p, int dtype, hipStream_t stream) {
    if (fwd_from_lists(p)) return dtype == 0 ? launch_lists<bf16_tag>(p, stream) : launch_lists<fp16_tag>(p, stream);
    if (p.d > 128 && fwd_blocks64(p) <= device_cus()) return dtype == 0 ? launch_t<bf16_tag, 256, 2>(p, stream) : launch_t<fp16_tag, 256, 2>(p, stream);
    if (p.d > 128) return dtype == 0 ? launch_t<bf16_tag, 256, 4>(p, stream) : launch_t<fp16_tag, 256, 4>(p, stream);
    if (p.d > 64) return dtype == 0 ? launch_t<bf16_tag, 128, 2>(p, stream) : launch_t<fp16_tag, 128, 2>(p, stream);
    return dtype == 0 ? launch_t<bf16_tag, 64, 2>(p, stream) : launch_t<fp16_tag, 64, 2>(p, stream);
}

}  // namespace fdma
