// Forward dynamic-mask attention for gfx950, column-mask specialisation.
//
// Same math and same reference counterparts as fdma_fwd.hip (compute_attn_1rowblock,
// csrc/flash_sparse_attn/src/flash_fwd_kernel.h:53-804 of the reference), for the case that dominates
// dynamic-mask attention in practice: mask and bias are absent or broadcast over the query
// dimension (shape [B, {1,Hk,H}, 1, Lk]), so "keep" is a property of the key column and the
// per-query part of the mask is only the causal triangle.
//
// What that buys:
//   * the set of KV tiles with at least one kept key is known before the main loop: the workgroup
//     scans its mask row once into an LDS bitmap and then visits active tiles only -- no per-tile
//     workgroup-wide OR, no loads and no MFMA work for skipped tiles;
//   * bias and mask fuse into one 16-element side row per key (pieces of bias*log2e, 0 / -inf for the mask and
//     for keys beyond Lk) staged in LDS, which the score MFMAs contract as one more k-step;
//   * causal masking costs instructions on diagonal tiles only.
//
// The matrix pipe is what the kernel is priced against, so the vector ALU gets as little as possible and what is
// left runs UNDER the MFMAs.
//   Softmax on the matrix pipe.  Q is scaled by softmax_scale*log2(e) once, and every key carries a 16-element
// side row in LDS that is contracted as one more 16-wide k-step of the score MFMAs against constants held per
// query row: three 16-bit pieces of bias*log2(e) (together the exact fp32 value) times 1, the mask (0 / -inf) times
// 1, and two ones that meet the two 16-bit pieces of MINUS the row's softmax reference point.  The accumulators
// start from the constant 0, and what leaves the MFMAs is the finished exp2 argument.  The reference point of a
// row is any number near its running maximum (the softmax does not depend on it); it is set by the first tile and
// then left alone as long as no probability exceeds 2^14 -- which the sum of the probabilities shows, so the
// common path has no maximum at all: exp2, convert to 16 bits (two per instruction), one addition to the row sum
// (plain fp32 additions: a 16-bit dot product with (1, 1) would halve their number, but it runs on the matrix pipe's
// side of the SIMD and cost 2-3 % of the kernel): 2.5 vector instructions per score.  A half tile that fails the check (or a wave whose rows have no
// reference yet) takes the classic path: maximum, new reference, rescale of O and of the sums.
//   Software pipeline over HALF tiles (32 keys).  One step issues the score MFMAs of half tile h+1, the P V MFMAs
// of half tile h-1 and, between them, the softmax instructions of half tile h: the three have no dependence on one
// another, so the vector instructions issue while the matrix pipe works, and the two waves of a SIMD no longer
// have to be in different phases for anything to overlap (phase by phase -- scores, softmax, P V -- the same loop
// ran at 49 % of the MFMA rate, the pipelined one is bound by LDS fragment reads and exp2 at 75-80 %).  A half tile
// in flight costs 16 score and 8 probability registers, two of them 48 -- what one whole tile cost before.
//   Staging.  K, V^T (V is transposed in registers while being staged) and the side rows are double-buffered in LDS;
// K runs one tile ahead of V (the P V product of a tile is issued a tile after its scores).  With 8 waves (256 query
// rows per workgroup) four waves stage V and four K and the side rows; one barrier per tile.  Global loads are one
// instruction each (scalar tile base + a loop-invariant per-thread offset) and sit a whole tile in front of their
// LDS stores.  Workgroup ids are remapped so that the workgroups sharing one XCD's L2 also share K / V.
//   Key groups (KG = 2).  A grid of no more 128-row workgroups than CUs leaves a CU with one wave per SIMD, which does not
// overlap its vector work, its LDS reads and its barriers with its MFMAs (1.4 us per tile of 0.5 us matrix work).  Then a
// workgroup is two groups of four waves over the SAME query rows, each with its own stages: they take the active tiles in
// turn, with a softmax of their own, and are merged through LDS at the end.  512 rows x 32 heads against 2048 kept keys,
// d = 128: 44 us with one group, 37.8 with two (and 31 in fdma_fwd_wide.hip, which takes that size).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_fwd_merge.h"

namespace fdma {

namespace {

constexpr int MAX_TILES = 16384;  // bitmap capacity: Lk <= 1 Mi keys

template <int D, int BN> struct CmSmem {
    static constexpr int SK = D + 8;        // K tile row stride (elements)
    static constexpr int SVT = BN + 8;      // V^T tile row stride (elements)
    static constexpr int K_BYTES = BN * SK * 2;
    static constexpr int VT_BYTES = D * SVT * 2;
    static constexpr int OFF_K = 0;
    static constexpr int OFF_VT = OFF_K + 2 * K_BYTES;
    static constexpr int X_BYTES = BN * 32;  // side rows: 16 elements of 16 bits per key
    static constexpr int OFF_X = OFF_VT + 2 * VT_BYTES;
    static constexpr int OFF_BITS = OFF_X + 2 * X_BYTES;
    static constexpr int OFF_FLAG = OFF_BITS + MAX_TILES / 8;  // one word: a wave left the range of the common path
    static constexpr int TOTAL = OFF_FLAG + 16;
};

// CMP: K / V are the compacted copies of the kept columns (see fdma_compact.hip).  The key axis then has
// `count` columns, all kept; the fused bias vector comes pre-gathered, and the causal limit of a query row
// is the number of kept columns at or below its diagonal instead of the column index itself.
// DC: the head dims that are worked on, 96 of a 128-wide tile for head dims 65 to 96 (here and in fdma_fwd_wide.hip): a quarter of the products
// less, the staging as it is.  d = 96, 128 dims / 96 of them, us: 4 x 13120 x 8/4 heads, 3606 kept 390 / 335; 22912 x 16/16, 1280 kept, not
// causal 235 / 204; ragged 4026 and others x 16/8 95.4 / 82.5; key groups 2 x 128 x 16/8 against 861 kept of 1817 24.2 / 22.7, 4 x 1152 x
// 16/8, 128 kept 22.7 / 21.8.
template <typename T, int D, int DC, int BN, bool CAUSAL, int NW, bool CMP, int KG>
__global__ void __launch_bounds__(64 * NW * KG, (NW == 4 && KG == 1) ? 2 : 1) fwd_colmask_kernel(const FwdParams p) {
    constexpr int NTHREADS = 64 * NW;         // of a key group
    static_assert(KG == 1 || NW == 4, "key groups are for small grids, which have 128-row workgroups");
    constexpr int STHREADS = 256;             // threads staging one operand
    constexpr bool SPLIT = NW == 8;           // 8 waves: the first four stage V, the last four K and the side rows
    static_assert(NW == 4 || NW == 8, "staging maps are written for 256 or 512 threads");
    static_assert(BN == 64, "the pipeline works on the two 32-key halves of a 64-key tile");
    using E = Elem<T>;
    using SM = CmSmem<D, BN>;
    constexpr int KQ = BN / 4;                // key quads per tile
    constexpr int KS = DC / 16;
    constexpr int DB = DC / 32;
    constexpr int BM = 32 * NW;
    constexpr int CH = D / 8;                 // 16-byte chunks per K row
    constexpr int K_RPP = STHREADS / CH;      // K rows staged per pass
    constexpr int K_IT = BN / K_RPP;          // passes (registers) per K tile
    constexpr int V_ITEMS = KQ * CH;          // (key quad, d chunk) items of a V tile
    constexpr int NL = SPLIT ? 4 : K_IT + 4;  // 16-byte loads per thread and tile
    constexpr int VB = SPLIT ? 0 : K_IT;      // first V staging register
    static_assert(V_ITEMS <= STHREADS, "one V item per thread");
    static_assert(!SPLIT || K_IT == 4, "the role split assumes four loads per thread for either operand");

    extern __shared__ __attribute__((aligned(16))) char smem_all[];
    const int kgrp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NTHREADS);  // key group of this wave
    // This group's LDS.  A lone group at d = 128 addresses the array itself: through the pointer variable the same places took 4
    // more registers, which the eight-wave kernels do not have (20 bytes spilled; ragged forward of 11 265 tokens x 32 heads
    // 370.0 -> 367.1 us, of 3 518 x 16 56.0 -> 55.2).  Elsewhere the pointer is ahead by as much (ragged, 18 000 tokens x 16,
    // d = 64: 127.3 and 128.9).
    char *const smem_grp = smem_all + kgrp * SM::TOTAL;
#define FWD_LDS (KG == 1 && D == 128 ? smem_all : smem_grp)
    uint32_t *sBits = (uint32_t *)(FWD_LDS + SM::OFF_BITS);
    uint32_t *sFlag = (uint32_t *)(smem_all + SM::OFF_FLAG);  // (one for all: the groups leave the common path together)

    const int tid = (int)threadIdx.x - kgrp * NTHREADS;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (tells the compiler that it is wave-uniform)
    const int lane = tid & 63;
    const int r = lane & 31;
    const int g = lane >> 5;

    // Workgroup -> (batch, kv head, query head, query block), XCD-aware.  Workgroups are dealt to the 8
    // XCDs round-robin by linear id and every XCD has its own L2.  The id is remapped (row_unit) so that the
    // workgroups running at the same time on one XCD share K / V: an XCD walks its lists of query blocks one after the
    // other, heaviest block first, the G query heads of a block side by side.  Re-reads of K / V
    // tiles then hit in that XCD's L2, and every XCD gets the same amount of work.
    const RowUnit ru = row_unit(p, blockIdx.x, BM);
    if (ru.block < 0) return;
    const int b = ru.b, hk = ru.hk, h = ru.h;
    const int m0 = ru.block * BM;
    const SeqInfo sq = seq_info(p, b);  // this batch entry's lengths and first rows (ragged batch: from cu_seqlens)
    const int LqS = sq.Lq, LkS = sq.Lk;
    const int shift = LkS - LqS;
    const int wrow0 = m0 + wave * 32;  // first query row of this wave

    // ---- Q fragments: the loads are issued first of all (they depend on the workgroup's coordinates only), the
    // values are looked at -- scaled -- after the set-up below, whose own memory traffic they overlap with
    u32x4_t qf[KS];
    {
        const int qrow = wrow0 + r;
        const int qc = qrow < LqS ? qrow : LqS - 1;
        const uint16_t *qp = (const uint16_t *)p.q + b * p.q_b + (sq.q0 + qc) * p.q_r + h * p.q_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            qf[ks] = *(const u32x4_t *)(qp + (c < p.d ? c : 0));  // (chunks beyond d are cleared when scaled)
        }
    }

    const int hm = p.mask ? (p.Hm == p.H ? h : (p.Hm == 1 ? 0 : hk)) : 0;
    const int hb = p.bias ? (p.Hb == p.H ? h : (p.Hb == 1 ? 0 : hk)) : 0;
    const uint8_t *mrow = p.mask ? p.mask + b * p.m_b + hm * p.m_h : nullptr;
    const uint16_t *brow = p.bias ? (const uint16_t *)p.bias + b * p.bi_b + hb * p.bi_h : nullptr;
    const uint16_t *kbase = (const uint16_t *)p.k + b * p.k_b + sq.k0 * p.k_r + hk * p.k_h;
    const uint16_t *vbase = (const uint16_t *)p.v + b * p.v_b + sq.k0 * p.v_r + hk * p.v_h;

    // key columns this workgroup iterates over, and the number of them a query row may see
    const int Lk = CMP ? p.cmp.count[b * p.Hk + hk] : LkS;
    const int32_t *ccnt = CMP ? p.cmp.cnt + (int64_t)(b * p.Hk + hk) * p.cmp.ld : nullptr;
    const float *fbrow = CMP ? p.cmp.fb + (int64_t)(b * p.cmp.Hfb + (p.cmp.Hfb == p.H ? h : hk)) * p.cmp.ld : nullptr;
    // causal limits: columns below vis_lane are visible to this lane's query row, and a half tile that ends at
    // or below vis_wave (the limit of the wave's first row) needs no masking at all
    const int vis_lane = CAUSAL ? visible_columns<CMP>(wrow0 + r, LqS, LkS, ccnt) : 0;
    const int vis_wave = CAUSAL ? visible_columns<CMP>(wrow0, LqS, LkS, ccnt) : 0;
    const int vis_block = CAUSAL ? visible_columns<CMP>(m0 + BM - 1, LqS, LkS, ccnt) : 0;

    int n_end = (Lk + BN - 1) / BN;
    if (CAUSAL) {
        const int ne = ((vis_block < 0 ? 0 : vis_block) + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }

    // ---- active-tile bitmap
    for (int base = 0; !CMP && base < n_end; base += NTHREADS) {
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
        if (lane == 0) {
            const int w0 = (base + wave * 64) >> 5;
            sBits[w0] = (uint32_t)ball;
            sBits[w0 + 1] = (uint32_t)(ball >> 32);
        }
    }
    // The upper halves of the side rows (both stages) are zero for good; the staging writes the lower halves.  V^T
    // stage 1 is cleared as well: the first pipeline step multiplies it with zero probabilities (there is no half tile
    // in front of the first one), and what an earlier workgroup left there need not be a number.  (All of it is made
    // visible by the barrier in front of the main loop.)
    if (tid < 2 * BN) *(u32x4_t *)(FWD_LDS + SM::OFF_X + tid * 32 + 16) = u32x4_t{0, 0, 0, 0};
    for (int i = tid; i < SM::VT_BYTES / 16; i += NTHREADS)
        *(u32x4_t *)(FWD_LDS + SM::OFF_VT + SM::VT_BYTES + i * 16) = u32x4_t{0, 0, 0, 0};
    if (!CMP) __syncthreads();  // (compacted keys have no bitmap: every tile up to n_end is active)

    // Iterator over the active tiles in ascending order (n_end once they are exhausted).  The current bitmap word
    // lives in a scalar register and loses a bit per call; LDS is read again only when a word runs out (readfirstlane
    // tells the compiler that the value is wave-uniform, so tile numbers, loop conditions and load addresses stay in
    // scalar registers).  Compacted keys have no bitmap: every tile up to n_end is active.
    uint32_t it_word = 0;
    int it_base = -32, it_next = 0;
    auto next_tile = [&]() -> int {
        if (CMP) {
            const int j = it_next < n_end ? it_next : n_end;
            it_next = j + 1;
            return j;
        }
        while (it_word == 0) {
            it_base += 32;
            if (it_base >= n_end) {
                it_base = n_end;  // (stays exhausted)
                return n_end;
            }
            it_word = __builtin_amdgcn_readfirstlane(sBits[it_base >> 5]);
        }
        const int j = it_base + __builtin_ctz(it_word);
        it_word &= it_word - 1;
        return j < n_end ? j : n_end;
    };
    // The tiles in turns of KG: `lead` is the first of a turn (what ends the loops, alike for all groups), `mine` this
    // group's -- n_end when the last turn has none left for it: its keys then count as masked, and the tile that is fetched
    // in its place (any existing one) is not looked at.
    struct Turn { int lead, mine; };
    auto next_turn = [&]() -> Turn {
        Turn t;
        t.lead = t.mine = next_tile();
        if (KG == 2) {
            const int second = next_tile();
            if (kgrp == 1) t.mine = second;
        }
        return t;
    };

    f32x16_t o[DB];
    float row_sum = 0.f;
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;

    // ---- staging (global -> registers -> LDS).  A tile is BN * CH 16-byte chunks of K plus V_ITEMS (key quad, d chunk)
    // items of V with four loads each (V is transposed in registers on its way to LDS).  Every load is unconditional,
    // from an always valid address: rows beyond the end of the keys are clamped to the last row (their side row says
    // -inf, so the duplicate never counts) and head-dim chunks beyond d to chunk 0 (they meet zero Q fragments /
    // columns of O that are not stored).  The per-thread byte offsets are loop invariants -- one set for full tiles,
    // one for the (only) partial tile at the end of the keys -- so a load is one instruction with a scalar tile base.
    const bool role_v = !SPLIT || wave < 4, role_k = !SPLIT || wave >= 4;  // wave-uniform
    const bool role_x = wave == 0;  // the side rows of a tile: lane l of wave 0 makes the row of key l
    const int kt = tid & (STHREADS - 1);
    const int kc = kt % CH, kr0 = kt / CH;
    const int vkg = kt % KQ, vc = (kt / KQ) % CH;  // V: key quad and d chunk of this thread
    const uint32_t k_r2 = (uint32_t)(p.k_r * 2), v_r2 = (uint32_t)(p.v_r * 2);  // bytes per row
    const uint32_t kcolb = (kc * 8 < p.d ? kc * 16 : 0);
    const int j_last = Lk > 0 ? (Lk - 1) / BN : 0, last_row = Lk > 0 ? (Lk - 1) % BN : 0;
    uint32_t soff[NL], soff_l[NL];  // byte offsets of this thread's loads inside a full / the last tile
#pragma unroll
    for (int n = 0; n < NL; n++) {
        const bool is_v = SPLIT ? role_v : n >= K_IT;
        const int item = SPLIT ? n : (n >= K_IT ? n - K_IT : n);  // V: four loads (keys of the quad) per item
        const int row = is_v ? 4 * vkg + (item & 3) : kr0 + item * K_RPP;
        const uint32_t vcolb = (vc * 8 < p.d ? vc * 16 : 0);
        const uint32_t r2 = is_v ? v_r2 : k_r2, colb = is_v ? vcolb : kcolb;
        soff[n] = (uint32_t)row * r2 + colb;
        soff_l[n] = (uint32_t)(row < last_row ? row : last_row) * r2 + colb;
    }
    u32x4_t sreg[NL];             // staging registers
    uint32_t braw = 0, mraw = 0;  // raw bias / mask of this thread's column of the tile whose side rows are in flight
    // an absent mask / bias is the first element of K instead (its rows may lie on each other: nothing behind them is K's) and ignored
    // when the value is used
    const uint8_t *mrow_ld = mrow ? mrow : (const uint8_t *)kbase;
    const uint16_t *brow_ld = brow ? brow : kbase;
    bool bcol_ok = false;
    gptr_t tb_k = nullptr, tb_v = nullptr;        // tile bases (wave-uniform, in scalar registers)
    bool last_k = false, last_v = false;          // the K / V tile in flight is the partial one

    // next fetches: K and the side-row inputs of tile jk / V of tile jv (with split roles a wave has one of the two)
    auto set_tile_k = [&](Turn tk) {
        if (!role_k) return;
        const int jk = KG == 1 || tk.mine < n_end ? tk.mine : tk.lead;
        tb_k = uniform_ptr((const char *)kbase + (int64_t)jk * BN * p.k_r * 2);
        last_k = jk == j_last;
    };
    // side-row inputs of this thread's column of tile jx: only the raw loads here -- the values are looked at when
    // the row is stored
    auto set_tile_x = [&](Turn tx) {
        if (!role_x) return;
        const int col = tx.mine * BN + lane;
        bcol_ok = col < Lk && (KG == 1 || tx.mine < n_end);
        const int cc = bcol_ok ? col : 0;
        // (unconditional loads: a load in one arm of a select would have to be waited for right here)
        if (CMP) {
            braw = __float_as_uint(fbrow[cc]);
        } else {
            mraw = mrow_ld[mrow ? cc : 0];
            braw = brow_ld[brow ? cc : 0];
        }
    };
    auto set_tile_v = [&](Turn tv) {
        if (!role_v) return;
        const int jv = KG == 1 || tv.mine < n_end ? tv.mine : tv.lead;
        tb_v = uniform_ptr((const char *)vbase + (int64_t)jv * BN * p.v_r * 2);
        last_v = jv == j_last;
    };
    // the loads of this thread's K registers / V registers (with split roles: all NL registers, in the waves of that role)
    auto load_regs = [&](bool v) {
        if (SPLIT ? (v ? !role_v : !role_k) : false) return;
        const gptr_t base = v ? tb_v : tb_k;
        const bool last = v ? last_v : last_k;
        const int n0 = SPLIT ? 0 : (v ? K_IT : 0), n1 = SPLIT ? NL : (v ? NL : K_IT);
#pragma unroll
        for (int n = n0; n < n1; n++)
            sreg[n] = *(const __attribute__((address_space(1))) u32x4_t *)(base + (last ? soff_l[n] : soff[n]));
    };
    // registers -> LDS: K into stage kbuf, the side rows into stage xbuf, V^T into stage vbuf
    auto store_k = [&](int kbuf) {
        if (role_k) {
            char *sK = FWD_LDS + SM::OFF_K + kbuf * SM::K_BYTES;
#pragma unroll
            for (int it = 0; it < K_IT; it++)
                *(u32x4_t *)(sK + ((kr0 + it * K_RPP) * SM::SK + kc * 8) * 2) = sreg[it];
        }
    };
    auto store_x = [&](int xbuf) {
        if (role_x) {  // side row of this lane's key: pieces of bias * log2e, the mask term, the two ones
            float v = 0.f;
            bool keep = bcol_ok;
            if (CMP) {
                v = __uint_as_float(braw);
            } else {
                keep = keep && (!mrow || mraw);
                if (brow) v = E::lo(braw) * kLog2e;
            }
            const u32x2_t pc = split3<T>(keep ? v : 0.f);
            u32x4_t row;
            row[0] = pc[0];
            row[1] = pc[1] | (E::pack2(0.f, keep ? 0.f : -INFINITY) & 0xffff0000u);
            row[2] = E::pack2(E::kRefWeight, 1.f);
            row[3] = 0;
            *(u32x4_t *)(FWD_LDS + SM::OFF_X + xbuf * SM::X_BYTES + lane * 32) = row;
        }
    };
    auto store_v = [&](int vbuf) {
        if (role_v && kt < V_ITEMS) {  // transpose 4 keys x 8 d in registers, write V^T[d][key quad]
            char *sVt = FWD_LDS + SM::OFF_VT + vbuf * SM::VT_BYTES;
#pragma unroll
            for (int dd = 0; dd < 8; dd++) {
                const int w = dd >> 1;
                const uint32_t sel = (dd & 1) ? 0x07060302u : 0x05040100u;
                u32x2_t out;
                out[0] = __builtin_amdgcn_perm(sreg[VB + 1][w], sreg[VB][w], sel);
                out[1] = __builtin_amdgcn_perm(sreg[VB + 3][w], sreg[VB + 2][w], sel);
                *(u32x2_t *)(sVt + ((vc * 8 + dd) * SM::SVT + 4 * vkg) * 2) = out;
            }
        }
    };

    const int a_row = pi_row(r);

    // Constants of a query row that meet the side rows of the keys (B operand of the extra k-step; the lanes of
    // the upper half supply zeros against the zero half of the side rows): 1 / kPieceScale for the three bias
    // pieces, 1 for the mask term, and the two pieces of minus the row's reference point.
    const float side_mult = 1.f / E::kPieceScale;
    u32x4_t qx;
    qx[0] = g == 0 ? E::pack2(side_mult, side_mult) : 0u;
    qx[1] = g == 0 ? E::pack2(side_mult, 1.f) : 0u;
    qx[2] = 0u;
    qx[3] = 0u;
    // Softmax state of a row: O and row_sum are relative to exp2(row_ref); enc_ref is what the pieces in qx stand
    // for, i.e. what the score MFMAs subtract.  row_ref = -inf: no visible key met yet (enc_ref is 0 then).  On the
    // common path row_ref == enc_ref for every row of the wave (`fast`, wave-uniform).
    float row_ref = -INFINITY, enc_ref = 0.f;
    bool fast = false;

    // Fragment addresses of a half tile.  Scores: side rows + KS k-steps of K for the 32 keys of half `kh` of stage
    // `kbuf`; P V: the two 16-key k-steps of half `vh` of V^T stage `vbuf`, DB row blocks each.
    constexpr int NQK = KS + 1, NPV = 2 * DB, NF = NQK + NPV;
    constexpr int FR = 4;  // fragment reads run FR MFMAs ahead of their MFMAs (8 ahead: 19 spilled registers)
    auto frag_ptr = [&](int f, int kbuf, int kh, int vbuf, int vh) -> const u32x4_t * {
        if (f == 0) return (const u32x4_t *)(FWD_LDS + SM::OFF_X + kbuf * SM::X_BYTES + (32 * kh + a_row) * 32 + g * 16);
        if (f < NQK)
            return (const u32x4_t *)(FWD_LDS + SM::OFF_K + kbuf * SM::K_BYTES + ((32 * kh + a_row) * SM::SK + (f - 1) * 16 + g * 8) * 2);
        const int kb = (f - NQK) / DB, db = (f - NQK) % DB;
        return (const u32x4_t *)(FWD_LDS + SM::OFF_VT + vbuf * SM::VT_BYTES + ((32 * db + a_row) * SM::SVT + 32 * vh + 16 * kb + 8 * g) * 2);
    };
    const f32x16_t zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    // causal masking of a half tile whose first column is col0 (register i <-> column 16 (i / 8) + 8 g + i % 8)
    auto causal_mask = [&](f32x16_t &s, int col0) {
        const int lim = vis_lane - 1 - col0 - 8 * g;  // local column limit for this lane
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int lc = 16 * (i >> 3) + (i & 7);
            s[i] = lc <= lim ? s[i] : -INFINITY;
        }
    };

    // Classic softmax of one half tile (the safe path, and the first tile of the common path's set-up): maximum, a new
    // reference point where the row has none yet or a score exceeds the old one by more than 2^8 (then O and the sums are
    // rescaled, and the pieces in qx replaced), probabilities.  The scores in `s` are relative to enc_ref as it is on entry.
    auto classic = [&](f32x16_t &s, uint32_t (&pk)[8], int col0) {
        if (CAUSAL && col0 + 32 > vis_wave) causal_mask(s, col0);
        float tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, s[i]);
        tmax = xhalf_max(tmax);
        const bool unset = row_ref == -INFINITY;
        const float cand = enc_ref + tmax;  // the half tile's maximum as an absolute score
        const bool move = unset ? tmax > -INFINITY : cand > row_ref + 8.f;
        float shift_s = unset ? 0.f : enc_ref - row_ref;  // probabilities are exp2(s + shift_s)
        if (__any(move)) {
            float enc;
            const uint32_t w = encode_ref<T>(cand, enc);
            // the reference becomes exactly what the pieces stand for, unless they cannot express it (fp16,
            // scores beyond 4e6): then the remainder stays in shift_s
            const float new_ref = move ? (fabsf(enc - cand) <= 0.5f ? enc : cand) : row_ref;
            const float alpha = (move && !unset) ? fast_exp2(row_ref - new_ref) : 1.f;
            row_sum *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
            if (move) {
                shift_s = enc_ref - new_ref;
                enc_ref = enc;
                if (g == 0) qx[2] = w;
            }
            row_ref = new_ref;
        }
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const uint32_t w = E::pack2(fast_exp2(s[i] + shift_s), fast_exp2(s[i + 1] + shift_s));
            psum = E::add_pair(w, psum);
            pk[i / 2] = w;
        }
        row_sum += psum;
    };
    // scores of half kh of K stage kbuf / P V of half vh of V^T stage vbuf, on their own (set-up, tail, safe path)
    auto scores_half = [&](f32x16_t &s, int kbuf, int kh) {
        u32x4_t a[NQK];
#pragma unroll
        for (int f = 0; f < NQK; f++) a[f] = *frag_ptr(f, kbuf, kh, 0, 0);
        s = E::mfma(a[0], qx, zero16);
#pragma unroll
        for (int f = 1; f < NQK; f++) s = E::mfma(a[f], qf[f - 1], s);
    };
    auto pv_half = [&](const uint32_t (&pk)[8], int vbuf, int vh) {
        u32x4_t a[NPV];
#pragma unroll
        for (int f = 0; f < NPV; f++) a[f] = *frag_ptr(NQK + f, 0, 0, vbuf, vh);
#pragma unroll
        for (int f = 0; f < NPV; f++) {
            const int kb = f / DB, db = f % DB;
            const u32x4_t bop = {pk[4 * kb], pk[4 * kb + 1], pk[4 * kb + 2], pk[4 * kb + 3]};
            o[db] = E::mfma(a[f], bop, o[db]);
        }
    };

    // One step of the pipeline.  MFMAs: scores of the NEXT half tile (half kh of K stage kbuf) into `snext`, and
    // O^T += V^T P^T of the PREVIOUS half tile (probabilities pprev, half vh of V^T stage vbuf).  Vector ALU, between
    // them: softmax of the CURRENT half tile `scur` (first column col0) into `pcur` -- the common path, no maximum.
    // A step also moves one staged operand from the registers to LDS, piece by piece between its MFMAs, and issues that
    // operand's next loads behind them: V (and, in wave 0, the side rows) in the first step of a tile (STAGE), K in the
    // second.  With split roles the two waves of a SIMD have different roles.  (Staging as a phase of its own, after or
    // in front of the MFMAs, left the matrix pipe to the SIMD's other wave alone for a fifth of every tile.  Half tiles
    // on the causal diagonal are masked before the step, in code of their own: only they pay for it.)
    auto step = [&](auto stage_c, auto do_v_c, auto do_k_c, f32x16_t &scur, f32x16_t &snext, uint32_t (&pcur)[8],
                    const uint32_t (&pprev)[8], int kbuf, int kh, int vbuf, int vh, Turn j_next, Turn jx_next) {
        constexpr bool STAGE = decltype(stage_c)::value;
        constexpr bool DO_V = STAGE && decltype(do_v_c)::value, DO_K = !STAGE && decltype(do_k_c)::value;
        char *const sVt_w = FWD_LDS + SM::OFF_VT + (vbuf ^ 1) * SM::VT_BYTES;  // V(t) goes to the stage the P V product has left
        char *const sK_w = FWD_LDS + SM::OFF_K + (kbuf ^ 1) * SM::K_BYTES;     // K(t+2) to the stage whose scores are finished
        // Order of issue: a wave issues in program order, so the vector instructions have to sit BETWEEN the MFMAs to run
        // under them.  The step is written slot by slot -- one MFMA, the fragment read of the MFMA FR slots later, an even
        // share of the softmax (the two exp2 of a pair of scores in one slot, their conversion to 16 bits and their
        // addition to the row sum in the next, a piece of the staging) -- with a scheduling barrier after every slot.
        // The probabilities are relative to the reference the MFMAs have already subtracted; the row sum adds the
        // fp32 values, as the reference does (src/softmax.h: the sum is taken before the conversion to 16 bits).
        if (DO_K) set_tile_k(j_next);  // base of the tile whose pieces are requested between the MFMAs below
        u32x4_t a[NF];
#pragma unroll
        for (int f = 0; f < FR; f++) a[f] = *frag_ptr(f, kbuf, kh, vbuf, vh);
        float psum0 = 0.f, psum1 = 0.f, x0[8], x1[8];
#pragma unroll
        for (int f = 0; f < NF; f++) {
            if (f + FR < NF) a[f + FR] = *frag_ptr(f + FR, kbuf, kh, vbuf, vh);
            if (f == 0) {
                snext = E::mfma(a[f], qx, zero16);
            } else if (f < NQK) {
                snext = E::mfma(a[f], qf[f - 1], snext);
            } else {
                const int kb = (f - NQK) / DB, db = (f - NQK) % DB;
                const u32x4_t bop = {pprev[4 * kb], pprev[4 * kb + 1], pprev[4 * kb + 2], pprev[4 * kb + 3]};
                o[db] = E::mfma(a[f], bop, o[db]);
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int slot = k * (NF - 1) / 8;  // the pair's exp2 slot; its conversion follows one slot later
                if (slot == f) {
                    x0[k] = fast_exp2(scur[2 * k]);
                    x1[k] = fast_exp2(scur[2 * k + 1]);
                }
                if (slot + 1 == f) {
                    pcur[k] = E::pack2(x0[k], x1[k]);
                    psum0 += x0[k];
                    psum1 += x1[k];
                }
            }
            // staging, a piece per slot: one transposed row pair of V (two permutes, one 8-byte store) / one 16-byte
            // chunk of K
            if (DO_V) {
#pragma unroll
                for (int dd = 0; dd < 8; dd++)
                    if (f == 1 + dd * ((NF - 1) / 8)) {
                        const int w = dd >> 1;
                        const uint32_t sel = (dd & 1) ? 0x07060302u : 0x05040100u;
                        u32x2_t out;
                        out[0] = __builtin_amdgcn_perm(sreg[VB + 1][w], sreg[VB][w], sel);
                        out[1] = __builtin_amdgcn_perm(sreg[VB + 3][w], sreg[VB + 2][w], sel);
                        *(u32x2_t *)(sVt_w + ((vc * 8 + dd) * SM::SVT + 4 * vkg) * 2) = out;
                    }
            }
            if (DO_K) {
                // (a register goes back to fetching -- the same piece of K(j_next) -- as soon as it is stored: a whole
                // tile then lies between every load and its store; all four loads behind the last MFMA had half a tile)
#pragma unroll
                for (int it = 0; it < K_IT; it++)
                    if (f == 1 + it * ((NF - 1) / K_IT)) {
                        *(u32x4_t *)(sK_w + ((kr0 + it * K_RPP) * SM::SK + kc * 8) * 2) = sreg[it];
                        sreg[it] = *(const __attribute__((address_space(1))) u32x4_t *)(tb_k + (last_k ? soff_l[it] : soff[it]));
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const float psum = psum0 + psum1;
        row_sum += psum;
        // (the results are pinned here: left alone, the compiler sinks the softmax below the staging code that follows,
        // away from the MFMAs it is meant to run under)
#pragma unroll
        for (int i = 0; i < 8; i++) asm volatile("" : "+v"(pcur[i]));
        asm volatile("" : "+v"(row_sum));
        __builtin_amdgcn_sched_barrier(0);
        if (STAGE) {  // the loads of V(j_next); side rows of the next tile, inputs of those of the tile after it
            store_x(kbuf ^ 1);  // (in front of the new loads: its inputs must not be waited for together with them)
            if (DO_V) {
                set_tile_v(j_next);
                load_regs(true);
            }
            set_tile_x(jx_next);
        }
        if (__any(!(psum <= 16384.f))) *sFlag = 1u;
    };

    const Turn j0 = next_turn();
    bool redo = false;
    if (j0.lead < n_end) {
        // ---- common path.  Set-up: the first tile is staged, its scores are computed once just for their row maxima,
        // and the reference point of every row is put kRefMargin above its maximum: probabilities start around
        // 2^-margin, and the rest of the row may exceed the first tile by margin + 14 before the check fails.
        Turn jc = j0, jn1 = next_turn(), jn2 = next_turn(), jn3 = next_turn();
        auto or_else = [&](Turn t, Turn e) -> Turn { return t.lead < n_end ? t : e; };
        if (threadIdx.x == 0) *sFlag = 0u;
        // K(0), K(1) and the side rows of tile 0 go to LDS; the registers then fetch K(2), V(0) (kept until step A)
        // and the side-row inputs of tile 1
        set_tile_k(j0);
        set_tile_v(j0);
        set_tile_x(j0);
        load_regs(false);
        load_regs(true);
        u32x4_t k1[K_IT];  // K(1) travels in registers of its own, together with K(0)
        set_tile_k(or_else(jn1, j0));
        if (role_k) {
#pragma unroll
            for (int it = 0; it < K_IT; it++)
                k1[it] = *(const __attribute__((address_space(1))) u32x4_t *)(tb_k + (last_k ? soff_l[it] : soff[it]));
        }
        store_k(0);
        store_x(0);
        set_tile_x(or_else(jn1, j0));
        if (role_k) {
#pragma unroll
            for (int it = 0; it < K_IT; it++) sreg[it] = k1[it];
        }
        store_k(1);
        set_tile_k(or_else(jn2, j0));
        load_regs(false);
        // Q is scaled by softmax_scale * log2(e) once, here (the reference also rounds the scaled Q to the input type,
        // flash_fwd_kernel.h:428-439): the MFMAs then produce exp2-domain scores directly
        {
            const bool row_ok = wrow0 + r < LqS;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) qf[ks] = scaled8<T>(qf[ks], p.scale_log2, row_ok && ks * 16 + g * 8 < p.d);
        }
        __syncthreads();

        f32x16_t sA, sB;
        uint32_t pA[8], pB[8];
        {
            scores_half(sA, 0, 0);
            scores_half(sB, 0, 1);
            const int col0 = j0.mine * BN;
            if (CAUSAL && col0 + 32 > vis_wave) causal_mask(sA, col0);
            if (CAUSAL && col0 + 64 > vis_wave) causal_mask(sB, col0 + 32);
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, fmaxf(sA[i], sB[i]));
            tmax = xhalf_max(tmax);
            bool bad = false;
            if (tmax > -INFINITY) {  // (a row that sees nothing in the first tile sees nothing at all)
                const float want = tmax + (std::is_same<T, bf16_tag>::value ? 8.f : 4.f);
                float enc;
                const uint32_t w = encode_ref<T>(want, enc);
                bad = !(fabsf(enc - want) <= 0.5f);  // the pieces cannot express it: safe path
                enc_ref = row_ref = enc;
                if (g == 0) qx[2] = w;
            }
            if (__any(bad)) *sFlag = 1u;
            scores_half(sA, 0, 0);  // again, against the reference
        }
#pragma unroll
        for (int i = 0; i < 8; i++) pB[i] = 0u;

        // ---- main loop.  Iteration t works on active tile t (halves 2t and 2t+1 go through the softmax).  On entry K(t)
        // and K(t+1) are in the two K stages (K(t) in stage t & 1), the side rows of tile t in stage t & 1 and V(t-1) in
        // V^T stage (t-1) & 1; the registers hold K(t+2), V(t) and the side-row inputs of tile t+1; sA holds the scores of
        // half 2t, pB the probabilities of half 2t-1.
        //   step A: scores of half 2t+1 (K(t), second half), softmax of half 2t, P V of half 2t-1 (V(t-1), second half);
        //           then V(t) -> V^T stage t & 1 and the loads of V(t+1); side rows of tile t+1 -> stage (t+1) & 1,
        //           inputs of those of tile t+2
        //   barrier
        //   step B: K(t+2) -> K stage t & 1 and the loads of K(t+3); then scores of half 2t+2 (K(t+1), first half),
        //           softmax of half 2t+1, P V of half 2t (V(t), first half)
        // A stage is written after the barrier that follows its last read, and read after the barrier that follows its
        // write.  Past the last tile an existing tile is fetched and stored again and what is computed from it is dropped.
        const std::true_type yes;
        const std::false_type no;
        int t = 0;
        // (the loop exists once per staging role, so that the staging pieces inside the steps are unconditional code)
        auto tile_loop = [&](auto do_v_c, auto do_k_c) {
            while (true) {
                const int kb = t & 1;
                const int col0 = jc.mine * BN;
                if (CAUSAL && col0 + 32 > vis_wave) causal_mask(sA, col0);
                __builtin_amdgcn_sched_barrier(0);
                step(yes, do_v_c, do_k_c, sA, sB, pA, pB, kb, 1, kb ^ 1, 1, or_else(jn1, jc), or_else(jn2, jc));
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
                if (CAUSAL && col0 + 64 > vis_wave) causal_mask(sB, col0 + 32);
                step(no, do_v_c, do_k_c, sB, sA, pB, pA, kb ^ 1, 0, kb, 0, or_else(jn3, jc), jc);
                __builtin_amdgcn_sched_barrier(0);
                t++;
                jc = jn1; jn1 = jn2; jn2 = jn3;
                if (jc.lead >= n_end) break;
                jn3 = next_turn();
            }
        };
        const bool do_v = __builtin_amdgcn_readfirstlane((int)(role_v && kt < V_ITEMS)) != 0;
        if (do_v) {
            tile_loop(yes, std::integral_constant<bool, !SPLIT>());
        } else {
            tile_loop(no, yes);
        }
        pv_half(pB, (t - 1) & 1, 1);  // P V of the last half: V of the last tile, second half
        __syncthreads();
        redo = *sFlag != 0u;  // (the same for every wave)
    }
    if (redo) {
        // ---- safe path: the whole workgroup again, tile by tile, with the classic softmax (maximum per half tile,
        // reference moved and O rescaled as needed).  One stage, no prefetch: this path is for inputs whose scores
        // climb by more than the common path's range after the first tile, not for speed.
        row_sum = 0.f;
        row_ref = -INFINITY;
        enc_ref = 0.f;
        qx[2] = 0u;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[db][i] = 0.f;
        it_word = 0;
        it_base = -32;
        it_next = 0;
        for (Turn j = next_turn(); j.lead < n_end; j = next_turn()) {
            set_tile_k(j);
            set_tile_v(j);
            set_tile_x(j);
            load_regs(false);
            load_regs(true);
            __syncthreads();  // every wave is done with the stage
            store_k(0);
            store_v(0);
            store_x(0);
            __syncthreads();
            f32x16_t s0, s1;
            uint32_t p0[8], p1[8];
            scores_half(s0, 0, 0);
            scores_half(s1, 0, 1);  // (both against the same pieces: classic() below may replace them)
            const float enc_before = enc_ref;
            classic(s0, p0, j.mine * BN);
            pv_half(p0, 0, 0);  // (before the second half may move the reference and rescale O again)
            const float fix = enc_before - enc_ref;
#pragma unroll
            for (int i = 0; i < 16; i++) s1[i] += fix;
            classic(s1, p1, j.mine * BN + 32);
            pv_half(p1, 0, 1);
        }
    }

    // ---- epilogue
    {
        const int qrow = wrow0 + r;
        float total = xhalf_sum(row_sum);
        if constexpr (KG == 2) {
            // the second group hands over its sums, its reference points and O; the first merges and stores
            float *xs = (float *)smem_all + wave * 64 + lane;  // sum, reference: 2 * NW * 64 floats
            f32x4_t *xo = (f32x4_t *)(smem_all + 2 * NW * 256) + wave * DB * 4 * 64 + lane;
            static_assert(2 * NW * 256 + NW * DB * 4 * 64 * 16 <= SM::OFF_BITS, "the hand-over fits the first group's stages");
            __syncthreads();  // (the stages' last reads)
            if (kgrp == 1) {
                xs[0] = total;
                xs[NW * 64] = row_ref;
#pragma unroll
                for (int db = 0; db < DB; db++)
#pragma unroll
                    for (int q = 0; q < 4; q++) xo[(db * 4 + q) * 64] = f32x4_t{o[db][4 * q], o[db][4 * q + 1], o[db][4 * q + 2], o[db][4 * q + 3]};
            }
            __syncthreads();
            if (kgrp == 1) return;
            const float t1 = xs[0], r1 = xs[NW * 64], top = fmaxf(row_ref, r1), safe = top == -INFINITY ? 0.f : top;
            const float w0 = fast_exp2(row_ref - safe), w1 = fast_exp2(r1 - safe);
            total = total * w0 + t1 * w1;
            row_ref = top;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x4_t v = xo[(db * 4 + q) * 64];
#pragma unroll
                    for (int e = 0; e < 4; e++) o[db][4 * q + e] = o[db][4 * q + e] * w0 + v[e] * w1;
                }
        }
        const float inv = total > 0.f ? 1.f / total : 0.f;
        if (qrow < LqS) {
            uint16_t *op = (uint16_t *)p.o + b * p.o_b + (sq.q0 + qrow) * p.o_r + h * p.o_h;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int blk = 0; blk < 2; blk++) {
                    const int c = 32 * db + 16 * blk + 8 * g;
                    if (c < p.d) {
                        u32x4_t w;
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            w[e] = E::pack2(o[db][8 * blk + 2 * e] * inv, o[db][8 * blk + 2 * e + 1] * inv);
                        *(u32x4_t *)(op + c) = w;
                    }
                }
            if (g == 0) {
                const float lse = total > 0.f ? (row_ref + __builtin_amdgcn_logf(total)) * kLn2 : INFINITY;
                p.lse[b * p.lse_b + h * p.lse_h + sq.q0 + qrow] = lse;
            }
        }
    }
}
#undef FWD_LDS

// Adds up the shares of a call with split keys and no arrival counters.  A thread has 8 elements of one row.
template <typename T> __global__ void __launch_bounds__(256) fwd_merge_kernel(const FwdParams p) {
    const int CH = p.d / 8;
    const int64_t rows = (int64_t)p.B * p.H * p.Lq, at = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= rows * CH) return;
    const int64_t row = at / CH;
    const int c = (int)(at % CH) * 8;
    float l[MAX_KEY_SPLITS];
    f32x4_t v[MAX_KEY_SPLITS][2];
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) l[s] = s < p.splits ? p.lse_part[s * rows + row] : -INFINITY;
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) {  // (the rows of O of a share without a visible key hold nothing and are not read)
        v[s][0] = v[s][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (l[s] != -INFINITY) {
            v[s][0] = *(const f32x4_t *)(p.o_part + (s * rows + row) * p.d + c);
            v[s][1] = *(const f32x4_t *)(p.o_part + (s * rows + row) * p.d + c + 4);
        }
    }
    const ShareWeights r = share_weights(l);
    f32x4_t a[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) add_share(a, r.w[s], v[s]);
    const int q = (int)(row % p.Lq), h = (int)(row / p.Lq % p.H), b = (int)(row / p.Lq / p.H);
    *(u32x4_t *)((uint16_t *)p.o + b * p.o_b + q * p.o_r + h * p.o_h + c) = merged8<T>(r.inv, a);
    if (c == 0) p.lse[b * p.lse_b + h * p.lse_h + q] = r.lse;
}

template <typename T> hipError_t launch_merge(const FwdParams &p, hipStream_t stream) {
    const int64_t items = (int64_t)p.B * p.H * p.Lq * (p.d / 8);
    hipLaunchKernelGGL((fwd_merge_kernel<T>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream, p);
    return hipGetLastError();
}

template <typename T, int D, int BN, bool CAUSAL, bool CMP, int NW = 4, int KG = 1>
hipError_t launch_one(const FwdParams &p, hipStream_t stream) {
    constexpr int BM = 32 * NW;
    constexpr int LESS = D == 128 ? 96 : D;
    const bool less = p.d <= LESS;
    auto kern = less ? fwd_colmask_kernel<T, D, LESS, BN, CAUSAL, NW, CMP, KG> : fwd_colmask_kernel<T, D, D, BN, CAUSAL, NW, CMP, KG>;
    const int smem = KG * CmSmem<D, BN>::TOTAL;
    static DynSmemLimit smem_limit[2];  // one per instantiation
    hipError_t e = smem_limit[less].ensure((const void *)kern, (int)smem);
    if (e != hipSuccess) return e;
    FwdParams pr = p;
    const int grid = row_grid(pr, BM);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW * KG), smem, stream, pr);
    return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_d(const FwdParams &p, hipStream_t stream) {
    // 256-row workgroups (8 waves, one workgroup per CU) stage every K / V tile once for twice the rows and win
    // whenever the grid still has a few workgroups per CU; smaller problems keep 128-row workgroups, two per CU
    const int64_t groups256 = (int64_t)p.B * p.H * ((p.Lq + 255) / 256);
    if constexpr (D == 128) if (groups256 >= 512) {
        if (p.cmp.on) return p.causal ? launch_one<T, D, 64, true, true, 8>(p, stream) : launch_one<T, D, 64, false, true, 8>(p, stream);
        return p.causal ? launch_one<T, D, 64, true, false, 8>(p, stream) : launch_one<T, D, 64, false, false, 8>(p, stream);
    }
    // no more 128-row workgroups than CUs: two key groups each (a row that sees a single tile gains nothing, and pays
    // a merge of a microsecond; at d <= 64 takes_key_groups() has them)
    if constexpr (D > 64) if ((int64_t)p.B * p.H * ((p.Lq + 127) / 128) <= device_cus() && p.Lk > 128) {
        if (p.cmp.on) return p.causal ? launch_one<T, D, 64, true, true, 4, 2>(p, stream) : launch_one<T, D, 64, false, true, 4, 2>(p, stream);
        return p.causal ? launch_one<T, D, 64, true, false, 4, 2>(p, stream) : launch_one<T, D, 64, false, false, 4, 2>(p, stream);
    }
    if (p.cmp.on) return p.causal ? launch_one<T, D, 64, true, true>(p, stream) : launch_one<T, D, 64, false, true>(p, stream);
    return p.causal ? launch_one<T, D, 64, true, false>(p, stream) : launch_one<T, D, 64, false, false>(p, stream);
}

}  // namespace

hipError_t launch_fwd_merge(const FwdParams &p, int dtype, hipStream_t stream) {
    return dtype == 0 ? launch_merge<bf16_tag>(p, stream) : launch_merge<fp16_tag>(p, stream);
}

// Shares that the key tiles of a row block are cut into: a chunk of a prompt against a long cache has too few row blocks for the
// chip, and a workgroup's time is the chain of its tiles.  The shares' fp32 results cost what they weigh -- 256 workgroups of 128 rows
// wrote and read 17 MB, 12 us, and two shares of 128 blocks were no faster than none -- so at most 128 blocks of 128 rows, and only
// from three shares on; a share has at least 1024 keys and (in the kernel) 512 kept ones.  The kernel is that of 64-row blocks
// (takes_key_groups).
// Only where the keys are twice the queries or more: a training step keeps the forward's workspace until its backward, which
// would hold the shares, and has as many queries as keys.  Whole keys / shares in us (a workspace without / with room for them;
// medians over 1 to 40 blocks of 2 to 300 rows, d = 128; at d = 64 0.7 to 0.85 of that), with a sixteenth, a quarter and all of the
// keys kept:
//   3072 keys   13.1 / 16.3    19.1 / 22.7    41.2 / 28.4        16384 keys   21.5 / 20.9    49.7 / 26.2    157.2 / 45.7
//   6144 keys   15.2 / 18.6    26.0 / 21.0    70.0 / 33.7        32768 keys   31.6 / 23.1    87.3 / 34.2    297.6 / 70.2
// How much is kept is not known here: with under 1024 kept keys there is a single share, whose workgroup writes the result itself
// (arrival counters; without, a merge of 3 to 4 us for nothing: 214 rows x 16/8 heads, 216 kept of 5056 16.2 / 12.8, 27 x 2/1, 644 of
// 3456, d = 64 16.6 / 13.8, in shares 223 x 16/4, 2496 of 23360 28.3 / 26.8); the other way round a share too few costs more.
// Causal calls whose last row block takes twice the average gain nothing from shares: d = 256, whole / in two, 3001 x 8/4 heads, 1024
// kept 44.7 / 53.1, 8192 x 2/1, 2048 kept 51.7 / 55.1, all 3001 kept 92 / 80; d = 128, 2048 x 8/4, all kept 32.8 / 37.9.
int key_shares(const FwdParams &p) {
    if (p.cu_q || p.d > 128 || p.Lq < 2 || p.Lk / 2 < p.Lq) return 1;
    const int64_t blocks = (int64_t)p.B * p.H * ((p.Lq + 127) / 128);
    int64_t s = blocks > 0 ? device_cus() / 2 / blocks : 1;
    if (s > p.Lk / 1024) s = p.Lk / 1024;
    if (s > MAX_KEY_SPLITS) s = MAX_KEY_SPLITS;
    return s < 3 ? 1 : (int)s;
}
int fwd_key_splits(const FwdParams &p) {
    return use_compact(p) && fwd_colmask_applicable(p) && !fwd_stream_applicable(p) ? key_shares(p) : 1;
}

bool fwd_colmask_applicable(const FwdParams &p) {
    const bool mask_ok = !p.mask || p.m_r == 0;
    const bool bias_ok = !p.bias || p.bi_r == 0;
    return mask_ok && bias_ok && (p.Lk + 31) / 32 <= MAX_TILES;
}

// Whether 64-row workgroups of four key groups (fdma_fwd_wide.hip) take a call at head dims up to 128: twice the workgroups of
// 128-row ones, with half the chain of tiles and a merge of a microsecond.
//   * d = 65 .. 128, one to a CU, as long as all of them run at once: 1.13 to 1.35 times as fast over 24 calls of 4 to 256 blocks; 352
//     blocks (2 x 700 rows x 16 heads) 29.9 against 21.6 us.  A row that sees a single tile gains nothing (128 x 128: 10.7
//     either way).
//   * d <= 64, two to a CU: up to two and a half blocks per CU 1.25 to 1.65 times over 11 calls; 768 blocks (2 x 1500 x 16 heads, 700
//     kept) 29.3 against 27.8 us, ragged 4000 to 1000 x 16 140 against 125.
// Causal ragged batches further, up to two blocks per CU, three at d <= 64, where one entry of 1024 rows or more has half of them all: the call
// takes what the last blocks of that entry take.  128-row blocks / these, us: 2000, 100, 700, 30 x 8/4 heads, d = 128 45.5 / 27.7 (forward + backward
// 146 / 129), 3000, 1000 x 8/4 58.6 / 42.1, 4000, 4000 x 4/2 60.7 / 55.6; d = 96 5000, 50, 60 x 4/2 89 / 51; d = 64 1500, 1500 x 16/4 29.7 / 26.3.
// Entries of one length keep the line: four of 1024 x 8/8, d = 128 25.2 / 26.2, three of 1100 24.7 / 26.9, not causal or compacted calls as well
// (2600 x 8/2, d = 128, causal, 96 / 500 / all kept 15.9 / 17.6, 21.3 / 19.7, 48.8 / 39.4, not causal 15.0 / 17.2, 20.9 / 24.5, 51.0 / 66.2).
// (A ragged batch has at most total / 64 blocks per head and one more per entry.)
int64_t fwd_blocks64(const FwdParams &p) { return p.cu_q ? (int64_t)p.H * (p.total_q / 64 + p.B) : (int64_t)p.B * p.H * ((p.Lq + 63) / 64); }
static bool takes_key_groups(const FwdParams &p) {
    const int64_t blocks64 = fwd_blocks64(p);
    if (p.cu_q && p.causal && p.Lq >= 1024 && 2 * (int64_t)p.Lq >= p.total_q && blocks64 <= (p.d > 64 ? 2 : 3) * device_cus()) return true;
    if (p.d > 64) return blocks64 <= device_cus() && p.Lk > 128;
    return 2 * blocks64 <= 5 * (int64_t)device_cus();
}

// Whether the forward can take handed-over lists of kept keys as they are, without copies of their rows (which a backward wants: a call whose
// workspace holds them makes them).  The gather in front, 5 to 7 us, is gone; a tile pays two reads of LDS and a product per row piece.  Copies /
// rows where they lie, us, the whole layer: 3001 tokens x 8/4 heads, d = 256, 1024 kept 50.7 / 47.4, 8192 x 8/4, 2048 kept 101 / 100, 2 x 6000
// x 8/4, all kept 321 / 319; d = 128: 2000 x 8/4, 500 kept 25.2 / 21.5, 2 x 1024 x 8/4, all kept 31.1 / 26.1, 7000 x 2/1, 3000 kept 48.4 / 43.9;
// d = 96 2000 x 8/4, 128 kept 22.0 / 20.1; d = 64 2 x 3000 x 2/1, 900 kept 25.5 / 21.7.  Above head dim 128 not with 64-row blocks, whose
// registers it spills (1000 x 8/4, 300 kept 36.7 / 37.3).
// Causal calls up to two blocks of 64 rows per CU, three at head dims up to 64, beyond what takes_key_groups gives the kernel where it reads copies.  96 / 500 / all
// kept: d = 128 2048 x 16/8 (512 blocks) 28.4 / 25.6, 33.8 / 30.5, 55.2 / 45.2; d = 96 4000 x 8/4 (504) 25.4 / 23.6, 29.4 / 27.4, 69.1 / 58.6;
// d = 64 3072 x 16/8 (768) 25.2 / 22.1, 29.0 / 25.2, 64.8 / 49.2; 30 layers near the lines 1.12 times, none slower.  Beyond: d = 128 1500 x 32/16 (768),
// 128, 512, 1400 kept 30.9 / 33.6, 38.8 / 41.2, 57.9 / 55.6, d = 64 4096 x 16/8 (1024) 24.8 / 25.7, 29.1 / 29.5, 42.4 / 37.9.
bool fwd_from_lists(const FwdParams &p) {
    if (!p.kept_idx || !p.mask || p.cmp.on || p.cu_q || p.kv_share > 1 || !use_compact(p) || !fwd_colmask_applicable(p) || fwd_stream_applicable(p)) return false;
    const int64_t r = p.k_r > p.v_r ? p.k_r : p.v_r;  // (row offsets are 32-bit numbers)
    const int64_t blocks64 = fwd_blocks64(p), cus = device_cus();
    const bool grid_ok = p.d > 128 ? blocks64 > cus : takes_key_groups(p) || (p.causal && p.Lk > 128 && blocks64 <= (p.d > 64 ? 2 : 3) * cus);
    return grid_ok && key_shares(p) == 1 && p.k_r >= 0 && p.v_r >= 0 && (p.Lk * r + p.d) * 2 < (int64_t)1 << 32;
}

int64_t fwd_share_units(const FwdParams &p) {
    FwdParams pr = p;
    return row_grid(pr, fwd_share_block(p));
}
int fwd_share_block(const FwdParams &p) { return p.d > 128 && fwd_blocks64(p) > device_cus() ? 128 : 64; }

hipError_t launch_fwd_colmask(const FwdParams &p, int dtype, hipStream_t stream) {
    if (p.cmp.on && p.cmp.img_kv) return launch_fwd_stream(p, dtype, stream);  // (the pre-pass has written tile images)
    // head dims up to 64 / 128 (a head dim in between runs in the next larger instantiation), above in a kernel of their own
    if (p.d > 128) return launch_fwd_wide(p, dtype, stream);
    if (fwd_from_lists(p) || takes_key_groups(p)) {  // (and all calls in shares: three shares are at most a third of a 64-row block per CU, see key_shares)
        const hipError_t e = launch_fwd_wide(p, dtype, stream);
        if (e != hipSuccess || !p.cmp.on || p.splits <= 1 || p.dec_counter) return e;
        return launch_fwd_merge(p, dtype, stream);
    }
    if (dtype == 0) return p.d <= 64 ? launch_d<bf16_tag, 64>(p, stream) : launch_d<bf16_tag, 128>(p, stream);
    return p.d <= 64 ? launch_d<fp16_tag, 64>(p, stream) : launch_d<fp16_tag, 128>(p, stream);
}

}  // namespace fdma
