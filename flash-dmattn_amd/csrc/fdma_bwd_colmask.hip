// Backward dynamic-mask attention for gfx950, column-mask specialisation of the two main kernels.
//
// Same math and same reference counterparts as fdma_bwd.hip
// (compute_dq_dk_dv_1colblock, csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the reference), for
// mask and bias that are absent or broadcast over the query dimension ([B, {1,Hk,H}, 1, Lk]).
// "Keep" and the bias are then properties of the key column:
//   * in the dK/dV kernel a lane owns one key column for the whole kernel, so mask and bias
//     collapse to one fused per-lane constant (bias*log2e, or -inf when masked / beyond Lk): no
//     mask or bias loads in the loop, no selects -- exp2(-inf) = 0 does the masking;
//   * dBias is the column sum of dS, accumulated in a register and written once;
//   * in the dQ kernel the fused vector is staged per tile exactly as in the forward kernel and
//     fully masked 64-key tiles are skipped through the same LDS bitmap.
// K and V are stationary in the dK/dV kernel (B operands: in registers, except V at d = 128, which every
// lane parks in LDS as a private spill so that two workgroups fit on a CU); Q / dO tiles and the row
// statistics stream through double-buffered LDS, fetched two steps ahead of their use.  Workgroup ids
// are remapped so that workgroups sharing an XCD's L2 share the streamed operands.
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_bwd_reduce.h"
#include "fdma_bwd_units.h"

namespace fdma {

namespace {

constexpr int NTHREADS = 256;

// ------------------------------------------------------------------------------------------------
// dK / dV / dBias
// ------------------------------------------------------------------------------------------------
// Query rows per step.  At d = 128 the stationary K / V fragments and the dK / dV accumulators alone take 192 registers
// per lane; with 32-row steps and V parked in LDS (every lane re-reads its own row: a private spill, no sharing) the
// kernel fits in 256 registers and 70 KB of LDS, so that two workgroups share a CU and fill each other's stalls.
template <int D> struct KvcSmem {
    static constexpr int BM = D > 64 ? 32 : 64;
    static constexpr bool V_LDS = D > 64;
    static constexpr int S = LdsTile<D>::S;
    static constexpr int Q_BYTES = BM * S * 2;
    static constexpr int STAGE = 2 * Q_BYTES + 2 * BM * 4;  // Q, dO, LSE, D
    static constexpr int OFF_V = 2 * STAGE;
    static constexpr int TOTAL = OFF_V + (V_LDS ? KV_BN * S * 2 : 0);
};

// Entries of a ragged batch longest first and dealt to all XCDs (ragged_lists_per_pair), up to head dim 128; at 256 the plain order.
template <int D> constexpr bool RAGGED_TURNS = D <= 128;

// CMP: the key axis is the compacted list of kept columns (fdma_compact.hip); a lane still owns one key,
// reads it from the dense copies, and writes its gradients to the key's original row / column.
// DC: the head dims that are worked on, 96 of a 128-wide tile for head dims 65 to 96 (here and in dQ).  The tile itself stays as wide: its
// swizzle and the direct loads are made for rows of 256 bytes.  A quarter of the products is gone, and with it the spilled registers (256 and up
// to 52 bytes of scratch a lane; 223 and none).  Forward + backward at d = 96, 128 dims / 96 of them, us: ragged 3601 and others x 32/8
// heads 658 / 587, 4466 and others x 16/16 519 / 461, 2752 and others x 2/1 137 / 126; layer of 4 x 2432 x 16/8 365 / 333; 8256 x 16/8, 128 kept
// 124 / 116.
template <typename T, int D, int DC, bool CAUSAL, bool CMP>
__global__ void __launch_bounds__(NTHREADS, 2) bwd_dkdv_colmask_kernel(const BwdParams p) {
    using E = Elem<T>;
    using SM = KvcSmem<D>;
    using TL = LdsTile<D>;
    constexpr int BM = SM::BM;       // query rows per step
    constexpr int SUB = KV_BM / BM;  // steps per planning block
    constexpr bool V_LDS = SM::V_LDS;
    constexpr int KS = DC / 16;
    constexpr int DB = DC / 32;
    constexpr int MB = BM / 32;
    constexpr int CH = D / 8, RPP = NTHREADS / CH, Q_IT = BM / RPP;
    // DMA: the Q / dO tiles and the row statistics of a step go from global memory straight into LDS
    // (global_load_lds: a wave writes 64 consecutive 16-byte or 4-byte pieces, so the swizzle of the tile is applied
    // to the GLOBAL address of each lane's piece); no staging registers, no LDS stores, and the loads are issued
    // between the MFMAs a whole step ahead of the barrier that publishes them.  Needs rows of exactly 256 bytes.
    constexpr bool DMA = TL::SWZ;
    static_assert(!DMA || (BM == 32 && NTHREADS == 256), "the direct loads are laid out for 32-row steps and four waves");

    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int G = f.H / f.Hk;
    const KvItem it = kv_item<CMP>(p, RAGGED_TURNS<D>);
    if (!it.valid) return;
    const int pair = it.pair, n_block = it.n_block, g_lo = it.g_lo, g_hi = it.g_hi, seg = it.seg, Sm = it.Sm, Q = it.Q, part = it.part;
    int slot = it.slot;
    const int b = pair / f.Hk, hk = pair % f.Hk;
    const int n0 = n_block * KV_BN;
    const SeqInfo sq = seq_info(f, b);  // this batch entry's lengths and first rows (ragged batch: from cu_seqlens)
    const int LqS = sq.Lq, LkS = sq.Lk;
    const int Lk = CMP ? f.cmp.count[pair] : LkS;  // key columns on this pair's (possibly compacted) key axis
    if (n0 >= Lk) return;  // the compacted list, or a shorter sequence of a ragged batch, ends before this block
    // original key axis: this part's steps [first_step, first_step + part_steps) of the unit's
    int first_step = 0, part_steps = 0;
    if (!CMP && p.kv_most > 1) {
        const int steps = G * kv_unit_steps(LqS, LkS, CAUSAL, n0, BM);
        const int n_parts = kv_parts_of(steps, p.kv_quota ? p.kv_quota : ragged_part_quota(f, BM), p.kv_most);
        if (part >= n_parts) return;
        if (n_parts > 1) {
            first_step = (int)((int64_t)steps * part / n_parts);
            part_steps = (int)((int64_t)steps * (part + 1) / n_parts) - first_step;
            slot = kv_unit_slot(p, b, hk, n_block) + part;
        }
    }
    const int key = n0 + wave * 32 + r;  // the key column this lane owns
    const int key_c = key < Lk ? key : Lk - 1;
    const int shift = LkS - LqS;
    // original column indices: of this lane's key, of the workgroup's first key and of the wave's last key
    const int32_t *cidx = CMP ? f.cmp.idx + (int64_t)pair * f.cmp.ld : nullptr;
    const int okey = CMP ? cidx[key_c] : key;
    const int okey_first = CMP ? cidx[n0] : n0;
    const int okey_wlast = CMP ? cidx[n0 + wave * 32 + 31 < Lk ? n0 + wave * 32 + 31 : Lk - 1] : n0 + wave * 32 + 31;

    // ---- stationary K / V fragments (B operands): lane holds K[key][16ks + 8g .. +8]
    u32x4_t kf[KS], vf[V_LDS ? 1 : KS];
    char *sVt = smem + SM::OFF_V;
    uint32_t v_base = TL::frag_base(wave * 32 + r, g);  // V_LDS: this lane's V row, its chunks
    {
        const uint16_t *kp = (const uint16_t *)f.k + b * f.k_b + (sq.k0 + key_c) * f.k_r + hk * f.k_h;
        const uint16_t *vp = (const uint16_t *)f.v + b * f.v_b + (sq.k0 + key_c) * f.v_r + hk * f.v_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            u32x4_t kv = {0, 0, 0, 0}, vv = {0, 0, 0, 0};
            if (c < f.d) { kv = *(const u32x4_t *)(kp + c); vv = *(const u32x4_t *)(vp + c); }
            // K is only used for the scores here: scale it by softmax_scale * log2(e) once, so that the MFMA
            // accumulates exp2-domain scores on top of the column constant (no multiply per element later)
#pragma unroll
            for (int e = 0; e < 4; e++) kv[e] = E::pack2(E::lo(kv[e]) * f.scale_log2, E::hi(kv[e]) * f.scale_log2);
            kf[ks] = kv;
            if (V_LDS) *(u32x4_t *)(sVt + TL::frag_at(v_base, ks)) = vv;
            else vf[ks] = vv;
        }
    }

    v_base += lds0 + SM::OFF_V;  // from here on an absolute LDS address (see lds_ld128)

    f32x16_t dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) { dk[db][i] = 0.f; dv[db][i] = 0.f; }

    const int M_blocks = (LqS + KV_BM - 1) / KV_BM;
    // query blocks that see the workgroup's first key: [m_start, M_blocks)
    const int m_start = M_blocks - dkdv_query_blocks(LqS, LkS, CAUSAL, okey_first);
    // this workgroup's query blocks [m_lo, m_hi): all of them, or one of the unit's equal segments
    int m_lo = m_start, m_hi = M_blocks;
    if (CMP && slot >= 0) {
        const int n_seg = dkdv_segments(M_blocks - m_start, Q, Sm);
        if (seg >= n_seg) return;  // the reduce kernel knows that this slot stays unwritten
        const int len = (M_blocks - m_start + n_seg - 1) / n_seg;
        m_lo = m_start + seg * len;
        m_hi = m_lo + len < M_blocks ? m_lo + len : M_blocks;
    }
    // the planning blocks [m_lo, m_hi) in steps of BM rows: [s_lo, s_hi), without steps entirely beyond Lq
    const int S_blocks = (LqS + BM - 1) / BM;
    const int s_lo = m_lo * SUB, s_hi = m_hi * SUB < S_blocks ? m_hi * SUB : S_blocks;
    const int n_m = s_hi > s_lo ? s_hi - s_lo : 0;
    // (g outer, m inner); the query blocks are walked from the LAST one down, so that the
    // workgroups of one (batch, kv head) pair, which run side by side on an XCD, all begin at the same
    // Q / dO tile and stream the same tiles at the same time (L2 hits instead of re-fetches)
    const int n_steps = !CMP && slot >= 0 ? part_steps : n_m * (g_hi - g_lo);

    const bool has_bias = f.bias != nullptr;
    const bool use_accum = p.dbias_accum != nullptr;

    // Fused per-lane column constant for query head h: bias*log2e, or -inf when the column is dropped.  It travels
    // with the prefetch of the step that needs it: raw, unconditional loads (an absent mask / bias is read from K,
    // any valid address, and ignored) issued first in load_step, turned into the constant after the compute.
    uint32_t cm_raw = 1, cb_raw = 0;
    const uint8_t *mask_ld = f.mask ? f.mask : (const uint8_t *)f.k;
    const uint16_t *bias_ld = has_bias ? (const uint16_t *)f.bias : (const uint16_t *)f.k;
    auto column_const_load = [&](int h) {
        if (CMP) {
            cb_raw = __float_as_uint(f.cmp.fb[(int64_t)(b * f.cmp.Hfb + (f.cmp.Hfb == f.H ? h : hk)) * f.cmp.ld + key_c]);
        } else {
            const int hm = f.mask ? (f.Hm == f.H ? h : (f.Hm == 1 ? 0 : hk)) : 0;
            const int hb = has_bias ? (f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk)) : 0;
            cm_raw = mask_ld[f.mask ? b * f.m_b + hm * f.m_h + key_c : 0];
            cb_raw = bias_ld[has_bias ? b * f.bi_b + hb * f.bi_h + key_c : 0];
        }
    };
    auto column_const_value = [&]() -> float {
        if (key >= Lk) return -INFINITY;
        if (CMP) return __uint_as_float(cb_raw);
        if (f.mask && !cm_raw) return -INFINITY;
        return has_bias ? E::lo(cb_raw) * kLog2e : 0.f;
    };

    // ---- staging of Q / dO / LSE / D for one step (global -> registers -> LDS)
    const int qc = tid % CH, qr0 = tid / CH;
    const int qcol = (qc * 8 < f.d) ? qc * 8 : 0;  // head-dim chunks beyond d: re-read chunk 0 (K/V fragments there are zero)
    u32x4_t qreg[Q_IT], doreg[Q_IT];
    float lreg = INFINITY, dreg = 0.f;
    bool stat_ok = false;
    // Byte offsets of this thread's loads inside a 64-row block are loop invariants -- one set for full blocks, one
    // for the (only) partial block at the end of the queries, whose rows beyond Lq are clamped to the last row
    // (finite duplicates, cancelled by LSE = +inf) -- so a load is one instruction with a scalar block base.
    const int m_last = (LqS - 1) / BM, row_last = (LqS - 1) % BM;
    uint32_t qoff[Q_IT], qoff_l[Q_IT], dooff[Q_IT], dooff_l[Q_IT];
#pragma unroll
    for (int it = 0; it < Q_IT; it++) {
        // DMA: load n = 2 * wave + it of a tile fills LDS bytes [1024 n, 1024 n + 1024): rows 4n .. 4n+3, lane l the
        // chunk POSITION l % 16 of row 4n + l / 16, which holds chunk position ^ swz(row) of the global row
        const int n = 2 * wave + it;
        const int row = DMA ? 4 * n + (lane >> 4) : qr0 + it * RPP, row_c = row < row_last ? row : row_last;
        const int chunk = (lane & 15) ^ (int)TL::swz(row);
        const int col = DMA ? ((chunk * 8 < f.d) ? chunk * 8 : 0) : qcol;
        qoff[it] = (uint32_t)(row * f.q_r + col) * 2;
        qoff_l[it] = (uint32_t)(row_c * f.q_r + col) * 2;
        dooff[it] = (uint32_t)(row * p.do_r + col) * 2;
        dooff_l[it] = (uint32_t)(row_c * p.do_r + col) * 2;
    }
    gptr_t ld_qbase = nullptr, ld_dobase = nullptr;  // block bases of the step being fetched (scalar registers)
    bool ld_partial = false;
    // tile load `n` of the step being fetched: 0 .. Q_IT-1 are Q rows, Q_IT .. 2*Q_IT-1 dO rows
    auto load_item = [&](int n) {
        if (n < Q_IT) qreg[n] = *(const __attribute__((address_space(1))) u32x4_t *)(ld_qbase + (ld_partial ? qoff_l[n] : qoff[n]));
        else doreg[n - Q_IT] = *(const __attribute__((address_space(1))) u32x4_t *)(ld_dobase + (ld_partial ? dooff_l[n - Q_IT] : dooff[n - Q_IT]));
    };
    // everything of a step's fetch except the tile loads: block bases, column constant, row statistics
    auto load_step = [&](int step, bool with_tiles) {
        const int gi = g_lo + (step + first_step) / n_m, mi = s_hi - 1 - (step + first_step) % n_m;  // last query block first: see below
        const int h = hk * G + gi, m0 = mi * BM;
        column_const_load(h);
        ld_qbase = uniform_ptr((const uint16_t *)f.q + b * f.q_b + h * f.q_h + (sq.q0 + m0) * f.q_r);
        ld_dobase = uniform_ptr((const uint16_t *)p.dout + b * p.do_b + h * p.do_h + (sq.q0 + m0) * p.do_r);
        ld_partial = mi == m_last;
        if (with_tiles) {
#pragma unroll
            for (int n = 0; n < 2 * Q_IT; n++) load_item(n);
        }
        // row statistics: raw, unconditional loads from a clamped row (nothing may look at a loaded value here, or the
        // wait for it would also cover the tile loads above); range check and scaling happen in store_step
        {
            const int qq = m0 + (tid & (BM - 1));
            stat_ok = qq < LqS;
            const int qc = stat_ok ? qq : LqS - 1;
            lreg = f.lse[b * f.lse_b + h * f.lse_h + sq.q0 + qc];
            dreg = p.softmax_d[b * p.sd_b + h * p.sd_h + sq.q0 + qc];
        }
    };
    auto store_step = [&](int buf) {
        char *base = smem + buf * SM::STAGE;
#pragma unroll
        for (int it = 0; it < Q_IT; it++) {
            const uint32_t off = TL::chunk(qr0 + it * RPP, qc);
            *(u32x4_t *)(base + off) = qreg[it];
            *(u32x4_t *)(base + SM::Q_BYTES + off) = doreg[it];
        }
        if (tid < BM) {
            ((float *)(base + 2 * SM::Q_BYTES))[tid] = stat_ok ? lreg * kLog2e : INFINITY;
            ((float *)(base + 2 * SM::Q_BYTES + BM * 4))[tid] = stat_ok ? dreg : 0.f;
        }
    };

    // ---- DMA staging: block bases of the step being fetched, and its pieces one by one.  Piece 0 .. 2*Q_IT-1: this
    // wave's Q / dO loads (1 KB each); piece 2*Q_IT (wave 3 only): the row statistics, 32 LSE values and 32 D values
    // as ONE 4-byte load (lanes 0-31 / 32-63), raw -- log2(e) is applied where the LSE is used, and rows beyond the
    // end of the queries are clamped here and masked there.
    typedef __attribute__((address_space(3))) void lds_void_t;
    typedef const __attribute__((address_space(1))) void gvoid_t;
    // The steps are walked with counters and running pointers (no division, no 64-bit products per step): inside a
    // query head the query block index falls by one per step, at a head change everything jumps by loop constants.
    const int gi0 = CMP || n_steps == 0 ? g_lo : first_step / n_m, mi0 = s_hi - 1 - (CMP || n_steps == 0 ? 0 : first_step % n_m);
    int dma_gi = gi0, dma_mi = mi0;  // head and query block of the step being fetched
    gptr_t dma_q = nullptr, dma_do = nullptr, dma_stat = nullptr;  // its Q / dO block bases, this lane's statistic
    char *dma_dst = nullptr;
    const int64_t q_step = -(int64_t)BM * f.q_r * 2, do_step = -(int64_t)BM * p.do_r * 2;
    const int64_t q_head = (int64_t)f.q_h * 2 - (int64_t)(n_m - 1) * q_step, do_head = (int64_t)p.do_h * 2 - (int64_t)(n_m - 1) * do_step;
    const int64_t stat_head = (int64_t)(lane < 32 ? f.lse_h : p.sd_h) * 4 + (int64_t)(n_m - 1) * BM * 4;
    if (DMA && n_steps > 0) {
        const int h0 = hk * G + gi0, m00 = dma_mi * BM;
        dma_q = (gptr_t)((const uint16_t *)f.q + b * f.q_b + h0 * f.q_h + (sq.q0 + m00) * f.q_r);
        dma_do = (gptr_t)((const uint16_t *)p.dout + b * p.do_b + h0 * p.do_h + (sq.q0 + m00) * p.do_r);
        dma_stat = (gptr_t)(lane < 32 ? f.lse + b * f.lse_b + h0 * f.lse_h + sq.q0 + m00 + (lane & 31)
                                        : p.softmax_d + b * p.sd_b + h0 * p.sd_h + sq.q0 + m00 + (lane & 31));
    }
    // sets up the fetch of the step the counters stand at (into stage `buf`)
    auto dma_begin = [&](int buf) {
        ld_qbase = dma_q;
        ld_dobase = dma_do;
        ld_partial = dma_mi == m_last;
        dma_dst = smem + buf * SM::STAGE;
    };
    // moves the counters to the following step; past the last step they stay (its tiles are fetched again and dropped)
    auto dma_advance = [&](bool more) {
        if (!more) return;
        if (dma_mi == s_lo) {
            dma_mi = s_hi - 1;
            dma_gi++;
            dma_q += q_head; dma_do += do_head; dma_stat += stat_head;
        } else {
            dma_mi--;
            dma_q += q_step; dma_do += do_step; dma_stat -= BM * 4;
        }
    };
    // The direct loads are written in assembly and waited for by hand (publish() below): issued through the
    // compiler's builtin, every LDS read behind one of them waited for all LDS operations in flight -- the compiler
    // cannot tell which stage a direct load fills -- and the fragment reads could not run ahead of their MFMAs.
    // (m0 carries the LDS address of a direct load; it is a reserved register that nothing else in this kernel uses.)
    auto dma_piece = [&](int n) {
        const uint32_t dst = lds_addr(dma_dst);
        if (n < Q_IT) {
            load_lds16(ld_partial ? qoff_l[n] : qoff[n], ld_qbase, __builtin_amdgcn_readfirstlane(dst + (2 * wave + n) * 1024));
        } else if (n < 2 * Q_IT) {
            load_lds16(ld_partial ? dooff_l[n - Q_IT] : dooff[n - Q_IT], ld_dobase, __builtin_amdgcn_readfirstlane(dst + SM::Q_BYTES + (2 * wave + n - Q_IT) * 1024));
        } else {
            // (every wave fetches the same 256 bytes: cheaper than a branch in the middle of the MFMAs.)  In the last,
            // partial block the rows beyond the end of the queries read the last row's numbers (masked where used).
            const int over = ld_partial ? (lane & 31) - row_last : 0;
            gptr_t sp = dma_stat - (over > 0 ? over * 4 : 0);
            load_lds4_at(sp, __builtin_amdgcn_readfirstlane(dst + 2 * SM::Q_BYTES));
        }
    };
    // end of a step: a wave waits for its own direct loads (and LDS stores), then the barrier publishes everybody's
    auto publish = [&]() {
        if constexpr (DMA) {
            __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0); expcnt not waited for
            __builtin_amdgcn_s_barrier();
        } else {
            __syncthreads();
        }
    };

    const int a_row = pi_row(r);
    const TrLane tr = tr_lane(lane);
    uint32_t tr_off = lds0 + TL::tr_base(g, tr);  // (absolute LDS addresses of stage 0's Q tile)
    uint32_t a_off = lds0 + TL::frag_base(a_row, g);
    const uint32_t stat_off = lds0 + 32 * g;  // this lane's eight rows of a block of sixteen row statistics

    float colsum = 0.f;
    float cconst = 0.f;

    // Pipeline: step i is computed from LDS stage i & 1.  The registers hold step i+1 (fetched during the dK / dV
    // MFMAs of step i-1, a whole step earlier -- these tiles come from HBM, not from a cache); they go to the other
    // stage between the first GEMM pair and the softmax of step i, and the loads of step i+2 then reuse them, issued
    // one by one between the dK / dV MFMAs (all at once, from every wave at the same moment, they would queue up at the
    // CU's address unit while the matrix pipe idles).
    if (n_steps > 0) {
        if constexpr (DMA) {
            column_const_load(hk * G + gi0);
            dma_begin(0);
#pragma unroll
            for (int n = 0; n <= 2 * Q_IT; n++) dma_piece(n);
            dma_advance(n_steps > 1);
            cconst = column_const_value();
        } else {
            load_step(0, true);
            store_step(0);
            cconst = column_const_value();
            load_step(n_steps > 1 ? 1 : 0, true);
        }
        publish();
    }

    int cur_gi = gi0, cur_mi = mi0;  // (DMA: head and query block of the current step, walked like the fetch)
    // (one step; the LDS stage is a compile-time constant -- the loop below runs the steps in pairs -- so that every
    // stage base folds into the offset field of the LDS instructions instead of costing an addition per access)
    auto one_step = [&](auto buf_c, const int step) {
        constexpr int buf = decltype(buf_c)::value;
        const int gi = DMA ? cur_gi : g_lo + (step + first_step) / n_m;  // last query block first: see below
        const int mi = DMA ? cur_mi : s_hi - 1 - (step + first_step) % n_m;
        const int h = hk * G + gi;
        const int m0 = mi * BM;
        // The swizzled addresses are these lane constants XOR a compile-time value: recomputed where they are used
        // (one VALU operation each); hoisted out of the loop they would cost 30 registers that the kernel does not have.
        if (TL::SWZ) asm volatile("" : "+v"(a_off), "+v"(tr_off), "+v"(v_base));
        // DMA: the next step's tiles go to the other stage (its readers finished before the last barrier), a piece
        // every few MFMAs; the column constant is fetched again only when the next step belongs to another query head
        const bool head_next = DMA && step + 1 < n_steps && mi == s_lo;
        if constexpr (DMA) {
            dma_begin(buf ^ 1);
            if (head_next) column_const_load(h + 1);
        }

        // ---- S = Q K^T and dP = dO V^T (M = query, N = key); fragment reads run a batch ahead
        f32x16_t s[MB], dp[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                // (one move per accumulator register, written out: as a plain splat the compiler builds the vector in
                // other registers first and copies it over, 31 instructions for 16)
                asm volatile("v_mov_b32 %0, %1" : "=v"(s[mb][i]) : "v"(cconst));
                dp[mb][i] = 0.f;
            }
        {
            constexpr int NF = 2 * MB * KS, FR = D > 64 ? 3 : 8;  // fragment f: (ks, mb, which) with which = 0: Q, 1: dO
            u32x4_t a[NF];
            auto frag = [&](int fi) {
                const int which = fi & 1, mb = (fi >> 1) % MB, ks = (fi >> 1) / MB;
                return lds_ld128(TL::frag_at(a_off, ks) + (uint32_t)(buf * SM::STAGE + which * SM::Q_BYTES + 32 * mb * TL::ROW_BYTES));
            };
            // (V parked in LDS: its fragment of a k-step is read one k-step ahead as well -- read where it is used, every
            // dP MFMA waited for its own read; a scheduling barrier per MFMA keeps the reads ahead)
            constexpr int FRV = 1;
            u32x4_t vl[V_LDS ? KS : 1];
            if constexpr (V_LDS) {
#pragma unroll
                for (int ks = 0; ks < FRV; ks++) vl[ks] = lds_ld128(TL::frag_at(v_base, ks));
            }
#pragma unroll
            for (int fi = 0; fi < FR; fi++) a[fi] = frag(fi);
#pragma unroll
            for (int fi = 0; fi < NF; fi++) {
                if (fi + FR < NF) a[fi + FR] = frag(fi + FR);
                const int which = fi & 1, mb = (fi >> 1) % MB, ks = (fi >> 1) / MB;
                if constexpr (V_LDS) {
                    if (which && mb == 0 && ks + FRV < KS) vl[ks + FRV] = lds_ld128(TL::frag_at(v_base, ks + FRV));
                }
                if (which) dp[mb] = E::mfma(a[fi], V_LDS ? vl[V_LDS ? ks : 0] : vf[V_LDS ? 0 : ks], dp[mb]);
                else s[mb] = E::mfma(a[fi], kf[ks], s[mb]);
                if constexpr (DMA) {
                    constexpr int EVERY = NF / (2 * Q_IT + 1);
                    if (fi % EVERY == 1 && fi / EVERY <= 2 * Q_IT) dma_piece(fi / EVERY);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the registers (step i+1) go to the other LDS stage, whose readers finished before the last barrier
        __builtin_amdgcn_sched_barrier(0);
        float cconst_next = cconst;
        if constexpr (!DMA) {
            if (step + 1 < n_steps) {
                store_step(buf ^ 1);
                cconst_next = column_const_value();
            }
        }
        __builtin_amdgcn_sched_barrier(0);

        // ---- P = exp2(S - LSE*log2e), S already scaled and offset by the column constant ; dS = P * (dP - D)
        // diagonal step: some (query, key) pairs of this wave are above the causal diagonal
        // (DMA: the statistics are raw, so rows beyond the end of the queries -- clamped duplicates in the last, partial
        // block -- are masked here as well)
        const bool diag = (CAUSAL && (okey_wlast > m0 + shift)) || (DMA && m0 + BM > LqS);
        uint32_t ppk[MB * 8], dpk[MB * 8];
        float part = 0.f;
        // softmax and dS of one block of 16 query rows (8 per lane) in three pieces, so that the MFMAs of the rows whose
        // probabilities are finished can be issued between the pieces of the next block: A = statistics, exp2, dP - D;
        // M = masking (diagonal steps only: rows above the causal diagonal or beyond the end of the queries give
        // P = 0); B = dS, column sum, conversion to 16 bits
        float pv[8], dsv[8];
        auto soft_a = [&](auto mb_c, auto blk_c) {
            constexpr int mb = decltype(mb_c)::value, blk = decltype(blk_c)::value;
            const uint32_t so = buf * SM::STAGE + 2 * SM::Q_BYTES + (32 * mb + 16 * blk) * 4;  // LSE; D is BM floats on
            const f32x4_t l0 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so)), l1 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + 16));
            const f32x4_t d0 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + BM * 4)), d1 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + BM * 4 + 16));
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int ii = 8 * blk + e;
                const float lse2 = e < 4 ? l0[e] : l1[e - 4];
                const float dd = e < 4 ? d0[e] : d1[e - 4];
                pv[e] = fast_exp2(DMA ? __builtin_fmaf(lse2, -kLog2e, s[mb][ii]) : s[mb][ii] - lse2);
                dsv[e] = dp[mb][ii] - dd;
            }
        };
        auto soft_m = [&](auto mb_c, auto blk_c) {
            constexpr int mb = decltype(mb_c)::value, blk = decltype(blk_c)::value;
            if (diag) {
                asm volatile("" ::: "memory");  // keep a real branch: only diagonal steps pay
                int lim = CAUSAL ? okey - shift - m0 - 32 * mb - 16 * blk - 8 * g : 0;  // rows e >= lim see this key
                int lim_hi = DMA ? LqS - m0 - 32 * mb - 16 * blk - 8 * g : 8;            // rows e < lim_hi exist
                asm volatile("" : "+v"(lim), "+v"(lim_hi));  // (the comparisons stay inside the branch)
#pragma unroll
                for (int e = 0; e < 8; e++) pv[e] = (e >= lim && e < lim_hi) ? pv[e] : 0.f;
            }
        };
        auto soft_b = [&](auto mb_c, auto blk_c) {
            constexpr int mb = decltype(mb_c)::value, blk = decltype(blk_c)::value;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                dsv[e] *= pv[e];
                part += dsv[e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ppk[mb * 8 + blk * 4 + e] = E::pack2(pv[2 * e], pv[2 * e + 1]);
                dpk[mb * 8 + blk * 4 + e] = E::pack2(dsv[2 * e], dsv[2 * e + 1]);
            }
        };
        // ---- dV^T += dO^T P ; dK^T += Q^T dS   (M = d, N = key, contraction = query), pairs [idx0, idx1) of (16-row
        // block, d block); the transposing fragment reads run one pair ahead of the MFMAs that use them
        constexpr int NP = (BM / 16) * DB;
        u32x4_t a1[2], a2[2];
        auto tr_frag = [&](int idx, int slot) {
            const int qb = idx / DB, db = idx % DB;
            const uint32_t off = TL::tr_at(tr_off, qb, db, 0), off_hi = TL::tr_at(tr_off, qb, db, 1);
            constexpr uint32_t st = buf * SM::STAGE;
            const u32x2_t lo = lds_ld_tr16(off + st + SM::Q_BYTES), hi = lds_ld_tr16(off_hi + st + SM::Q_BYTES);
            const u32x2_t lo2 = lds_ld_tr16(off + st), hi2 = lds_ld_tr16(off_hi + st);
            a1[slot] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            a2[slot] = u32x4_t{lo2[0], lo2[1], hi2[0], hi2[1]};
        };
        auto gemm2 = [&](auto idx0_c, auto idx1_c) {
            constexpr int idx0 = decltype(idx0_c)::value, idx1 = decltype(idx1_c)::value;
#pragma unroll
            for (int idx = idx0; idx < idx1; idx++) {
                if (idx + 1 < NP) tr_frag(idx + 1, (idx + 1) & 1);
                const int qb = idx / DB, db = idx % DB;
                const u32x4_t pb = {ppk[4 * qb], ppk[4 * qb + 1], ppk[4 * qb + 2], ppk[4 * qb + 3]};
                const u32x4_t sb = {dpk[4 * qb], dpk[4 * qb + 1], dpk[4 * qb + 2], dpk[4 * qb + 3]};
                dv[db] = E::mfma(a1[idx & 1], pb, dv[db]);
                dk[db] = E::mfma(a2[idx & 1], sb, dk[db]);
                if constexpr (!DMA) {
#pragma unroll
                    for (int n = idx * 2 * Q_IT / NP; n < (idx + 1) * 2 * Q_IT / NP; n++) load_item(n);
                }
            }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        // (after the last steps an existing tile is fetched again and dropped)
        if constexpr (!DMA) load_step(step + 2 < n_steps ? step + 2 : step, false);
        if constexpr (MB == 1) {
            // the MFMAs of the first 16 rows need the probabilities of those rows only: the softmax of the other 16
            // rows is issued between them
            soft_a(I0(), I0()); soft_m(I0(), I0()); soft_b(I0(), I0());
            tr_frag(0, 0);
            gemm2(I0(), std::integral_constant<int, DB / 2>());
            soft_a(I0(), I1());
            soft_m(I0(), I1());
            gemm2(std::integral_constant<int, DB / 2>(), std::integral_constant<int, DB>());
            soft_b(I0(), I1());
            gemm2(std::integral_constant<int, DB>(), std::integral_constant<int, NP>());
        } else {
            static_assert(MB <= 2, "steps of 32 or 64 query rows");
            soft_a(I0(), I0()); soft_m(I0(), I0()); soft_b(I0(), I0());
            soft_a(I0(), I1()); soft_m(I0(), I1()); soft_b(I0(), I1());
            soft_a(I1(), I0()); soft_m(I1(), I0()); soft_b(I1(), I0());
            soft_a(I1(), I1()); soft_m(I1(), I1()); soft_b(I1(), I1());
            tr_frag(0, 0);
            gemm2(I0(), std::integral_constant<int, NP>());
            // pin the order: reads of pair idx+1, then the two MFMAs of pair idx
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int idx = 0; idx < NP; idx++) {
                if (idx + 1 < NP) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            }
        }
        colsum += part;

        // ---- dBias column sum: flush when the bias head changes
        if (has_bias) {
            // (a part: its own last step too; one sum for all its heads where they share the bias)
            const bool part_end = !CMP && slot >= 0 && step == n_steps - 1;
            if ((mi == s_lo && ((CMP && slot >= 0) || f.Hb == f.H || (gi == G - 1 && slot < 0))) || part_end) {
                const float tot = xhalf_sum(colsum);
                const int hb = f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk);
                if (slot >= 0) {  // per-head partial column sums; the reduce kernel folds them
                    if (g == 0) p.db_part[((int64_t)slot * G + (CMP || f.Hb == f.H ? gi - g_lo : 0)) * KV_BN + (key - n0)] = tot;
                } else if (g == 0 && key < Lk) {
                    if (use_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + okey, tot);
                    else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + okey] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
                }
                colsum = 0.f;
            }
        }

        if constexpr (DMA) {
            if (head_next) cconst = column_const_value();
            dma_advance(step + 2 < n_steps);
            if (cur_mi == s_lo) { cur_mi = s_hi - 1; cur_gi++; } else cur_mi--;
        } else {
            cconst = cconst_next;
        }
        publish();
    };
    if constexpr (DMA && CMP) {
        // A wave behind the last kept key fetches its share of the tiles and leaves the products to the others.  Forward + backward, d = 128, us:
        // 2 x 16000 x 16/4 heads, 400 kept, not causal 677 / 651, 2 x 19776 x 8/2, 96 kept 244 / 237, 4 x 8192 x 16/8, 170 kept 445 / 438; where no
        // wave is without, 2048 kept of 8192 x 32/8, 706 / 704.  (At head dims up to 64 it costs more scalar registers than it gives: 12000 x 32/8,
        // 300 kept 206 / 213; ragged calls, with few such blocks, the same either way.)
        if (n0 + wave * 32 >= Lk) {
            for (int step = 0; step < n_steps; step++) {
                dma_begin(~step & 1);
#pragma unroll
                for (int n = 0; n <= 2 * Q_IT; n++) dma_piece(n);
                dma_advance(step + 2 < n_steps);
                publish();
            }
            return;
        }
    }
    for (int step = 0; step < n_steps; step += 2) {
        one_step(std::integral_constant<int, 0>(), step);
        if (step + 1 < n_steps) one_step(std::integral_constant<int, 1>(), step + 1);
    }

    // a key block that no query can see still owns its dbias column
    if (has_bias && n_steps == 0 && slot >= 0 && g == 0) {
        for (int gl = 0; gl < g_hi - g_lo; gl++) p.db_part[((int64_t)slot * G + gl) * KV_BN + (key - n0)] = 0.f;
    }
    if (has_bias && n_steps == 0 && slot < 0 && !use_accum && g == 0 && key < Lk) {
        const int ngh = (f.Hb == f.H) ? G : 1;
        for (int gh = 0; gh < ngh; gh++) {
            const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
            ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + okey] = 0;
        }
    }

    // ---- a part: fp32 sums in the order the lanes hold them (1 KB per store); heads without a step in it have zero columns
    if (!CMP && slot >= 0) {
        if (has_bias && f.Hb == f.H && g == 0) {
            const int g_end = (first_step + part_steps - 1) / n_m;
            for (int gh = 0; gh < G; gh++)
                if (gh < gi0 || gh > g_end) p.db_part[((int64_t)slot * G + gh) * KV_BN + (key - n0)] = 0.f;
        }
        f32x4_t *dst = (f32x4_t *)p.dkv_part + (int64_t)slot * (2 * KV_BN * D / 4) + wave * (D / 32) * 4 * 64 + lane;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int at = (db * 4 + q) * 64;
                dst[at] = f32x4_t{dk[db][4 * q], dk[db][4 * q + 1], dk[db][4 * q + 2], dk[db][4 * q + 3]};
                dst[at + KV_BN * D / 4] = f32x4_t{dv[db][4 * q], dv[db][4 * q + 1], dv[db][4 * q + 2], dv[db][4 * q + 3]};
            }
        return;
    }
    // ---- shared block: fp32 partial dK^T / dV^T, [which][d][key] so that a wave writes 128-byte runs
    if (CMP && slot >= 0) {
        float *pk = p.dkv_part + (int64_t)slot * 2 * D * KV_BN + (key - n0);
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int dcol = 32 * db + 16 * (i >> 3) + 8 * g + (i & 7);
                pk[dcol * KV_BN] = dk[db][i];
                pk[(D + dcol) * KV_BN] = dv[db][i];
            }
        return;
    }

    // ---- store dK (scaled) and dV
    if (key < Lk) {
        uint16_t *dkp = (uint16_t *)p.dk + b * p.dk_b + (sq.k0 + okey) * p.dk_r + hk * p.dk_h;
        uint16_t *dvp = (uint16_t *)p.dv + b * p.dv_b + (sq.k0 + okey) * p.dv_r + hk * p.dv_h;
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

// Sums of the parts on the original key axis, in part order, to dK (scaled), dV and dBias.  Thread (matrix, wave, d block, half,
// lane) of a unit owns the eight head-dim elements that lane held in its register block; a workgroup takes every gridDim-th piece
// of 256 such threads.
template <typename T, int D>
__global__ void __launch_bounds__(NTHREADS) bwd_dkdv_parts_sum_kernel(const BwdParams p) {
    using E = Elem<T>;
    constexpr int DB = D / 32, PER = KV_BN * D, BPU = 2 * PER / 8 / NTHREADS;  // floats of one matrix of a part, pieces per unit
    const FwdParams &f = p.f;
    const int G = f.H / f.Hk, bm = KvcSmem<D>::BM;
    const int n_nb = (f.Lk + KV_BN - 1) / KV_BN;
    const int units = (f.cu_q ? 1 : f.B) * f.Hk * p.kv_units;
    const int quota = p.kv_quota ? p.kv_quota : ragged_part_quota(f, bm);
    for (int item = (int)blockIdx.x; item < units * BPU; item += (int)gridDim.x) {
        const int unit = item / BPU, piece = item % BPU;
        int n_block = unit % p.kv_units, hk = unit / p.kv_units, b = 0;
        if (f.cu_q) {
            const RaggedUnit ru = ragged_unit(f, n_block);
            b = ru.entry;
            n_block = ru.block;
        } else {
            b = hk / f.Hk;
            hk = hk % f.Hk;
        }
        const SeqInfo sq = seq_info(f, b);
        const int n0 = n_block * KV_BN;
        if (n_block < 0 || n_block >= n_nb || n0 >= sq.Lk) continue;
        const int n = kv_parts_of(G * kv_unit_steps(sq.Lq, sq.Lk, f.causal, n0, bm), quota, p.kv_most);
        if (n == 1) continue;  // (the dK/dV kernel wrote the results itself)
        const int slot = kv_unit_slot(p, b, hk, n_block);
        const int t = piece * NTHREADS + threadIdx.x;
        const int lane = t & 63, w = t >> 6;  // w = ((mat * 4 + wave) * DB + db) * 2 + blk
        const int blk = w & 1, db = (w >> 1) % DB, kw = (w >> 1) / DB % 4, mat = (w >> 1) / DB / 4;
        const float *src = p.dkv_part + (int64_t)slot * 2 * PER + mat * PER + (((kw * DB + db) * 4 + 2 * blk) * 64 + lane) * 4;
        const int key = n0 + kw * 32 + (lane & 31), c = 32 * db + 16 * blk + 8 * (lane >> 5);
        f32x4_t a0 = {0, 0, 0, 0}, a1 = {0, 0, 0, 0};
#pragma unroll 4
        for (int i = 0; i < (c < f.d ? n : 0); i++) {  // (columns beyond d need not have been written)
            const float *q = src + (int64_t)i * 2 * PER;
            a0 += *(const f32x4_t *)q;
            a1 += *(const f32x4_t *)(q + 256);
        }
        if (key < sq.Lk && c < f.d) {
            const float m = mat == 0 ? f.scale : 1.f;
            const u32x4_t o = {E::pack2(a0[0] * m, a0[1] * m), E::pack2(a0[2] * m, a0[3] * m), E::pack2(a1[0] * m, a1[1] * m), E::pack2(a1[2] * m, a1[3] * m)};
            uint16_t *dst = mat == 0 ? (uint16_t *)p.dk + b * p.dk_b + (sq.k0 + key) * p.dk_r + hk * p.dk_h
                                     : (uint16_t *)p.dv + b * p.dv_b + (sq.k0 + key) * p.dv_r + hk * p.dv_h;
            *(u32x4_t *)(dst + c) = o;
        }
        // columns of dBias: two query heads per piece where every head has its own, else one sum for all
        const int ngh = f.Hb == f.H ? G : 1, kk = (int)threadIdx.x & (KV_BN - 1), half = (int)threadIdx.x / KV_BN;
        if (f.bias && n0 + kk < sq.Lk) {
            for (int gh = 2 * piece + half; gh < ngh; gh += 2 * BPU) {
                const float *cp = p.db_part + ((int64_t)slot * G + gh) * KV_BN + kk;
                float tot = 0.f;
#pragma unroll 4
                for (int i = 0; i < n; i++) tot += cp[(int64_t)i * G * KV_BN];
                const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
                if (p.dbias_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + n0 + kk, tot);
                else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + n0 + kk] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
            }
        }
    }
}

template <typename T, int D, bool CAUSAL, bool CMP>
hipError_t launch_dkdv_grid(const BwdParams &p, int grid, hipStream_t stream) {
    if constexpr (D > 128) {
        return launch_bwd_dkdv_256(p, std::is_same<T, bf16_tag>::value ? 0 : 1, grid, stream);
    } else {
        constexpr int LESS = D == 128 ? 96 : D;
        const bool less = p.f.d <= LESS;
        auto kern = less ? bwd_dkdv_colmask_kernel<T, D, LESS, CAUSAL, CMP> : bwd_dkdv_colmask_kernel<T, D, D, CAUSAL, CMP>;
        const int smem = KvcSmem<D>::TOTAL;
        static DynSmemLimit smem_limit[2];  // one per instantiation
        hipError_t e = smem_limit[less].ensure((const void *)kern, (int)smem);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(NTHREADS), smem, stream, p);
        return hipGetLastError();
    }
}
template <typename T, int D, bool CAUSAL, bool CMP>
hipError_t launch_dkdv_c(const BwdParams &p, hipStream_t stream) {
    const FwdParams &f = p.f;
    if (CMP) {
        int grid, slots;
        dkdv_split_bounds(f.B * f.Hk, (f.Lk + KV_BN - 1) / KV_BN, f.H / f.Hk, grid, slots);
        return launch_dkdv_grid<T, D, CAUSAL, CMP>(p, grid, stream);  // (the partial results are summed by workgroups of the dQ launch)
    }
    const int n_nb = (f.Lk + KV_BN - 1) / KV_BN;
    const bool turns = RAGGED_TURNS<D> && f.cu_q;  // (a kv head's units are numbered over all entries)
    const int grid = turns ? xcd_grid(f.Hk, ragged_lists_per_pair(f), p.kv_units, p.kv_most) : xcd_grid(f.B * f.Hk, xcd_lists_per_pair(f.B * f.Hk), n_nb, p.kv_most);
    const hipError_t e = launch_dkdv_grid<T, D, CAUSAL, CMP>(p, grid, stream);
    if (e != hipSuccess || p.kv_most <= 1) return e;
    const int64_t pieces = (int64_t)(f.cu_q ? 1 : f.B) * f.Hk * p.kv_units * (2 * KV_BN * D / 8 / NTHREADS);
    hipLaunchKernelGGL((bwd_dkdv_parts_sum_kernel<T, D>), dim3((unsigned)(pieces < 2048 ? pieces : 2048)), dim3(NTHREADS), 0, stream, p);
    return hipGetLastError();
}
template <typename T, int D, bool CAUSAL>
hipError_t launch_dkdv(const BwdParams &p, hipStream_t stream) {
    return p.f.cmp.on ? launch_dkdv_c<T, D, CAUSAL, true>(p, stream) : launch_dkdv_c<T, D, CAUSAL, false>(p, stream);
}


// ------------------------------------------------------------------------------------------------
// dQ
// ------------------------------------------------------------------------------------------------
constexpr int Q_BM = 128;
constexpr int DQ_MAX_KEYS = 1 << 20;  // keys that the tile bitmap holds


template <int D, int BN> struct DqcSmem {
    static constexpr int S = LdsTile<D>::S;
    static constexpr int K_BYTES = BN * S * 2;
    static constexpr int NST = LdsTile<D>::SWZ ? 3 : 2;  // K / V stages: three where the tiles are fetched two ahead
    static constexpr int OFF_K = 0;
    static constexpr int OFF_V = OFF_K + NST * K_BYTES;
    static constexpr int OFF_BIAS = OFF_V + NST * K_BYTES;
    static constexpr int OFF_BITS = OFF_BIAS + 3 * 256;  // three bias columns (a direct load fills 256 bytes)
    static constexpr int TOTAL = OFF_BITS + DQ_MAX_KEYS / BN / 8;
    static constexpr int GROUP = (TOTAL + 255) / 256 * 256;  // of a key group
    static_assert(TOTAL >= RED_LDS, "the workgroups that sum parts use it");
};

// BARE: no compaction, no mask, no bias (ragged batches, plain attention): there is no bias column, and the K / V tiles can
// go the direct way as with compacted keys (a column made from mask bytes and bias values would have to come through
// registers, whose wait is a wait for every direct load in front of it).
// KG: key groups of four waves.  Two take the tiles in turn, each with LDS and barriers' worth of stages of its own, and add their sums
// up through LDS at the end: half the chain of tiles for grids that leave CUs empty (see dq_key_groups).
template <typename T, int D, int DC, int BN, bool CAUSAL, bool CMP, bool BARE, int KG>
__device__ __forceinline__ void dq_colmask(const BwdParams &p) {
    using E = Elem<T>;
    using SM = DqcSmem<D, BN>;
    using TL = LdsTile<D>;
    constexpr int KS = DC / 16;
    constexpr int DB = DC / 32;
    constexpr int MB = BN / 32;
    constexpr int KB = BN / 16;
    constexpr int CH = D / 8, RPP = NTHREADS / CH, K_IT = BN / RPP;
    // DMA (rows of exactly 256 bytes): the K / V tiles and, with compacted keys, the fused bias column go from global memory
    // straight into LDS (global_load_lds: a wave writes 64 consecutive 16-byte or 4-byte pieces, so the swizzle of the
    // tile is applied to the GLOBAL address of each lane's piece), TWO tiles ahead, into a third stage: no staging
    // registers, no LDS stores, and a tile has a whole tile time more to arrive.  (Through registers, loaded between the
    // MFMAs of the tile whose end stores them, the stores waited for the loads: without the loads the kernel was 12 %
    // shorter.)  The instruction is written in assembly: issued through the compiler's builtin, every later LDS read
    // waited for ALL direct loads in flight -- the compiler cannot tell which stage they fill -- and the loads of
    // the tile after the next one would be waited for at once.  The waits are placed by hand (publish()).
    static_assert(!(CMP && BARE), "compacted keys have a column");
    constexpr bool DMA = TL::SWZ && (CMP || BARE), DMA_COL = DMA && CMP;
    constexpr int SLOT = DMA ? 256 : 4 * BN;  // bytes of a bias column's slot
    constexpr int NST = SM::NST;
    static_assert(!DMA || (RPP == 16 && NTHREADS == 256), "the direct loads are laid out for 16 chunks per row and four waves");

    // (LDS is read and written by absolute address in the tile loop: an access through a pointer into `smem` makes the
    // compiler wait for every direct load in flight first)
    extern __shared__ __attribute__((aligned(256))) char smem_all[];
    const int kgrp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NTHREADS);  // key group of this wave
    char *const smem = smem_all + kgrp * SM::GROUP;
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)
    uint32_t *sBits = (uint32_t *)(smem + SM::OFF_BITS);

    const FwdParams &f = p.f;
    const int tid = KG == 1 ? threadIdx.x : threadIdx.x % NTHREADS, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    int lid = blockIdx.x;  // index among the dQ workgroups
    if (CMP) {
        // some workgroups sum partial results of the dK/dV kernel instead
        const int at = lid - p.red_first;
        if (at >= 0 && at < p.red_count) {
            dkdv_reduce_blocks<T, D>(kernel_args_apart<BwdParams>(), at, p.red_count, threadIdx.x, (float *)smem);
            return;
        }
        if (at >= 0) lid -= p.red_count;
    }
    const RowUnit ru = row_unit(f, lid, Q_BM);  // (heaviest first under causal)
    if (ru.block < 0) return;
    const int b = ru.b, hk = ru.hk, h = ru.h;
    const int m0 = ru.block * Q_BM;
    const SeqInfo sq = seq_info(f, b);  // this batch entry's lengths and first rows (ragged batch: from cu_seqlens)
    const int LqS = sq.Lq, LkS = sq.Lk;
    if (m0 >= LqS) return;
    const int qrow = m0 + wave * 32 + r;
    const int qrow_c = qrow < LqS ? qrow : LqS - 1;

    // ---- Q and dO fragments (B operands), O and the row statistics: requested first of all, raw, from places that exist (rows
    // beyond Lq: the last one, chunks beyond d: the first), and looked at when the first tiles are on their way.  One trip to memory
    // for the counts above the rows, one for all of this and one for the tiles were six behind one another.
    u32x4_t qf[KS], dof[KS], of[CMP ? 1 : KS];
    {
        const uint16_t *qp = (const uint16_t *)f.q + b * f.q_b + (sq.q0 + qrow_c) * f.q_r + h * f.q_h;
        const uint16_t *dp = (const uint16_t *)p.dout + b * p.do_b + (sq.q0 + qrow_c) * p.do_r + h * p.do_h;
        const uint16_t *op = (const uint16_t *)f.o + b * f.o_b + (sq.q0 + qrow_c) * f.o_r + h * f.o_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8 < f.d ? ks * 16 + g * 8 : 0;
            qf[ks] = *(const u32x4_t *)(qp + c);
            dof[ks] = *(const u32x4_t *)(dp + c);
            if constexpr (!CMP) of[ks] = *(const u32x4_t *)(op + c);
        }
    }
    const float lse_raw = f.lse[b * f.lse_b + h * f.lse_h + sq.q0 + qrow_c];
    const float dd_raw = CMP ? p.softmax_d[b * p.sd_b + h * p.sd_h + sq.q0 + qrow_c] : 0.f;

    const int hm = f.mask ? (f.Hm == f.H ? h : (f.Hm == 1 ? 0 : hk)) : 0;
    const int hb = f.bias ? (f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk)) : 0;
    const uint8_t *mrow = f.mask ? f.mask + b * f.m_b + hm * f.m_h : nullptr;
    const uint16_t *brow = f.bias ? (const uint16_t *)f.bias + b * f.bi_b + hb * f.bi_h : nullptr;
    const uint16_t *kbase = (const uint16_t *)f.k + b * f.k_b + sq.k0 * f.k_r + hk * f.k_h;
    const uint16_t *vbase = (const uint16_t *)f.v + b * f.v_b + sq.k0 * f.v_r + hk * f.v_h;

    // key columns this workgroup iterates over (the compacted list with CMP), and how many a row may see
    const int Lk = CMP ? f.cmp.count[ru.pair] : LkS;
    const int32_t *ccnt = CMP ? f.cmp.cnt + (int64_t)ru.pair * f.cmp.ld : nullptr;
    const float *fbrow = CMP ? f.cmp.fb + (int64_t)(b * f.cmp.Hfb + (f.cmp.Hfb == f.H ? h : hk)) * f.cmp.ld : nullptr;
    const int vis_lane = CAUSAL ? visible_columns<CMP>(qrow, LqS, LkS, ccnt) : 0;  // columns below it pass the causal test for this lane's row
    const int vis_wave = CAUSAL ? visible_columns<CMP>(m0 + wave * 32, LqS, LkS, ccnt) : 0;
    const int vis_block = CAUSAL ? visible_columns<CMP>(m0 + Q_BM - 1, LqS, LkS, ccnt) : 0;

    int n_end = (Lk + BN - 1) / BN;
    if (CAUSAL) {
        const int ne = ((vis_block < 0 ? 0 : vis_block) + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }

    // ---- active-tile bitmap (tiles with at least one kept key)
    for (int base = 0; !CMP && !BARE && base < n_end; base += NTHREADS) {
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
    if (!CMP && !BARE) __syncthreads();
    auto next_active = [&](int j) -> int {  // wave-uniform: keeps tile bases and loop conditions scalar
        if (CMP || BARE) return j < n_end ? j : n_end;
        while (j < n_end) {
            const uint32_t w = __builtin_amdgcn_readfirstlane(lds_ld32(lds0 + SM::OFF_BITS + 4 * (j >> 5))) >> (j & 31);
            if (w) {
                j += __builtin_ctz(w);
                return j < n_end ? j : n_end;
            }
            j = (j | 31) + 1;
        }
        return n_end;
    };

    f32x16_t dq[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dq[db][i] = 0.f;

    // ---- staging: rows beyond Lk are clamped (their fused bias is -inf), head-dim chunks beyond d re-read chunk 0
    const int kc = tid % CH, kr0 = tid / CH;
    // (DMA: the lane fills chunk POSITION kc of its row, which holds chunk kc ^ swz(row) of the global row; rows 16
    // apart have the same swizzle)
    const int kc_g = DMA ? (kc ^ (int)TL::swz(kr0)) : kc;
    const int kcol = (kc_g * 8 < f.d) ? kc_g * 8 : 0;
    u32x4_t kreg[DMA ? 1 : K_IT], vreg[DMA ? 1 : K_IT];
    // Byte offsets of this thread's loads inside a tile are loop invariants -- one set for full tiles, one for the
    // (only) partial tile at the end of the keys -- so a load is one instruction with a scalar tile base, and the
    // loads of the next tile can be issued one by one between the MFMAs of the current one.  The bias / mask of the
    // thread's column travel as raw, unconditional loads (an absent one is the first element of K, ignored) and are looked
    // at when they are stored.
    const int j_last = Lk > 0 ? (Lk - 1) / BN : 0, last_row = Lk > 0 ? (Lk - 1) % BN : 0;
    uint32_t koff[K_IT], koff_l[K_IT], voff[K_IT], voff_l[K_IT];
#pragma unroll
    for (int it = 0; it < K_IT; it++) {
        const int row = kr0 + it * RPP, row_c = row < last_row ? row : last_row;
        koff[it] = (uint32_t)(row * f.k_r + kcol) * 2;
        koff_l[it] = (uint32_t)(row_c * f.k_r + kcol) * 2;
        voff[it] = (uint32_t)(row * f.v_r + kcol) * 2;
        voff_l[it] = (uint32_t)(row_c * f.v_r + kcol) * 2;
    }
    gptr_t tb_k = nullptr, tb_v = nullptr;
    bool t_last = false, bcol_ok = false;
    uint32_t braw = 0, mraw = 0;
    const uint8_t *mrow_ld = mrow ? mrow : (const uint8_t *)kbase;
    const uint16_t *brow_ld = brow ? brow : kbase;
    gptr_t tb_b = nullptr;  // DMA: the fused bias row, and this lane's offset in it for the tile being fetched
    uint32_t boff = 0;
    // bases of the tile whose K / V are fetched next; the bias / mask column of tile jb
    auto set_tile = [&](int j, int jb) {
        tb_k = uniform_ptr(kbase + (int64_t)j * BN * f.k_r);
        tb_v = uniform_ptr(vbase + (int64_t)j * BN * f.v_r);
        t_last = j == j_last;
        if constexpr (DMA_COL) {
            // columns beyond the end of the kept keys read the last one (masked where the column is used)
            tb_b = uniform_ptr(fbrow);
            const int col = j * BN + (lane & 31);
            boff = (uint32_t)(col < Lk ? col : Lk - 1) * 4u;
        }
        if (!DMA && tid < BN) {
            j = jb;
            const int col = j * BN + tid;
            bcol_ok = col < Lk;
            const int cc = bcol_ok ? col : 0;
            if (CMP) {
                braw = __float_as_uint(fbrow[cc]);
            } else {
                mraw = mrow_ld[mrow ? cc : 0];
                braw = brow_ld[brow ? cc : 0];
            }
        }
    };
    // one direct load: 64 lanes x 16 (or 4) bytes from `base` (wave-uniform) + this lane's offset to LDS address `dst`
    // (wave-uniform) onwards, lane after lane.  (m0 carries the LDS address; it is a reserved register that nothing
    // else in this kernel uses, and it is written immediately in front of every use.)
    auto dma16 = [](gptr_t base, uint32_t off, uint32_t dst) {
        load_lds16(off, base, dst);
    };
    auto dma4 = [](gptr_t base, uint32_t off, uint32_t dst) {
        load_lds4(off, base, dst);
    };
    constexpr int N_DMA = 2 * K_IT + (DMA_COL ? 1 : 0);  // direct loads of a wave per tile
    int dma_stage = 0;                   // stage the tile being fetched goes to (DMA)
    auto load_item = [&](int n) {  // 0 .. K_IT-1: K rows, K_IT .. 2*K_IT-1: V rows, 2*K_IT: the bias column (DMA)
        if constexpr (DMA) {
            // this wave's piece `it` of a tile: LDS bytes [1024 (wave + 4 it), + 1024), rows 4 wave + 16 it .. + 3
            const uint32_t st0 = lds0 + (uint32_t)(dma_stage * SM::K_BYTES);
            if (n < K_IT) dma16(tb_k, t_last ? koff_l[n] : koff[n], __builtin_amdgcn_readfirstlane(st0 + SM::OFF_K + (wave + 4 * n) * 1024));
            else if (n < 2 * K_IT)
                dma16(tb_v, t_last ? voff_l[n - K_IT] : voff[n - K_IT], __builtin_amdgcn_readfirstlane(st0 + SM::OFF_V + (wave + 4 * (n - K_IT)) * 1024));
            else  // (every wave fetches the same 256 bytes -- lanes 32-63 repeat lanes 0-31 -- : no branch between the MFMAs)
                dma4(tb_b, boff, __builtin_amdgcn_readfirstlane(lds0 + SM::OFF_BIAS + dma_stage * 256));
        } else {
            if (n < K_IT) kreg[n] = *(const __attribute__((address_space(1))) u32x4_t *)(tb_k + (t_last ? koff_l[n] : koff[n]));
            else if (n < 2 * K_IT) vreg[n - K_IT] = *(const __attribute__((address_space(1))) u32x4_t *)(tb_v + (t_last ? voff_l[n - K_IT] : voff[n - K_IT]));
        }
    };
    auto load_tile = [&](int j, int jb) {
        set_tile(j, jb);
#pragma unroll
        for (int n = 0; n < (DMA ? N_DMA : 2 * K_IT); n++) load_item(n);
    };
    // registers -> LDS stage `buf` (not with DMA), and the fused bias column of that tile into slot `slot`
    auto store_tile = [&](int buf, int slot) {
        if constexpr (!DMA) {
            char *sK = smem + SM::OFF_K + buf * SM::K_BYTES;
            char *sV = smem + SM::OFF_V + buf * SM::K_BYTES;
#pragma unroll
            for (int it = 0; it < K_IT; it++) {
                const uint32_t off = TL::chunk(kr0 + it * RPP, kc);
                *(u32x4_t *)(sK + off) = kreg[it];
                *(u32x4_t *)(sV + off) = vreg[it];
            }
        }
        if (!DMA && tid < BN) {
            float v = -INFINITY;
            if (CMP) {
                if (bcol_ok) v = __uint_as_float(braw);
            } else if (bcol_ok && (!mrow || mraw)) {
                v = brow ? E::lo(braw) * kLog2e : 0.f;
            }
            lds_st32(lds0 + SM::OFF_BIAS + slot * SLOT + 4 * tid, __float_as_uint(v));
        }
    };

    const int a_row = pi_row(r);
    const uint32_t a_off = lds0 + SM::OFF_K + TL::frag_base(a_row, g);  // (absolute, stage 0 of K)
    const TrLane tr = tr_lane(lane);
    const uint32_t tr_off = lds0 + SM::OFF_K + TL::tr_base(g, tr);

    // A wave waits for its own pieces of the next tile, then the barrier publishes everybody's (DMA: by hand -- the
    // N_DMA loads of the tile after that, issued later, stay in flight; vmcnt in bits 3:0, lgkmcnt 0, expcnt not
    // waited for)
    auto publish = [&]() {
        if constexpr (DMA) {
            __builtin_amdgcn_s_waitcnt(0x0070 | N_DMA);
            __builtin_amdgcn_s_barrier();
        } else {
            __syncthreads();
        }
    };
    // The tiles in turns of KG, one for each group.  jc, jn, jnn: the group's own of this turn and the two behind it; the leads: the first
    // group's, which end the loop alike for all; tail: the newest turn's last
    int lead = 0, lead_n = n_end, lead_nn = n_end, tail = -1;
    auto next_turn = [&](int &first) -> int {
        first = next_active(tail + 1);
        tail = KG == 1 ? first : next_active(first + 1);
        return KG == 2 && kgrp ? tail : first;
    };
    int jc = next_turn(lead), jn = n_end, jnn = n_end;
    // (what was requested above has landed by now; waited for here, the tiles' own loads are not waited for with it)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(qf[ks]), "+v"(dof[ks]));
    jn = next_turn(lead_n);
    if constexpr (DMA) jnn = next_turn(lead_nn);
    if (jc < n_end) {
        load_tile(jc, jc);
        if constexpr (DMA) {  // the second tile is on its way before the first is looked at
            dma_stage = 1;
            load_tile(jn < n_end ? jn : jc, jc);
        }
    }
    const bool row_ok = qrow < LqS;
    const float lse2 = row_ok ? lse_raw * kLog2e : INFINITY;
    float dd = row_ok ? dd_raw : 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const bool ok = row_ok && ks * 16 + g * 8 < f.d;
        qf[ks] = scaled8<T>(qf[ks], f.scale_log2, ok);  // (Q only feeds the scores in this kernel: softmax_scale * log2(e) once)
        dof[ks] = kept8(dof[ks], ok);
    }
    if constexpr (!CMP) {
        // D = rowsum(dO * O) is made here, from the dO fragments, and left for the dK/dV kernel, which is launched behind
        // this one: a launch and a second read of dO less (52 us of 2.8 ms on 16384 ragged tokens x 32 heads).  (With
        // compacted keys this launch also sums that kernel's partial results and comes second; D is a layer of the pre-pass.)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {  // (dO is zero beyond d and beyond Lq)
#pragma unroll
            for (int e = 0; e < 4; e++) dd += E::lo(of[ks][e]) * E::lo(dof[ks][e]) + E::hi(of[ks][e]) * E::hi(dof[ks][e]);
        }
        dd = xhalf_sum(dd);
        if (!row_ok) dd = 0.f;
        // (fixed lengths: padded rows are zero)
        if (g == 0 && kgrp == 0 && (row_ok || (!f.cu_q && qrow < p.Lq_rounded))) p.softmax_d[b * p.sd_b + h * p.sd_h + sq.q0 + qrow] = dd;
    }
    if (lead < n_end) {
        if (KG == 1 || jc < n_end) store_tile(0, 0);
        publish();
    }
    int i = 0;
    constexpr bool S_EARLY = DMA && MB == 1;
    f32x16_t s[MB];
    auto one_tile = [&]() {
        const int n0 = jc * BN;
        const int st = DMA ? i % 3 : (i & 1);
        const uint32_t st_off = (uint32_t)(st * SM::K_BYTES);  // (a multiple of 256: the swizzles stay XORs)
        const uint32_t a_cur = a_off + st_off, tr_cur = tr_off + st_off;
        const uint32_t bs = lds0 + SM::OFF_BIAS + (i % 3) * SLOT + 32 * g;

        // ---- S^T = K Q^T, dP^T = V dO^T, dS^T = P^T * (dP^T - D), dQ^T += K^T dS^T.  A wave issues in program
        // order, so the vector work has to sit BETWEEN the MFMAs to run under them; the tile is written slot by slot --
        // one MFMA, the fragment read of the MFMA FR slots later, a share of the vector work, a piece of the next tile's
        // loads -- with a scheduling barrier after every slot:
        //   slots of S (all k-steps), then slots of dP with the exp2 of the finished scores between them, then the dQ
        //   slots of one 16-key block with the dS arithmetic of the next block between them.
        // The score accumulators start from the fused bias vector minus the row's log-sum-exp and the dP accumulators
        // from minus D, so that the MFMAs deliver the exp2 argument and dP - D themselves.
        // (direct loads: every wave fetches the whole bias column of a tile itself, two tiles ahead, so a wave can read
        // the next tile's column as soon as its own load has landed; the score accumulators of the NEXT tile are set up
        // between the last dQ MFMAs of this one -- `s` is free from the last exp2 on -- instead of in front of the first
        // MFMA, where nothing covers the LDS reads and the 16 subtractions)
        f32x16_t dp[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                if (!S_EARLY || i == 0) {
                    const f32x4_t b0 = BARE ? f32x4_t{0.f, 0.f, 0.f, 0.f} : __builtin_bit_cast(f32x4_t, lds_ld128(bs + 4 * (32 * mb + 16 * blk)));
                    const f32x4_t b1 = BARE ? b0 : __builtin_bit_cast(f32x4_t, lds_ld128(bs + 4 * (32 * mb + 16 * blk + 4)));
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s[mb][8 * blk + e] = b0[e] - lse2;
                        s[mb][8 * blk + 4 + e] = b1[e] - lse2;
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; e++) dp[mb][8 * blk + e] = -dd;
                if (DMA && jc == j_last) {  // (the bias column came as it is in memory: columns beyond the kept keys)
                    const int lim = Lk - n0 - 32 * mb - 16 * blk - 8 * g;  // local columns e < lim exist
#pragma unroll
                    for (int e = 0; e < 8; e++) s[mb][8 * blk + e] = e < lim ? s[mb][8 * blk + e] : -INFINITY;
                }
            }
        // the next tile's bases and side inputs (after the last tile the current one is fetched again and dropped); behind
        // the accumulator set-up: the load of the bias / mask column must not be waited for with the LDS reads above
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (DMA) {  // K / V of the tile after the next one into the stage the last tile has left
            dma_stage = (i + 2) % 3;
            set_tile(jnn < n_end ? jnn : jc, jn < n_end ? jn : jc);
        } else {
            set_tile(jn < n_end ? jn : jc, jn < n_end ? jn : jc);
        }
        float pv[16 * MB];
        {
            constexpr int NH = MB * KS, NF = 2 * NH, FR = 3;
            u32x4_t a[NF];
            auto frag = [&](int fi) {  // S slots first (K tile), then dP slots (V tile); k-step major, row block minor
                const int which = fi / NH, mb = (fi % NH) % MB, ks = (fi % NH) / MB;
                return lds_ld128(TL::frag_at(a_cur, ks) + (uint32_t)(which * (SM::OFF_V - SM::OFF_K) + 32 * mb * TL::ROW_BYTES));
            };
#pragma unroll
            for (int fi = 0; fi < FR; fi++) a[fi] = frag(fi);
#pragma unroll
            for (int fi = 0; fi < NF; fi++) {
                if (fi + FR < NF) a[fi + FR] = frag(fi + FR);
                const int which = fi / NH, mb = (fi % NH) % MB, ks = (fi % NH) / MB;
                if (which) dp[mb] = E::mfma(a[fi], dof[ks], dp[mb]);
                else s[mb] = E::mfma(a[fi], qf[ks], s[mb]);
                constexpr int NLD = DMA ? N_DMA : 2 * K_IT;
#pragma unroll
                for (int n = fi * NLD / NF; n < (fi + 1) * NLD / NF; n++) load_item(n);
                if (which) {
#pragma unroll
                    for (int e = 0; e < 16 * MB; e++)
                        if (e * NH / (16 * MB) == fi - NH) pv[e] = fast_exp2(s[e / 16][e % 16]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const bool diag = CAUSAL && (n0 + BN > vis_wave);
        if (diag) {
            asm volatile("" ::: "memory");  // (keeps this a branch: as selects, every tile would pay for the diagonal ones)
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int blk = 0; blk < 2; blk++) {
                    const int lim = vis_lane - 1 - n0 - 32 * mb - 16 * blk - 8 * g;  // local columns e <= lim are visible
#pragma unroll
                    for (int e = 0; e < 8; e++) pv[16 * mb + 8 * blk + e] = e <= lim ? pv[16 * mb + 8 * blk + e] : 0.f;
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        uint32_t dpk[8 * MB];
        auto ds_piece = [&](int kb, int e) {  // two elements of 16-key block kb: dS = P * (dP - D), rounded to 16 bits
            const int mb = kb >> 1, blk = kb & 1;
            const float d0 = pv[16 * mb + 8 * blk + 2 * e] * dp[mb][8 * blk + 2 * e];
            const float d1 = pv[16 * mb + 8 * blk + 2 * e + 1] * dp[mb][8 * blk + 2 * e + 1];
            dpk[4 * kb + e] = E::pack2(d0, d1);
        };
        {
            // K^T through transposing LDS reads of the row-major K tile, two reads per MFMA, FR2 MFMAs ahead (the first
            // ones in front of the first block's dS arithmetic)
            constexpr int NG = KB * DB, FR2 = 2;
            u32x2_t tl[NG], th[NG];
            f32x4_t nb[4];  // (S_EARLY: the next tile's bias column, 16 keys of this lane's half)
            auto tr_read = [&](int gi) {
                const int kb = gi / DB, db = gi % DB;
                tl[gi] = lds_ld_tr16(TL::tr_at(tr_cur, kb, db, 0));
                th[gi] = lds_ld_tr16(TL::tr_at(tr_cur, kb, db, 1));
            };
#pragma unroll
            for (int gi = 0; gi < FR2; gi++) tr_read(gi);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; e++) ds_piece(0, e);
#pragma unroll
            for (int gi = 0; gi < NG; gi++) {
                if (gi + FR2 < NG) tr_read(gi + FR2);
                const int kb = gi / DB, db = gi % DB;
                const u32x4_t bop = {dpk[4 * kb], dpk[4 * kb + 1], dpk[4 * kb + 2], dpk[4 * kb + 3]};
                const u32x4_t av = {tl[gi][0], tl[gi][1], th[gi][0], th[gi][1]};
                dq[db] = E::mfma(av, bop, dq[db]);
                if (kb + 1 < KB) {  // the next block's dS, spread over this block's slots
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (e * DB / 4 == db) ds_piece(kb + 1, e);
                }
                if constexpr (S_EARLY) {
                    // the next tile's bias column (slot (i + 1) % 3, complete since the last barrier): read in the slots
                    // of the first key block, used in those of the last
                    const uint32_t bs_n = lds0 + SM::OFF_BIAS + (uint32_t)(((i + 1) % 3) * SLOT + 32 * g);
                    // (this wave's own copy of that column was fetched a tile ago, in front of the N_DMA loads of the
                    // tile after it: wait for it alone -- vmcnt N_DMA, no wait for LDS reads or exports)
                    if (DMA_COL && kb == 0 && db == 0) __builtin_amdgcn_s_waitcnt(0x0F70 | N_DMA);
#pragma unroll
                    for (int x = 0; x < 4; x++)  // (four pieces over the block's slots)
                        if (x * DB / 4 == db) {
                            if (DMA_COL && kb == 0) nb[x] = __builtin_bit_cast(f32x4_t, lds_ld128(bs_n + 16 * (x & 1) + 64 * (x >> 1)));
                            if (kb == KB - 1) {
#pragma unroll
                                for (int e = 0; e < 4; e++) s[0][4 * x + e] = DMA_COL ? nb[x][e] - lse2 : -lse2;
                            }
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!DMA && jn < n_end) store_tile((i + 1) & 1, (i + 1) % 3);
    };
    while (lead < n_end) {
        // (a group without a tile in the last turn only takes part in its barrier)
        if (KG == 1 || jc < n_end) one_tile();
        publish();
        i++;
        jc = jn;
        lead = lead_n;
        if constexpr (DMA) {
            jn = jnn;
            lead_n = lead_nn;
            jnn = next_turn(lead_nn);
        } else {
            jn = next_turn(lead_n);
        }
    }

    // (direct loads still in flight -- tiles fetched past the last one -- must not land in LDS that belongs to the next
    // workgroup by then)
    if constexpr (DMA) __builtin_amdgcn_s_waitcnt(0x0070);
    if constexpr (KG == 2) {  // each group hands the other's half of the head dim over and finishes its own
        __syncthreads();  // (every wave's reads of the last tiles, and its direct loads)
        static_assert(2 * 4 * DB * 2048 <= 2 * SM::GROUP, "the halves lie where the tiles were");
        // (eight head-dim elements, 2 db + blk, at a time: the first DB of them are group 0's)
        f32x4_t *theirs = (f32x4_t *)smem_all + ((1 - kgrp) * 4 + wave) * DB * 2 * 64 + lane, *mine = (f32x4_t *)smem_all + (kgrp * 4 + wave) * DB * 2 * 64 + lane;
#pragma unroll
        for (int u = 0; u < 2 * DB; u++)
            if (u / DB != kgrp) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int e = 8 * (u & 1) + 4 * q;
                    theirs[(u % DB * 2 + q) * 64] = f32x4_t{dq[u / 2][e], dq[u / 2][e + 1], dq[u / 2][e + 2], dq[u / 2][e + 3]};
                }
            }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2 * DB; u++)
            if (u / DB == kgrp) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const f32x4_t t = mine[(u % DB * 2 + q) * 64];
#pragma unroll
                    for (int e = 0; e < 4; e++) dq[u / 2][8 * (u & 1) + 4 * q + e] += t[e];
                }
            }
    }
    if (qrow < LqS) {
        uint16_t *dqp = (uint16_t *)p.dq + b * p.dq_b + (sq.q0 + qrow) * p.dq_r + h * p.dq_h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                if (KG == 2 && (2 * db + blk) / DB != kgrp) continue;
                const int c = 32 * db + 16 * blk + 8 * g;
                if (c < f.d) {
                    u32x4_t w;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        w[e] = E::pack2(dq[db][8 * blk + 2 * e] * f.scale, dq[db][8 * blk + 2 * e + 1] * f.scale);
                    *(u32x4_t *)(dqp + c) = w;
                }
            }
    }
}

template <typename T, int D, int BN, bool CAUSAL, bool CMP, bool BARE>
__global__ void __launch_bounds__(NTHREADS, 2) bwd_dq_colmask_kernel(const BwdParams p) {
    dq_colmask<T, D, D, BN, CAUSAL, CMP, BARE, 1>(p);
}
template <typename T, bool CAUSAL, bool CMP, bool BARE>
__global__ void __launch_bounds__(NTHREADS, 2) bwd_dq_96_kernel(const BwdParams p) {
    dq_colmask<T, 128, 96, 32, CAUSAL, CMP, BARE, 1>(p);
}
template <typename T, int D, int DC, int BN, bool CAUSAL, bool BARE>
__global__ void __launch_bounds__(2 * NTHREADS, 2) bwd_dq_groups_kernel(const BwdParams p) {
    dq_colmask<T, D, DC, BN, CAUSAL, false, BARE, 2>(p);
}

// Two key groups to a workgroup of dQ where there is no mask and no bias, the rows are long and there are no more workgroups than CUs
// hold at once: a SIMD works a tile off in 0.65 us with two waves, in 0.75 with one, and the hand-over at the end is 2 us.  dQ with one group / two,
// us: ragged 3520 and others (4443 tokens) x 2/1 heads, d = 128 73 / 63; 3392 (7028) x 2/1, d = 96 77 / 61; 4717 (5549) x 8/2, d = 64 90.5 / 71;
// 3904 (3914) x 16/4, d = 64, 528 blocks, 87 / 74; short rows 334 (632) x 8/2 14.5 / 16.4; more blocks (1984 of 2708 x 32/8, 896)
// 69 / 90.  Not with a mask, where one group's fixed part weighs as much as its few tiles (768 tokens x 16/8 32.2 / 31.6, 576 x 16/8 x 2
// 25.4 / 26.5), nor with compacted keys, of which the host does not know how many there are (1733 x 16/4, 130 kept 16.1 / 21.1).
bool dq_key_groups(const FwdParams &f) {
    if (f.d > 128 || f.cmp.on || f.mask || f.bias || f.Lk < 1024) return false;
    const int64_t blocks = f.cu_q ? (int64_t)f.H * (f.total_q / Q_BM + f.B) : (int64_t)f.B * f.H * ((f.Lq + Q_BM - 1) / Q_BM);
    return blocks <= 9 * (int64_t)device_cus() / 4;
}

template <typename T, int D, int DC, bool CAUSAL>
hipError_t launch_dq_dims(const BwdParams &p, int grid, hipStream_t stream) {
    const FwdParams &f = p.f;
    constexpr int BN = D > 64 ? 32 : 64;  // at d = 128 a 64-key tile would spill registers
    constexpr bool SWZ = LdsTile<D>::SWZ;
    const int which = f.cmp.on ? 1 : (SWZ && !f.mask && !f.bias ? 2 : 0);
    const bool two = dq_key_groups(f);
    auto kern = bwd_dq_groups_kernel<T, D, DC, BN, CAUSAL, SWZ>;
    if constexpr (DC == D) {
        if (!two) kern = which == 1 ? bwd_dq_colmask_kernel<T, D, BN, CAUSAL, true, false>
                                    : (which == 2 ? bwd_dq_colmask_kernel<T, D, BN, CAUSAL, false, SWZ> : bwd_dq_colmask_kernel<T, D, BN, CAUSAL, false, false>);
    } else {
        if (!two) kern = which == 1 ? bwd_dq_96_kernel<T, CAUSAL, true, false> : (which == 2 ? bwd_dq_96_kernel<T, CAUSAL, false, true> : bwd_dq_96_kernel<T, CAUSAL, false, false>);
    }
    const int smem = two ? 2 * DqcSmem<D, BN>::GROUP : DqcSmem<D, BN>::TOTAL;
    static DynSmemLimit smem_limit[4];  // one per instantiation: the limit is a property of the kernel
    hipError_t e = smem_limit[two ? 3 : which].ensure((const void *)kern, (int)smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(two ? 2 * NTHREADS : NTHREADS), smem, stream, p);
    return hipGetLastError();
}
template <typename T, int D, bool CAUSAL>
hipError_t launch_dq_grid(const BwdParams &p, int grid, hipStream_t stream) {
    if constexpr (D > 128) return launch_bwd_dq_256(p, std::is_same<T, bf16_tag>::value ? 0 : 1, grid, stream);
    else if constexpr (D == 128) return p.f.d <= 96 ? launch_dq_dims<T, D, 96, CAUSAL>(p, grid, stream) : launch_dq_dims<T, D, D, CAUSAL>(p, grid, stream);
    else return launch_dq_dims<T, D, D, CAUSAL>(p, grid, stream);
}
template <typename T, int D, bool CAUSAL>
hipError_t launch_dq(const BwdParams &p, hipStream_t stream) {
    const FwdParams &f = p.f;
    BwdParams pr = p;
    const int n_dq = row_grid(pr.f, Q_BM);  // a multiple of 8
    return launch_dq_grid<T, D, CAUSAL>(pr, n_dq + (f.cmp.on ? pr.red_count : 0), stream);
}

}  // namespace

// The dQ launch of a compacted backward carries the reduction of the dK/dV partials along: `red_count` consecutive workgroups
// (a multiple of 8) do that instead of dQ work.  They only move memory, so side by side with dQ workgroups, which keep the matrix
// units busy, they cost little; as a launch of its own the reduction took as long as its memory traffic.
// One to a CU, in front of all others: they are done early, and the dQ workgroups then start heaviest first as if they were
// alone.  Spread through the launch instead, one beside three dQ workgroups, they kept those from their CUs (half of the CUs' time
// was idle).  Spread / in front (us, the whole step): 4 x 2048 tokens, 16/8 heads, d = 64 with its layer 174 / 165; 8192 x 8/4, d = 64
// 117 / 104; d = 128: 8192 x 32/8 724 / 718, 2048 x 32/8 126 / 117, 4096 x 16/4 164 / 149, 2 x 4096 x 8/2 132 / 119, 12000 x 8/2 263 / 240;
// half as many 0.95 to 1.16 times that, twice as many the same.
// Above head dim 128 a CU holds one workgroup of the launch: a quarter of the CUs is left to the heaviest dQ workgroups from the
// start.  All CUs / three quarters / half of them summing, the dQ launch, d = 256 (us): 3001 x 8/4 73.0 / 60.6 / 59.4, 2048 x 16/8, 1000 kept
// 78.4 / 64.3 / 62.0, 1300 x 16/8 52.3 / 47.2 / 44.0, 5000 x 16/4 82.0 / 81.5 / 81.8, 2 x 2048 x 16/8, 1500 kept 170 / 168 / 180; not causal 1300 x
// 16/8 65.0 / 63.7 / 69.1, 3001 x 8/4 82.1 / 75.8 / 82.2.
// Few query rows against many keys are the other way round: few dQ workgroups, which leave CUs free, and partials by the number
// of keys.  All that the items ask for then follow the dQ workgroups.  100 rows of 16 heads over 2048 kept keys, d = 128 (16 dQ
// workgroups): the launch 361 us with 16 summing workgroups, 54 with 1024.  Up to half a dQ workgroup per CU, or one where the keys
// are more than twice the rows: behind / in front (us, the step) 1300 rows x 16/4 heads over 1500 kept of 4000, d = 128 133.5 / 135.4;
// 4096 x 8/2, all 4096 keys to choose from, 124 / 121 at d = 128, 98.6 / 96.1 at 64.
void place_reduction(BwdParams &p) {
    FwdParams f = p.f;
    const int n_dq = row_grid(f, Q_BM), items = f.B * f.Hk * ((f.Lk + KV_BN - 1) / KV_BN) * (f.d / 4 + (f.bias ? 1 : 0));
    const bool few = (f.Lk > 2 * f.Lq ? 1 : 2) * n_dq <= device_cus();
    const int most = few ? 1024 : (f.d > 128 ? device_cus() * 3 / 4 : device_cus());
    p.red_count = ((items < most ? items : most) + 7) / 8 * 8;
    p.red_first = few ? n_dq : 0;
    // (a CU holds two workgroups up to head dim 128, and the second round of those is where the difference is gone)
    const float more = (float)(n_dq - device_cus()) / (float)(2 * device_cus());
    p.red_wait = more <= 0.f ? 0.f : (f.d > 128 || more > 1.f ? 1.f : more);
}

bool bwd_colmask_applicable(const BwdParams &p) {
    const bool mask_ok = !p.f.mask || p.f.m_r == 0;
    const bool bias_ok = !p.f.bias || p.f.bi_r == 0;
    return mask_ok && bias_ok && p.f.Lk <= DQ_MAX_KEYS;
}

// Parts of the units on the original key axis.  A call has a workgroup per 128 keys of a kv head, whose steps -- query blocks
// times grouped heads -- follow each other: a call of few heads takes what its first block takes, 1.2 us a step (d = 128; two
// workgroups on a CU 2 us), with most of the chip idle.  A part costs its start and its sums, written and read again (128 KB
// at d = 128) and the call the launch that adds them up (5 us):
// steps per part grow with the square root of the call's steps.  Measured, dK/dV with its sums, whole / rule / best of 13 quotas (us):
//   d = 128: 1 x 672 x 16/4 heads 110 / 31.6 / 30.8, 1 x 563 x 8/2 96 / 25.5 / 24.2, 4 x 302 x 32/8 62 / 39 / 36, 1 x 1000 x 8/8 47 / 29.6 / 29.6,
//   not causal 1 x 400 x 32/8 68 / 32.6 / 32.4; ragged, d = 96: 9 entries up to 5397 x 8/2 742 / 288 / 280, 6 up to 4664 x 2/1 323 / 77 / 64;
//   d = 128, 4 x 2048 x 32/8 417 / 383 / 368; d = 64, 4096 x 32/8 414 / 225 / 218, 962 x 8/4 55 / 24.6 / 22.9.
// Whole where there are 2.5 units per CU (16384 ragged tokens x 32/8: 1175 whole, 1258 to 1286 in parts of 96 to 140 steps), and, from
// half a unit per CU on, where the longest is not two and a half parts (1 x 700 x 32/32: 36.5 whole, 39 to 42 cut; d = 64,
// 2 x 1000 x 16/16: 35.6 and 41 to 49).  Whole up to 20 steps: 25 us at most, and the call is bound by the host, to which a launch
// more is 2.5 us (256 x 2/1, d = 64, forward and backward: 72.8 whole, 75.5 cut).  At most 16 parts, and 2048 places for sums: up to 128 / 256 / 512 MB
// at d = 64 / 128 / 256, which callers offer where they have it.
size_t plan_kv_parts(BwdParams &p, size_t *db_bytes) {
    const FwdParams &f = p.f;
    p.kv_most = 1;
    p.kv_quota = 0;
    p.kv_units = f.cu_q ? f.total_k / KV_BN + f.B : (f.Lk + KV_BN - 1) / KV_BN;
    *db_bytes = 0;
    if (f.Lq <= 0 || f.Lk <= 0 || f.cmp.on) return 0;
    const int G = f.H / f.Hk, bm = kv_step_rows(f.d);
    const int64_t longest = (int64_t)G * kv_unit_steps(f.Lq, f.Lk, f.causal, 0, bm);
    const int64_t units = (int64_t)(f.cu_q ? 1 : f.B) * f.Hk * p.kv_units;
    int64_t total;
    if (f.cu_q) {  // (at least: the longest entry, and the other rows in entries of one length)
        const int rest = f.B > 1 ? f.B - 1 : 1, rq = (f.total_q - f.Lq) / rest, rk = (f.total_k - f.Lk) / rest;
        total = (kv_head_steps(f.Lq, f.Lk, f.causal, bm) + (f.B > 1 ? rest * kv_head_steps(rq, rk, f.causal, bm) : 0)) * f.H;
    } else {
        total = kv_head_steps(f.Lq, f.Lk, f.causal, bm) * f.H * f.B;
    }
    const int quota = kv_part_quota(total), cus = device_cus();
    int64_t most = kv_parts_of((int)(longest < (1 << 30) ? longest : 1 << 30), quota, 16);
    // Ragged, d = 65 .. 128: while the longest block runs, a CU's other units, two at a time, fill it with less than 60 steps each;
    // what parts save then is less than their sums.  Over 37 calls, whole / parts (us): 11 entries up to 1187 x 32/16 (2.4 units per CU, longest 76
    // steps) 222 / 242, five of 800 x 64/16 (2.3, 128) 411 / 430, 11 entries x 8/8 (1.2, 38) 123 / 130; on the other side 11 entries x 48/12 (1.8,
    // 152) 354 / 318, the same x 16/8 (1.2, 76) 177 / 157; worst kept five of 800 x 48/12 (1.7, 128) 339 / 351 and 4000, 3000, 700, 1 x 8/8 (2, 125) 375 / 390.  At d <= 64 parts lose nowhere.
    if (f.cu_q && f.d > 64 && f.d <= 128 && longest * cus < 60 * units) most = 1;
    if (longest <= 20 || units >= cus * 5 / 2 || (units >= cus / 2 && 2 * longest <= 5 * (int64_t)quota)) most = 1;
    if (most * units > 2048) most = 2048 / units;
    if (most <= 1) return 0;
    if (!f.cu_q) p.kv_quota = quota;
    p.kv_most = (int32_t)most;
    const int dpad = f.d <= 64 ? 64 : (f.d <= 128 ? 128 : 256);
    if (f.bias) *db_bytes = (size_t)units * most * G * KV_BN * sizeof(float);
    return (size_t)units * most * 2 * dpad * KV_BN * sizeof(float);
}

hipError_t launch_bwd_dkdv_colmask(const BwdParams &p, int dtype, hipStream_t stream) {
    // head dims up to 64 / 128 / 256 (a head dim in between runs in the next larger instantiation)
    const int dc = p.f.d <= 64 ? 0 : (p.f.d <= 128 ? 1 : 2);
    const bool c = p.f.causal != 0;
    if (dtype == 0) {
        if (dc == 0) return c ? launch_dkdv<bf16_tag, 64, true>(p, stream) : launch_dkdv<bf16_tag, 64, false>(p, stream);
        if (dc == 1) return c ? launch_dkdv<bf16_tag, 128, true>(p, stream) : launch_dkdv<bf16_tag, 128, false>(p, stream);
        return c ? launch_dkdv<bf16_tag, 256, true>(p, stream) : launch_dkdv<bf16_tag, 256, false>(p, stream);
    }
    if (dc == 0) return c ? launch_dkdv<fp16_tag, 64, true>(p, stream) : launch_dkdv<fp16_tag, 64, false>(p, stream);
    if (dc == 1) return c ? launch_dkdv<fp16_tag, 128, true>(p, stream) : launch_dkdv<fp16_tag, 128, false>(p, stream);
    return c ? launch_dkdv<fp16_tag, 256, true>(p, stream) : launch_dkdv<fp16_tag, 256, false>(p, stream);
}

}  // namespace fdma

namespace fdma {
hipError_t launch_bwd_dq_colmask(const BwdParams &p, int dtype, hipStream_t stream) {
    const int dc = p.f.d <= 64 ? 0 : (p.f.d <= 128 ? 1 : 2);
    const bool c = p.f.causal != 0;
    if (dtype == 0) {
        if (dc == 0) return c ? launch_dq<bf16_tag, 64, true>(p, stream) : launch_dq<bf16_tag, 64, false>(p, stream);
        if (dc == 1) return c ? launch_dq<bf16_tag, 128, true>(p, stream) : launch_dq<bf16_tag, 128, false>(p, stream);
        return c ? launch_dq<bf16_tag, 256, true>(p, stream) : launch_dq<bf16_tag, 256, false>(p, stream);
    }
    if (dc == 0) return c ? launch_dq<fp16_tag, 64, true>(p, stream) : launch_dq<fp16_tag, 64, false>(p, stream);
    if (dc == 1) return c ? launch_dq<fp16_tag, 128, true>(p, stream) : launch_dq<fp16_tag, 128, false>(p, stream);
    return c ? launch_dq<fp16_tag, 256, true>(p, stream) : launch_dq<fp16_tag, 256, false>(p, stream);
}
}  // namespace fdma
