// Backward dynamic-mask attention for gfx950, general form (mask and / or bias vary per query row): the dQ kernel.
//
// First kernel of the backward pass (see fdma_bwd.hip), which also leaves D = rowsum(dO * O) for the next: one workgroup per (128-query block, batch, head) loops over
// the key tiles like the forward kernel and computes, per 64-key tile,
//     S^T = K Q^T (+ bias, mask),  P^T = exp2(S^T - LSE),  dP^T = V dO^T,  dS^T = P^T o (dP^T - D),  dQ^T += K^T dS^T
// -- the dQ part of compute_dq_dk_dv_1colblock (csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the
// reference), with Q-stationary accumulation instead of fp32 atomics into a dQ workspace plus a convert pass
// (flash_bwd_kernel.h:940, flash_bwd_preprocess_kernel.h:212-304).
//
// Like the general forward kernel (fdma_fwd.hip) it is built around the mask / bias stream, which bounds this path:
// coalesced loads of every 128 x 64 mask and bias tile, fused in registers into one 16-bit tile in LDS that the score
// accumulators start from; K, V and the fused tile double-buffered and fetched a tile ahead, the mask two tiles
// ahead so that a tile without any kept element costs its mask bytes only; one barrier per tile (the OR reduction).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

// Workgroups have 4 waves (128 query rows; two per CU at d <= 64) or, at d = 128, 8: one workgroup fits on a CU there, and
// a second wave per SIMD hides what a single wave's in-order issue cannot.  On grids that stay large enough the 8 waves
// cover 256 rows; on smaller ones (KSPLIT) 128 rows, two waves per 32 rows that take the lower and the upper half of every
// key tile and add their sums through LDS at the end (B = 1, L = 1999, H = 16, d = 128, fp16: 128 us with four waves, 108
// so, odd rows read where they lie; 78 with K / V by direct loads, one barrier per tile and four heads to a workgroup).  Key tiles have 64 keys, and 32 with 256 rows (the 64-key tile's score and dP accumulators
// do not fit next to dQ and the Q / dO fragments in the 256 registers a wave has when two share a SIMD).
template <int D, int BM, int BN> struct DqSmem {
    static constexpr int SF = BN + 8;    // fused mask+bias tile row stride
    static constexpr int K_BYTES = BN * LdsTile<D>::ROW_BYTES;
    static constexpr int F_BYTES = BM * SF * 2;
    static constexpr int STAGE = (2 * K_BYTES + F_BYTES + 255) / 256 * 256;
    static constexpr int OFF_VOTE = 2 * STAGE;  // three words: "a tile has a kept element"
    static constexpr int OFF_D = OFF_VOTE + 16;  // KSPLIT: D of the workgroup's 128 rows
    static constexpr int TOTAL = OFF_D + 512;
};

template <typename T> struct NegInf2;
template <> struct NegInf2<bf16_tag> { static constexpr uint32_t value = 0xFF80FF80u; };
template <> struct NegInf2<fp16_tag> { static constexpr uint32_t value = 0xFC00FC00u; };

// GH query heads of a kv group that share mask and bias rows: a workgroup takes BM / GH query rows of GH heads (see fwd_kernel).
// SHARES: a workgroup takes one of p.dq_shares shares of the key tiles (an instantiation of its own, as in fwd_kernel).
template <typename T, int D, bool CAUSAL, int NW, int KSPLIT, int GH, bool ODD, bool SHARES>
__global__ void __launch_bounds__(64 * NW, (D <= 64 && NW == 4) ? 2 : 1) bwd_dq_kernel(const BwdParams p) {
    constexpr int NTHREADS = 64 * NW, BM = 32 * NW / KSPLIT / GH, RB = BM / 32, BN = ((NW == 8 && KSPLIT == 1) || D > 128) ? 32 : 64;
    constexpr int BK = BN / KSPLIT;         // keys of a tile per wave
    constexpr int FCH = BN / 8;             // 8-key chunks per mask / bias row of a tile
    constexpr int F_RPP = NTHREADS / FCH;   // mask / bias rows staged per pass
    using E = Elem<T>;
    using SM = DqSmem<D, BM, BN>;
    constexpr int KS = D / 16, DB = D / 32, MB = BK / 32, KB = BK / 16;
    constexpr int CH = D / 8;               // 16-byte chunks per K / V row
    constexpr int K_RPP = NTHREADS / CH;    // rows staged per pass
    constexpr int K_IT = BN / K_RPP;
    constexpr int F_CHUNKS = BM * FCH;         // 8-key chunks of the mask / bias tile
    constexpr int F_IT = F_CHUNKS > NTHREADS ? F_CHUNKS / NTHREADS : 1;  // ... per thread (the last waves fetch some again, when there are fewer)
    using TL = LdsTile<D>;
    constexpr bool DMA = TL::SWZ;  // K and V tiles by direct loads (see fwd_kernel)

    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = DMA ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : (int)threadIdx.x >> 6, lane = tid & 63, r = lane & 31, g = lane >> 5;
    // linear workgroup id -> (query block, member of the kv group, kv head, batch) with the query block OUTERMOST and
    // descending: under causal masking the blocks with the most KV tiles of every head start first, the light ones fill the
    // tail.  The members of a group, which read the same K / V and often the same mask and bias, are a multiple of the kv
    // head count apart: on one XCD (ids are dealt to the 8 XCDs in turn) when that is a multiple of 8.
    const int hb_count = f.H / GH * f.B, pairs = f.Hk * f.B;
    const int m_block = (int)gridDim.x / hb_count - 1 - (int)blockIdx.x / hb_count;
    const int pair = (int)blockIdx.x % pairs, hk = pair % f.Hk, b = pair / f.Hk;
    const int hs = wave % (RB * GH) / RB;  // head of this wave among the workgroup's
    const int h = hk * (f.H / f.Hk) + ((int)blockIdx.x % hb_count) / pairs * GH + hs;
    const int m0 = m_block * BM;
    const int rw = wave % RB, kh = wave / (RB * GH);  // row block and key half of this wave
    const int xw = wave % (RB * GH);  // (rows and heads: where the halves meet)
    const int wrow0 = m0 + rw * 32;
    const int qrow = wrow0 + r;
    const int qrow_c = qrow < f.Lq ? qrow : f.Lq - 1;
    const int shift = f.Lk - f.Lq;

    // ---- Q (scaled by softmax_scale * log2(e): it only feeds the scores here) and dO fragments, row statistics
    u32x4_t qf[KS], dof[KS];
    {
        const uint16_t *qp = (const uint16_t *)f.q + b * f.q_b + (int64_t)qrow_c * f.q_r + h * f.q_h;
        const uint16_t *dp = (const uint16_t *)p.dout + b * p.do_b + (int64_t)qrow_c * p.do_r + h * p.do_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            u32x4_t qv = {0, 0, 0, 0}, dv = {0, 0, 0, 0};
            if (qrow < f.Lq && c < f.d) { qv = *(const u32x4_t *)(qp + c); dv = *(const u32x4_t *)(dp + c); }
#pragma unroll
            for (int e = 0; e < 4; e++) qv[e] = E::pack2(E::lo(qv[e]) * f.scale_log2, E::hi(qv[e]) * f.scale_log2);
            qf[ks] = qv;
            dof[ks] = dv;
        }
    }
    float lse2 = INFINITY, dd = 0.f;
    if (qrow < f.Lq) lse2 = f.lse[((int64_t)b * f.H + h) * f.Lq + qrow] * kLog2e;
    // D = rowsum(dO * O) is made here, from the dO fragments, and left for the dK/dV kernel, which is launched behind this one: a launch less
    // (forward + backward, us: 1212 tokens x 8/4 heads, d = 64 124.5 / 121.8, 4 x 511 x 16/8, d = 256 242.1 / 236.8, 576 x 16/4, d = 128 89.9 / 86.1).  Of two waves with the same rows the first makes it, and the other finds it in LDS.
    if (KSPLIT == 1 || kh == 0) {
        const uint16_t *op = (const uint16_t *)f.o + b * f.o_b + (int64_t)qrow_c * f.o_r + h * f.o_h;
        u32x4_t of[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) of[ks] = *(const u32x4_t *)(op + (ks * 16 + g * 8 < f.d ? ks * 16 + g * 8 : 0));
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const bool on = qrow < f.Lq && ks * 16 + g * 8 < f.d;
            u32x4_t v = kept8(of[ks], on);  // (what is clamped need not be a number; dO is zero there)
#pragma unroll
            for (int e = 0; e < 4; e++) dd += E::lo(v[e]) * E::lo(dof[ks][e]) + E::hi(v[e]) * E::hi(dof[ks][e]);
        }
        dd = xhalf_sum(dd);
        float *d_out = p.softmax_d + b * p.sd_b + h * p.sd_h;
        if (g == 0 && (!SHARES || blockIdx.y == 0)) {
            if (qrow < p.Lq_rounded) d_out[qrow] = dd;  // (padded rows are zero)
            if (m0 + BM >= f.Lq && rw == 0)
                for (int row = m0 + BM + r; row < p.Lq_rounded; row += 32) d_out[row] = 0.f;
        }
        if (KSPLIT == 2 && g == 0) lds_st32(lds0 + SM::OFF_D + (xw * 32 + r) * 4, __float_as_uint(dd));
    }

    int n_end = (f.Lk + BN - 1) / BN;
    if (CAUSAL) {
        int lim = m0 + BM + shift;
        if (lim > f.Lq + shift) lim = f.Lq + shift;
        if (lim < 0) lim = 0;
        const int ne = (lim + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }
    // this workgroup's share of them (see general_key_shares), whole pairs: the LDS stage of a tile stays a compile-time constant
    int t_first = 0;
    if constexpr (SHARES) {
        const int y = (int)blockIdx.y, twos = (n_end + 1) / 2;
        t_first = 2 * (twos * y / p.dq_shares);
        if (y + 1 < p.dq_shares) n_end = 2 * (twos * (y + 1) / p.dq_shares);
    }

    f32x16_t dq[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dq[db][i] = 0.f;

    const int hm = f.mask ? (f.Hm == f.H ? h : (f.Hm == 1 ? 0 : h / (f.H / f.Hm))) : 0;
    const int hb = f.bias ? (f.Hb == f.H ? h : (f.Hb == 1 ? 0 : h / (f.H / f.Hb))) : 0;
    const uint8_t *mbase = f.mask ? f.mask + b * f.m_b + hm * f.m_h : nullptr;
    const uint16_t *bbase = f.bias ? (const uint16_t *)f.bias + b * f.bi_b + hb * f.bi_h : nullptr;
    const uint16_t *kbase = (const uint16_t *)f.k + b * f.k_b + hk * f.k_h;
    const uint16_t *vbase = (const uint16_t *)f.v + b * f.v_b + hk * f.v_h;

    // ---- staging maps; all tile loads are unconditional, from clamped (always valid) addresses: rows of K / V beyond
    // Lk and head-dim chunks beyond d are finite duplicates that meet a -inf score or a zero fragment, and the mask
    // words are ANDed with a validity pattern when they are consumed
    const int kc = tid % CH, kr0 = tid / CH;
    const int kcol = kc * 8 < f.d ? kc * 8 : 0;
    const int kc_g = kc ^ (int)TL::swz(kr0), kcol_g = kc_g * 8 < f.d ? kc_g * 8 : 0;  // (DMA: what chunk position kc of its rows holds)
    const int fc = tid % FCH, fr0 = tid / FCH % BM;  // mask / bias: 8-key chunk, first row (rows fr0 + F_RPP it)
    u32x4_t kreg[DMA ? 1 : K_IT], vreg[DMA ? 1 : K_IT], breg[F_IT];
    u32x2_t mreg[F_IT], mnext[F_IT];

    // (a mask that comes packed to bits: one byte per 8-key chunk instead of eight, expanded where it is looked at)
    const uint8_t *mbits = (mbase && f.mbits) ? f.mbits + b * f.mb_b + hm * f.mb_h : nullptr;
    auto load_mask = [&](int j, u32x2_t (&dst)[F_IT]) {
        if (!mbase) return;
        int kk = j * BN + 8 * fc;
        kk = kk < f.Lk ? kk : 0;
        const int at = chunk8_at<ODD>(j * BN + 8 * fc, f.Lk);
#pragma unroll
        for (int it = 0; it < F_IT; it++) {
            int row = m0 + fr0 + F_RPP * it;
            row = row < f.Lq ? row : f.Lq - 1;
            // (one 8-byte load either way, from an address chosen without a branch: mask bytes of the chunk, or the
            // aligned piece of the bit row that holds the chunk's byte)
            const uint8_t *src = mbits ? mbits + (int64_t)row * f.mb_r + ((kk >> 3) & ~7) : mbase + (int64_t)row * f.m_r + at;
            dst[it] = *(const u32x2_any_t *)src;
        }
    };
    auto finish_mask = [&](int j, u32x2_t (&dst)[F_IT]) -> bool {
        const int kk = j * BN + 8 * fc;
        uint32_t any = 0;
#pragma unroll
        for (int it = 0; it < F_IT; it++) {
            const int row = m0 + fr0 + F_RPP * it;
            u32x2_t mv = mbase ? (mbits ? mask_bits_to_bytes(mask_bits_byte(dst[it], kk)) : chunk8_fix_mask<ODD>(dst[it], kk, f.Lk)) : u32x2_t{0x01010101u, 0x01010101u};
            const bool ok = row < f.Lq && kk < f.Lk && !(CAUSAL && kk > row + shift);
            uint64_t keepm = ok ? ~0ull : 0ull;
            if (kk + 8 > f.Lk && kk < f.Lk) keepm = (1ull << (8 * (f.Lk - kk))) - 1ull;
            mv[0] &= (uint32_t)keepm;
            mv[1] &= (uint32_t)(keepm >> 32);
            dst[it] = mv;
            any |= mv[0] | mv[1];
        }
        return any != 0;
    };
    auto load_rest = [&](int j) {
        const int n0 = j * BN;
        if (bbase) {
            const int at = chunk8_at<ODD>(n0 + 8 * fc, f.Lk);
#pragma unroll
            for (int it = 0; it < F_IT; it++) {
                int row = m0 + fr0 + F_RPP * it;
                row = row < f.Lq ? row : f.Lq - 1;
                breg[it] = *(const u32x4_el_t *)(bbase + (int64_t)row * f.bi_r + at);
            }
        } else {
#pragma unroll
            for (int it = 0; it < F_IT; it++) breg[it] = u32x4_t{0, 0, 0, 0};
        }
        if constexpr (DMA) {
            const gptr_t kb = uniform_ptr(kbase + (int64_t)n0 * f.k_r), vb = uniform_ptr(vbase + (int64_t)n0 * f.v_r);
            const int last = f.Lk - 1 - n0;
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)((j & 1) * SM::STAGE) + (uint32_t)wave * 1024);
#pragma unroll
            for (int it = 0; it < K_IT; it++) {
                const int row = kr0 + it * K_RPP, row_c = row < last ? row : last;
                const uint32_t ko = (uint32_t)(row_c * (int)f.k_r + kcol_g) * 2, vo = (uint32_t)(row_c * (int)f.v_r + kcol_g) * 2;
                load_lds16<true>(ko, kb, dst + it * K_RPP * 256);
                load_lds16<true>(vo, vb, dst + SM::K_BYTES + it * K_RPP * 256);
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < K_IT; it++) {
            int key = n0 + kr0 + it * K_RPP;
            key = key < f.Lk ? key : f.Lk - 1;
            kreg[it] = *(const u32x4_t *)(kbase + (int64_t)key * f.k_r + kcol);
            vreg[it] = *(const u32x4_t *)(vbase + (int64_t)key * f.v_r + kcol);
        }
    };
    auto store_stage = [&](int j, const u32x2_t (&mv)[F_IT]) {
        const int buf = j & 1, kk = j * BN + 8 * fc;
        char *sK = smem + buf * SM::STAGE;
        char *sV = sK + SM::K_BYTES;
        char *sF = sV + SM::K_BYTES;
        if constexpr (!DMA) {
#pragma unroll
            for (int it = 0; it < K_IT; it++) {
                *(u32x4_t *)(sK + TL::chunk(kr0 + it * K_RPP, kc)) = kreg[it];
                *(u32x4_t *)(sV + TL::chunk(kr0 + it * K_RPP, kc)) = vreg[it];
            }
        }
        if (F_CHUNKS < NTHREADS && wave >= F_CHUNKS / 64) return;
#pragma unroll
        for (int it = 0; it < F_IT; it++) {
            u32x4_t bv = bbase ? chunk8_fix<ODD>(breg[it], kk, f.Lk) : breg[it];
#pragma unroll
            for (int hlf = 0; hlf < 2; hlf++) {
                uint32_t x = mv[it][hlf];
                x = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) >> 7) & 0x01010101u;  // nonzero byte -> 0x01
                const uint32_t z = (x << 8) - x;                                      // 0x01 -> 0xFF per byte
                const uint32_t m0w = __builtin_amdgcn_perm(0, z, 0x01010000u);        // [b0 b0 b1 b1]
                const uint32_t m1w = __builtin_amdgcn_perm(0, z, 0x03030202u);        // [b2 b2 b3 b3]
                bv[2 * hlf] = (bv[2 * hlf] & m0w) | (NegInf2<T>::value & ~m0w);
                bv[2 * hlf + 1] = (bv[2 * hlf + 1] & m1w) | (NegInf2<T>::value & ~m1w);
            }
            *(u32x4_t *)(sF + ((fr0 + F_RPP * it) * SM::SF + 8 * fc) * 2) = bv;
        }
    };

    const int a_row = pi_row(r);
    const uint32_t a_off = lds0 + TL::frag_base(a_row, g);
    const TrLane tr = tr_lane(lane);
    const uint32_t tr_off = lds0 + TL::tr_base(g, tr);

    auto compute = [&](int j, int buf) {
        const int n0 = j * BN + kh * BK;
        const uint32_t st = (uint32_t)(buf * SM::STAGE + kh * BK * TL::ROW_BYTES);
        uint32_t a_cur = a_off + st, tr_cur = tr_off + st;
        if (TL::SWZ) asm volatile("" : "+v"(a_cur), "+v"(tr_cur));  // (the swizzled addresses are recomputed where used)
        const char *sF = smem + buf * SM::STAGE + 2 * SM::K_BYTES + ((rw * 32 + r) * SM::SF + kh * BK + 8 * g) * 2;
        // ---- S^T = K Q^T on top of the fused mask+bias tile, dP^T = V dO^T
        f32x16_t s[MB], dp[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const u32x4_t fv = *(const u32x4_t *)(sF + (32 * mb + 16 * blk) * 2);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s[mb][8 * blk + 2 * e] = E::lo(fv[e]) * kLog2e;
                    s[mb][8 * blk + 2 * e + 1] = E::hi(fv[e]) * kLog2e;
                    dp[mb][8 * blk + 2 * e] = 0.f;
                    dp[mb][8 * blk + 2 * e + 1] = 0.f;
                }
            }
        {
            constexpr int NF = 2 * MB * KS, FR = DMA || ODD ? 6 : 8;  // fragment fi: (ks, mb, which) with which = 0: K, 1: V
            u32x4_t a[NF];
            auto frag = [&](int fi) {
                const int which = fi & 1, mb = (fi >> 1) % MB, ks = (fi >> 1) / MB;
                return lds_ld128(TL::frag_at(a_cur, ks) + (uint32_t)(which * SM::K_BYTES + 32 * mb * TL::ROW_BYTES));
            };
#pragma unroll
            for (int fi = 0; fi < FR; fi++) a[fi] = frag(fi);
#pragma unroll
            for (int fi = 0; fi < NF; fi++) {
                if (fi + FR < NF) a[fi + FR] = frag(fi + FR);
                const int which = fi & 1, mb = (fi >> 1) % MB, ks = (fi >> 1) / MB;
                if (which) dp[mb] = E::mfma(a[fi], dof[ks], dp[mb]);
                else s[mb] = E::mfma(a[fi], qf[ks], s[mb]);
            }
        }
        // ---- dS^T = P^T o (dP^T - D); causal selects on diagonal tiles only (wave-uniform branch)
        const bool diag = CAUSAL && (n0 + BK - 1 > wrow0 + shift);
        uint32_t dpk[8 * MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                float pv[8];
#pragma unroll
                for (int e = 0; e < 8; e++) pv[e] = fast_exp2(s[mb][8 * blk + e] - lse2);
                if (diag) {
                    asm volatile("" ::: "memory");
                    const int lim = qrow + shift - n0 - 32 * mb - 16 * blk - 8 * g;  // local columns e <= lim are visible
#pragma unroll
                    for (int e = 0; e < 8; e++) pv[e] = e <= lim ? pv[e] : 0.f;
                }
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float d0 = pv[2 * e] * (dp[mb][8 * blk + 2 * e] - dd);
                    const float d1 = pv[2 * e + 1] * (dp[mb][8 * blk + 2 * e + 1] - dd);
                    dpk[8 * mb + 4 * blk + e] = E::pack2(d0, d1);
                }
            }
        // ---- dQ^T += K^T dS^T  (K^T through transposing LDS reads of the row-major K tile, one pair ahead)
        {
            constexpr int NP = KB * DB;
            u32x4_t a[2];
            auto frag = [&](int idx, int slot) {
                const int kb = idx / DB, db = idx % DB;
                const u32x2_t lo = lds_ld_tr16(TL::tr_at(tr_cur, kb, db, 0)), hi = lds_ld_tr16(TL::tr_at(tr_cur, kb, db, 1));
                a[slot] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            };
            frag(0, 0);
#pragma unroll
            for (int idx = 0; idx < NP; idx++) {
                if (idx + 1 < NP) frag(idx + 1, (idx + 1) & 1);
                const int kb = idx / DB, db = idx % DB;
                const u32x4_t bop = {dpk[4 * kb], dpk[4 * kb + 1], dpk[4 * kb + 2], dpk[4 * kb + 3]};
                dq[db] = E::mfma(a[idx & 1], bop, dq[db]);
            }
        }
    };

    // the end of a step (see fwd_kernel): the vote of a tile's mask, published by the barrier that publishes the step's tiles
    int vote_at = 0;
    if (tid < 3) lds_st32(lds0 + SM::OFF_VOTE + 4 * tid, 0u);
    auto step_end = [&](bool any) -> bool {
        const uint32_t at = lds0 + SM::OFF_VOTE + 4 * vote_at;
        vote_at = vote_at == 2 ? 0 : vote_at + 1;
        if (__any(any)) lds_st32(at, 1u);
        if (tid == 0) lds_st32(lds0 + SM::OFF_VOTE + 4 * vote_at, 0u);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        return __builtin_amdgcn_readfirstlane(lds_ld32(at)) != 0u;
    };

    // ---- main loop.  At the top of iteration j: tile j sits in LDS stage j&1 if it is active, the mask of tile j+1 is
    // in registers (finished) and `act_next` says whether that tile has any kept element.
    if (t_first < n_end) {
        load_mask(t_first, mreg);
        if (t_first + 1 < n_end) load_mask(t_first + 1, mnext);
        bool act_cur = __syncthreads_or(finish_mask(t_first, mreg));
        if (KSPLIT == 2 && kh == 1) dd = __uint_as_float(lds_ld32(lds0 + SM::OFF_D + (xw * 32 + r) * 4));
        if (act_cur) {
            load_rest(t_first);
            store_stage(t_first, mreg);
        }
        if (DMA) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        bool act_next = __syncthreads_or(t_first + 1 < n_end && finish_mask(t_first + 1, mnext));
        auto step = [&](int j, u32x2_t (&m_next)[F_IT], u32x2_t (&m_new)[F_IT]) {
            const bool have_next = j + 1 < n_end && act_next;
            if (have_next) load_rest(j + 1);
            if (j + 2 < n_end) load_mask(j + 2, m_new);
            __builtin_amdgcn_sched_barrier(0);  // loads above, their first use below the compute
            if (act_cur) compute(j, j & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (have_next) store_stage(j + 1, m_next);
            const bool act_nn = step_end(j + 2 < n_end && finish_mask(j + 2, m_new));
            act_cur = have_next;
            act_next = act_nn;
        };
        for (int j = t_first; j < n_end; j += 2) {
            step(j, mnext, mreg);
            if (j + 1 < n_end) step(j + 1, mreg, mnext);
        }
    }

    if constexpr (KSPLIT == 2) {  // the upper key half hands over its sums
        f32x4_t *xo = (f32x4_t *)smem + xw * DB * 4 * 64 + lane;
        __syncthreads();  // (the tiles' last reads)
        if (kh == 1) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    xo[(db * 4 + q) * 64] = f32x4_t{dq[db][4 * q], dq[db][4 * q + 1], dq[db][4 * q + 2], dq[db][4 * q + 3]};
        }
        __syncthreads();
        if (kh == 1) return;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4_t v = xo[(db * 4 + q) * 64];
#pragma unroll
                for (int e = 0; e < 4; e++) dq[db][4 * q + e] += v[e];
            }
    }
    if constexpr (SHARES) {  // its sums in fp32, which bwd_dq_sum_kernel adds up (zeros where it has no tile)
        if (qrow < f.Lq) {
            float *at = p.dq_part + ((((int64_t)blockIdx.y * f.B + b) * f.H + h) * f.Lq + qrow) * f.d;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int c = 32 * db + 16 * (q >> 1) + 8 * g + 4 * (q & 1);
                    if (c < f.d) *(f32x4_t *)(at + c) = f32x4_t{dq[db][4 * q], dq[db][4 * q + 1], dq[db][4 * q + 2], dq[db][4 * q + 3]};
                }
        }
        return;
    }
    if (qrow < f.Lq) {
        uint16_t *dqp = (uint16_t *)p.dq + b * p.dq_b + (int64_t)qrow * p.dq_r + h * p.dq_h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
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

// dQ = scale * sum of the shares, in their order.  A thread has 8 elements of one row.
template <typename T> __global__ void __launch_bounds__(256) bwd_dq_sum_kernel(const BwdParams p) {
    using E = Elem<T>;
    const FwdParams &f = p.f;
    const int CH = f.d / 8;
    const int64_t rows = (int64_t)f.B * f.H * f.Lq, at = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= rows * CH) return;
    const int64_t row = at / CH;
    const int c = (int)(at % CH) * 8;
    f32x4_t v[MAX_KEY_SPLITS][2];
#pragma unroll
    for (int s = 0; s < MAX_KEY_SPLITS; s++) {
        v[s][0] = v[s][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (s < p.dq_shares) {
            v[s][0] = *(const f32x4_t *)(p.dq_part + (s * rows + row) * f.d + c);
            v[s][1] = *(const f32x4_t *)(p.dq_part + (s * rows + row) * f.d + c + 4);
        }
    }
#pragma unroll
    for (int s = 1; s < MAX_KEY_SPLITS; s++)
#pragma unroll
        for (int e = 0; e < 4; e++) { v[0][0][e] += v[s][0][e]; v[0][1][e] += v[s][1][e]; }
    const int q = (int)(row % f.Lq), h = (int)(row / f.Lq % f.H), b = (int)(row / f.Lq / f.H);
    u32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = E::pack2(v[0][e >> 1][2 * (e & 1)] * f.scale, v[0][e >> 1][2 * (e & 1) + 1] * f.scale);
    *(u32x4_t *)((uint16_t *)p.dq + b * p.dq_b + q * p.dq_r + h * p.dq_h + c) = w;
}

template <typename T, int D, bool CAUSAL, int NW, int KSPLIT, int GH, bool ODD, bool SHARES = false>
hipError_t launch_dq_o(const BwdParams &p, hipStream_t stream) {
    constexpr int BM = 32 * NW / KSPLIT / GH, NTHREADS = 64 * NW, BN = ((NW == 8 && KSPLIT == 1) || D > 128) ? 32 : 64;
    if constexpr (!SHARES) {
        if (p.dq_shares > 1) {
            if constexpr (KSPLIT == 2 || NW == 4) return launch_dq_o<T, D, CAUSAL, NW, KSPLIT, GH, ODD, true>(p, stream);
            else return hipErrorInvalidValue;  // (general_key_shares plans none for the kernels of 256 rows)
        }
    }
    auto kern = bwd_dq_kernel<T, D, CAUSAL, NW, KSPLIT, GH, ODD, SHARES>;
    constexpr int merge = KSPLIT == 2 ? (NW / 2) * (D / 32) * 4096 : 0;  // the upper halves' sums
    constexpr int smem = DqSmem<D, BM, BN>::TOTAL > merge ? DqSmem<D, BM, BN>::TOTAL : merge;
    static DynSmemLimit smem_limit;
    hipError_t e = smem_limit.ensure((const void *)kern, (int)smem);
    if (e != hipSuccess) return e;
    dim3 grid(((p.f.Lq + BM - 1) / BM) * (p.f.H / GH) * p.f.B);
    if constexpr (SHARES) grid.y = p.dq_shares;
    hipLaunchKernelGGL(kern, grid, dim3(NTHREADS), smem, stream, p);
    return hipGetLastError();
}

template <typename T, int D, bool CAUSAL, int NW, int KSPLIT = 1>
hipError_t launch_dq_n(const BwdParams &p, hipStream_t stream) {
    const int gh = shared_rows(p.f);
    // (at d = 65 .. 128 whole aligned chunks / rows read where they lie, forward and backward, us: 2000 tokens x 16/4 heads 215 / 220,
    // 1024 x 16/8, causal 117 / 120, 1000 x 8/2 103 / 106)
    auto pick = [&](auto odd) -> hipError_t {
        constexpr bool O = decltype(odd)::value;
        if constexpr (D <= 128) if (gh == 4) return launch_dq_o<T, D, CAUSAL, NW, KSPLIT, 4, O>(p, stream);
        if constexpr (D > 64) if (gh == 2) return launch_dq_o<T, D, CAUSAL, NW, KSPLIT, 2, O>(p, stream);
        return launch_dq_o<T, D, CAUSAL, NW, KSPLIT, 1, O>(p, stream);
    };
    if (D > 128 || odd_rows(p.f)) return pick(std::true_type());
    return pick(std::bool_constant<(D > 128)>());
}

template <typename T, int D, bool CAUSAL>
hipError_t launch_dq_c(const BwdParams &p, hipStream_t stream) {
    if constexpr (D > 64 && D <= 128) {
        if (general_rows_256(p.f)) return launch_dq_n<T, D, CAUSAL, 8>(p, stream);
        return launch_dq_n<T, D, CAUSAL, 8, 2>(p, stream);
    } else {
        return launch_dq_n<T, D, CAUSAL, 4>(p, stream);
    }
}

}  // namespace

static hipError_t launch_dq_d(const BwdParams &p, int dtype, hipStream_t stream) {
    // head dims up to 64 / 128 / 256 (a head dim in between runs in the next larger instantiation)
    const int dc = p.f.d <= 64 ? 0 : (p.f.d <= 128 ? 1 : 2);
    const bool c = p.f.causal != 0;
    if (dtype == 0) {
        if (dc == 0) return c ? launch_dq_c<bf16_tag, 64, true>(p, stream) : launch_dq_c<bf16_tag, 64, false>(p, stream);
        if (dc == 1) return c ? launch_dq_c<bf16_tag, 128, true>(p, stream) : launch_dq_c<bf16_tag, 128, false>(p, stream);
        return c ? launch_dq_c<bf16_tag, 256, true>(p, stream) : launch_dq_c<bf16_tag, 256, false>(p, stream);
    }
    if (dc == 0) return c ? launch_dq_c<fp16_tag, 64, true>(p, stream) : launch_dq_c<fp16_tag, 64, false>(p, stream);
    if (dc == 1) return c ? launch_dq_c<fp16_tag, 128, true>(p, stream) : launch_dq_c<fp16_tag, 128, false>(p, stream);
    return c ? launch_dq_c<fp16_tag, 256, true>(p, stream) : launch_dq_c<fp16_tag, 256, false>(p, stream);
}

hipError_t launch_bwd_dq(const BwdParams &p, int dtype, hipStream_t stream) {
    const hipError_t e = launch_dq_d(p, dtype, stream);
    if (e != hipSuccess || p.dq_shares <= 1) return e;
    const int64_t items = (int64_t)p.f.B * p.f.H * p.f.Lq * (p.f.d / 8);
    const dim3 grid((unsigned)((items + 255) / 256));
    if (dtype == 0) hipLaunchKernelGGL(bwd_dq_sum_kernel<bf16_tag>, grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL(bwd_dq_sum_kernel<fp16_tag>, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace fdma
