// Forward dynamic-mask attention for gfx950, general form: mask and / or bias vary per query row.
//
// Replaces compute_attn_1rowblock (csrc/flash_sparse_attn/src/flash_fwd_kernel.h:53-804) with its
// online softmax (src/softmax.h:127-221), masking (src/mask.h:94-161) and mask-tile OR skip
// (src/utils.h:339-352) of the reference.  Same math:
//     S = Q K^T * scale + bias ; S[~mask or non-causal] = -inf ; P = softmax(S) ; O = P V
// with the causal mask aligned bottom-right, O = 0 and LSE = +inf for rows with no visible key.
// (Mask and bias that are absent or broadcast over queries take the kernels of fdma_fwd_colmask.hip.)
//
// One workgroup = 4 waves = 128 query rows of one (batch, head); each wave owns 32 rows and computes the
// TRANSPOSED score tile S^T = K Q^T (K rows from LDS as the MFMA A operand, its pre-scaled Q rows in
// registers as the B operand), so a lane owns one query row and row max / row sum are in-lane reductions
// plus one cross-half swap.  P^T feeds O^T = V^T P^T straight from the accumulator registers; V^T comes out of the
// row-major V tile through transposing LDS reads.
//
// With a [Lq, Lk] bias (2 B) and mask (1 B) per score this path is bound by HBM, not by the matrix pipe, so the
// kernel is built around the mask / bias stream:
//   * every 128 x 64 mask and bias tile is fetched with coalesced 8- / 16-byte loads (a row's 64 keys are
//     contiguous), fused in registers into one 16-bit tile (bias where kept, -inf where dropped or beyond Lk) and
//     parked in LDS; the score accumulators then START from that tile, so bias and mask cost nothing later;
//   * everything is double-buffered and fetched a tile ahead, the mask two tiles ahead: the workgroup-wide OR
//     of the next tile's mask is known before that tile's bias / K / V loads are issued, and a tile without
//     any kept element costs its mask bytes only (no bias, K, V traffic, no MFMA work);
//   * one barrier per tile, which the vote of the OR is published by (__syncthreads_or is three: 6 us of 74 at 1999 x 16 heads,
//     d = 128).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_fwd_merge.h"

namespace fdma {

namespace {

// Workgroups have 4 waves (128 query rows; two per CU at d <= 64) or, at d = 128, 8: only one workgroup fits on a CU there,
// and with a single wave per SIMD nothing hides the in-order issue of that wave -- a second wave per SIMD does.  On grids
// that stay large enough the 8 waves cover 256 rows; on smaller ones (KSPLIT) 128 rows, two waves per 32 rows that take
// the lower and the upper half of every key tile with a softmax of their own and are merged through LDS at the end
// (B = 1, L = 1999, H = 16, d = 128, fp16: 108 us with four waves, 88 so, the rows read where they lie; 57 with K / V by direct
// loads, one barrier per tile and four heads to a workgroup).
constexpr int BN_DEFAULT = 64;  // keys per tile (32 at head dims above 128: LDS)

template <int D, int BM, int BN> struct FwdSmem {
    static constexpr int SF = BN + 8;    // fused mask+bias tile row stride
    static constexpr int K_BYTES = BN * LdsTile<D>::ROW_BYTES;  // a K or V tile (row-major both; V is read through transposing LDS reads)
    static constexpr int F_BYTES = BM * SF * 2;
    static constexpr int STAGE = (2 * K_BYTES + F_BYTES + 255) / 256 * 256;
    static constexpr int OFF_VOTE = 2 * STAGE;  // three words: "a tile has a kept element"
    static constexpr int TOTAL = OFF_VOTE + 16;
};

template <typename T> struct NegInf2;
template <> struct NegInf2<bf16_tag> { static constexpr uint32_t value = 0xFF80FF80u; };
template <> struct NegInf2<fp16_tag> { static constexpr uint32_t value = 0xFC00FC00u; };

// GH query heads of a kv group that share mask and bias rows: a workgroup takes BM / GH query rows of GH heads, so that a fused tile
// is fetched, fused and stored once for all of them.
// SHARES: a workgroup takes one of p.splits shares of the key tiles (an instantiation of its own: what it adds costs the others 2 %).
template <typename T, int D, bool CAUSAL, int NW, int BN, int KSPLIT, int GH, bool ODD, bool SHARES>
__global__ void __launch_bounds__(64 * NW, (D <= 64 && NW == 4) ? 2 : 1) fwd_kernel(const FwdParams p) {
    constexpr int NTHREADS = 64 * NW, BK = BN / KSPLIT;  // (BK: keys of a tile per wave)
    constexpr int BM = 32 * NW / KSPLIT / GH, RB = BM / 32;  // query rows and 32-row blocks per head
    constexpr int FCH = BN / 8;             // 8-key chunks per mask / bias row of a tile
    constexpr int F_RPP = NTHREADS / FCH;   // mask / bias rows staged per pass (FCH threads cover the keys of a row)
    using E = Elem<T>;
    using SM = FwdSmem<D, BM, BN>;
    constexpr int KS = D / 16;  // contraction steps of Q K^T
    constexpr int DB = D / 32;  // 32-wide blocks of the head dimension
    constexpr int MB = BK / 32, KB = BK / 16;
    constexpr int CH = D / 8;               // 16-byte chunks per K row
    constexpr int K_RPP = NTHREADS / CH;    // K rows staged per pass
    constexpr int K_IT = BN / K_RPP;
    constexpr int F_CHUNKS = BM * (BN / 8);  // 8-key chunks of the mask / bias tile
    constexpr int F_IT = F_CHUNKS > NTHREADS ? F_CHUNKS / NTHREADS : 1;  // ... per thread (the last waves fetch some again, when there are fewer)

    using TL = LdsTile<D>;
    // DMA (rows of exactly 256 bytes): K and V tiles go from global memory straight into LDS (global_load_lds; the swizzle of the
    // tile is applied to the global address of each lane's piece).  Through registers, their loads and stores were a fifth of
    // the kernel at head dim 128.
    constexpr bool DMA = TL::SWZ;

    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const int tid = threadIdx.x, wave = DMA ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : (int)threadIdx.x >> 6, lane = tid & 63, r = lane & 31, g = lane >> 5;
    // linear workgroup id -> (query block, member of the kv group, kv head, batch) with the query block OUTERMOST and
    // descending: under causal masking the blocks with the most KV tiles of every head start first, the light ones fill the
    // tail.  The members of a group, which read the same K / V and often the same mask and bias, are a multiple of the kv
    // head count apart: on one XCD (ids are dealt to the 8 XCDs in turn) when that is a multiple of 8.
    const int hb_count = p.H / GH * p.B, pairs = p.Hk * p.B;
    const int m_block = (int)gridDim.x / hb_count - 1 - (int)blockIdx.x / hb_count;
    const int pair = (int)blockIdx.x % pairs, hk = pair % p.Hk, b = pair / p.Hk;
    const int hs = wave % (RB * GH) / RB;  // head of this wave among the workgroup's
    const int h = hk * (p.H / p.Hk) + ((int)blockIdx.x % hb_count) / pairs * GH + hs;
    const int m0 = m_block * BM;
    const int rw = wave % RB, kh = wave / (RB * GH);  // row block and key half of this wave
    const int xw = wave % (RB * GH);  // (rows and heads: where the halves meet)
    const int wrow0 = m0 + rw * 32;
    const int qrow = wrow0 + r;
    const int shift = p.Lk - p.Lq;  // bottom-right causal alignment

    // ---- Q fragments (B operand of S^T = K Q^T), scaled by softmax_scale * log2(e) once (the reference also rounds
    // the scaled Q to the input type, flash_fwd_kernel.h:428-439) and kept in registers for the whole KV loop
    u32x4_t qf[KS];
    {
        const int qc = qrow < p.Lq ? qrow : p.Lq - 1;
        const uint16_t *qp = (const uint16_t *)p.q + b * p.q_b + (int64_t)qc * p.q_r + h * p.q_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            u32x4_t v = {0, 0, 0, 0};
            if (qrow < p.Lq && c < p.d) v = *(const u32x4_t *)(qp + c);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = E::pack2(E::lo(v[e]) * p.scale_log2, E::hi(v[e]) * p.scale_log2);
            qf[ks] = v;
        }
    }

    int n_end = (p.Lk + BN - 1) / BN;
    if (CAUSAL) {
        int lim = m0 + BM + shift;  // first invisible column for the last row of the block
        if (lim > p.Lq + shift) lim = p.Lq + shift;
        if (lim < 0) lim = 0;
        const int ne = (lim + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }
    // this workgroup's share of them (see general_key_shares), whole pairs: the LDS stage of a tile stays a compile-time constant
    int t_first = 0;
    if constexpr (SHARES) {
        const int y = (int)blockIdx.y, twos = (n_end + 1) / 2;
        t_first = 2 * (twos * y / p.splits);
        if (y + 1 < p.splits) n_end = 2 * (twos * (y + 1) / p.splits);
    }

    f32x16_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;
    float row_max = -INFINITY;  // exp2 domain
    float row_sum = 0.f;        // per-lane partial (this lane's half of the keys)

    const int hm = p.mask ? (p.Hm == p.H ? h : (p.Hm == 1 ? 0 : h / (p.H / p.Hm))) : 0;
    const int hb = p.bias ? (p.Hb == p.H ? h : (p.Hb == 1 ? 0 : h / (p.H / p.Hb))) : 0;
    const uint8_t *mbase = p.mask ? p.mask + b * p.m_b + hm * p.m_h : nullptr;
    const uint16_t *bbase = p.bias ? (const uint16_t *)p.bias + b * p.bi_b + hb * p.bi_h : nullptr;
    const uint16_t *kbase = (const uint16_t *)p.k + b * p.k_b + hk * p.k_h;
    const uint16_t *vbase = (const uint16_t *)p.v + b * p.v_b + hk * p.v_h;

    // ---- staging maps
    const int kc = tid % CH, kr0 = tid / CH;             // K: d chunk, first row
    const bool k_dvalid = kc * 8 < p.d;
    const int fc = tid % FCH, fr0 = tid / FCH % BM;      // mask / bias: 8-key chunk, first row (rows fr0 + F_RPP it)
    u32x4_t kreg[DMA ? 1 : K_IT], vreg[DMA ? 1 : K_IT], breg[F_IT];
    u32x2_t mreg[F_IT], mnext[F_IT];

    // All tile loads are unconditional, from clamped (always valid) addresses, so that they can be issued early and
    // stay in flight; what a clamped load fetched in place of a missing element is neutralised later: the mask
    // words are ANDed with a validity pattern when they are consumed, rows of K / V beyond Lk and head-dim chunks
    // beyond d are finite duplicates that meet a -inf score or a zero Q fragment.
    const int kcol = k_dvalid ? kc * 8 : 0;
    // (DMA: the lane fills chunk POSITION kc of its rows, which holds chunk kc ^ swz(row) of the global row; rows 32 apart have the
    // same swizzle)
    const int kc_g = kc ^ (int)TL::swz(kr0), kcol_g = kc_g * 8 < p.d ? kc_g * 8 : 0;
    // (a mask that comes packed to bits: one byte per 8-key chunk instead of eight, expanded where it is looked at)
    const bool bits = mbase && p.mbits;
    const uint8_t *mrows = bits ? p.mbits + b * p.mb_b + hm * p.mb_h : mbase;
    const int64_t mrow_bytes = bits ? p.mb_r : p.m_r;
    // One 8-byte load from one address: with the choice left to the loads they become two, in branches (d = 256, 2316 x 2/1, causal 170
    // us, so 155; 4 x 2047 x 16, d = 128 200, so 188).
    auto load_mask = [&](int j, u32x2_t (&dst)[F_IT]) {
        if (!mbase) return;
        const int at = mask_piece_at(bits, j * BN + 8 * fc, p.Lk);
#pragma unroll
        for (int it = 0; it < F_IT; it++) {
            int row = m0 + fr0 + F_RPP * it;
            row = row < p.Lq ? row : p.Lq - 1;
            dst[it] = *(const u32x2_any_t *)(mrows + (int64_t)row * mrow_bytes + at);
        }
    };
    // validity of the chunks (rows < Lq, keys < Lk, not entirely above the causal diagonal) applied to the loaded
    // mask words; returns "any element kept"
    auto finish_mask = [&](int j, u32x2_t (&dst)[F_IT]) -> bool {
        const int kk = j * BN + 8 * fc;
        uint32_t any = 0;
#pragma unroll
        for (int it = 0; it < F_IT; it++) {
            const int row = m0 + fr0 + F_RPP * it;
            u32x2_t mv = mbase ? (bits ? mask_bits_to_bytes(mask_bits_byte(dst[it], kk)) : chunk8_fix_mask<ODD>(dst[it], kk, p.Lk)) : u32x2_t{0x01010101u, 0x01010101u};
            const bool ok = row < p.Lq && kk < p.Lk && !(CAUSAL && kk > row + shift);
            uint64_t keepm = ok ? ~0ull : 0ull;
            if (kk + 8 > p.Lk && kk < p.Lk) keepm = (1ull << (8 * (p.Lk - kk))) - 1ull;  // chunk straddles the end of the keys
            mv[0] &= (uint32_t)keepm;
            mv[1] &= (uint32_t)(keepm >> 32);
            dst[it] = mv;
            any |= mv[0] | mv[1];
        }
        return any != 0;
    };
    // bias of tile j into registers
    auto load_bias = [&](int j, u32x4_t (&dst)[F_IT]) {
        const int n0 = j * BN;
        if (bbase) {
            const int at = chunk8_at<ODD>(n0 + 8 * fc, p.Lk);
#pragma unroll
            for (int it = 0; it < F_IT; it++) {
                int row = m0 + fr0 + F_RPP * it;
                row = row < p.Lq ? row : p.Lq - 1;
                dst[it] = *(const u32x4_el_t *)(bbase + (int64_t)row * p.bi_r + at);
            }
        } else {
#pragma unroll
            for (int it = 0; it < F_IT; it++) dst[it] = u32x4_t{0, 0, 0, 0};
        }
    };
    // K and V of tile j into registers, or (DMA) on their way into the tile's stage: in assembly and waited for by hand (kv_landed),
    // because behind the compiler's builtin every LDS read waits for all LDS operations in flight
    auto load_kv = [&](int j) {
        const int n0 = j * BN;
        if constexpr (DMA) {
            const gptr_t kb = uniform_ptr(kbase + (int64_t)n0 * p.k_r), vb = uniform_ptr(vbase + (int64_t)n0 * p.v_r);
            const int last = p.Lk - 1 - n0;
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)((j & 1) * SM::STAGE) + (uint32_t)wave * 1024);
#pragma unroll
            for (int it = 0; it < K_IT; it++) {
                const int row = kr0 + it * K_RPP, row_c = row < last ? row : last;
                const uint32_t ko = (uint32_t)(row_c * (int)p.k_r + kcol_g) * 2, vo = (uint32_t)(row_c * (int)p.v_r + kcol_g) * 2;
                load_lds16<true>(ko, kb, dst + it * K_RPP * 256);
                load_lds16<true>(vo, vb, dst + SM::K_BYTES + it * K_RPP * 256);
            }
            return;
        }
#pragma unroll
        for (int it = 0; it < K_IT; it++) {
            int key = n0 + kr0 + it * K_RPP;
            key = key < p.Lk ? key : p.Lk - 1;
            kreg[it] = *(const u32x4_t *)(kbase + (int64_t)key * p.k_r + kcol);
            // (V rows the same way: a wave's load covers whole rows -- one cache line per row at head dim 64 -- where a
            // (key quad, d chunk) item per thread, as a transposition in registers wants it, touched every line twice)
            vreg[it] = *(const u32x4_t *)(vbase + (int64_t)key * p.v_r + kcol);
        }
    };
    auto load_rest = [&](int j) {
        load_bias(j, breg);
        load_kv(j);
    };
    // registers -> LDS stage `buf`: K and V rows, mask and bias fused (bias where kept, -inf elsewhere)
    auto store_stage = [&](int j, const u32x2_t (&mv)[F_IT], const u32x4_t (&bsrc)[F_IT]) {
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
            u32x4_t bv = bbase ? chunk8_fix<ODD>(bsrc[it], kk, p.Lk) : bsrc[it];
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
    // (this lane's part of the address of a transposing read of the V tile)
    const uint32_t tr_base = TL::tr_base(g, tr_lane(lane));

    // ---- one tile from LDS stage `buf`
    auto compute = [&](int j, int buf) {
        const int n0 = j * BN + kh * BK;
        const uint32_t a_k = lds0 + (uint32_t)(buf * SM::STAGE + kh * BK * TL::ROW_BYTES) + TL::frag_base(a_row, g);
        const uint32_t tr_v = lds0 + (uint32_t)(buf * SM::STAGE + SM::K_BYTES + kh * BK * TL::ROW_BYTES) + tr_base;
        const char *sF = smem + buf * SM::STAGE + 2 * SM::K_BYTES + ((rw * 32 + r) * SM::SF + kh * BK + 8 * g) * 2;
        // scores start from the fused mask+bias tile (exp2 domain)
        f32x16_t s[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const u32x4_t fv = *(const u32x4_t *)(sF + (32 * mb + 16 * blk) * 2);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s[mb][8 * blk + 2 * e] = E::lo(fv[e]) * kLog2e;
                    s[mb][8 * blk + 2 * e + 1] = E::hi(fv[e]) * kLog2e;
                }
            }
        {
            constexpr int NF = MB * KS, FR = NF < 8 ? NF : 8;
            u32x4_t a[NF];
            auto frag = [&](int f) {
                const int ks = f / MB, mb = f % MB;
                return lds_ld128(TL::frag_at(a_k, ks) + (uint32_t)(32 * mb * TL::ROW_BYTES));
            };
#pragma unroll
            for (int f = 0; f < FR; f++) a[f] = frag(f);
#pragma unroll
            for (int f = 0; f < NF; f++) {
                if (f + FR < NF) a[f + FR] = frag(f + FR);
                s[f % MB] = E::mfma(a[f], qf[f / MB], s[f % MB]);
            }
        }
        // causal selects on diagonal tiles only (wave-uniform branch)
        if (CAUSAL && n0 + BK - 1 > wrow0 + shift) {
            asm volatile("" ::: "memory");
            const int lim = qrow + shift - n0 - 8 * g;  // local column limit for this lane
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int lc = 32 * mb + 16 * (i >> 3) + (i & 7);
                    s[mb][i] = lc <= lim ? s[mb][i] : -INFINITY;
                }
        }
        float tmax = -INFINITY;
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int i = 0; i < 16; i++) tmax = fmaxf(tmax, s[mb][i]);
        tmax = xhalf_max(tmax);
        // lazy rescale: the running maximum is only the reference point of the exp2, so it moves (and O and the row
        // sums are rescaled) only when a score exceeds it by more than 2^8 -- rare after the first tiles
        if (__any(tmax > row_max + 8.f)) {
            const float new_max = fmaxf(row_max, tmax);
            const float safe = new_max == -INFINITY ? 0.f : new_max;
            const float alpha = fast_exp2(row_max - safe);
            row_max = new_max;
            row_sum *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= alpha;
        }
        const float m_use = row_max == -INFINITY ? 0.f : row_max;
        float psum = 0.f;
        uint32_t pk[8 * MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                const float p0 = fast_exp2(s[mb][i] - m_use);
                const float p1 = fast_exp2(s[mb][i + 1] - m_use);
                psum += p0 + p1;
                pk[8 * mb + i / 2] = E::pack2(p0, p1);
            }
        row_sum += psum;
        {
            // V^T (rows of the A operand = head dim) through transposing reads of the row-major V tile
            constexpr int NF = KB * DB, FR = NF < 8 ? NF : 8;
            u32x4_t a[NF];
            auto frag = [&](int f) {
                const int kb = f / DB, db = f % DB;
                const u32x2_t lo = lds_ld_tr16(TL::tr_at(tr_v, kb, db, 0)), hi = lds_ld_tr16(TL::tr_at(tr_v, kb, db, 1));
                return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            };
#pragma unroll
            for (int f = 0; f < FR; f++) a[f] = frag(f);
#pragma unroll
            for (int f = 0; f < NF; f++) {
                if (f + FR < NF) a[f + FR] = frag(f + FR);
                const int kb = f / DB, db = f % DB;
                const u32x4_t bop = {pk[4 * kb], pk[4 * kb + 1], pk[4 * kb + 2], pk[4 * kb + 3]};
                o[db] = E::mfma(a[f], bop, o[db]);
            }
        }
    };

    // The end of a step: "has any thread a kept element of that tile", published by the barrier that publishes the step's LDS
    // stores and direct loads.  (The word of vote i is set in front of barrier i, read behind it, and cleared between barriers i + 1
    // and i + 2 for vote i + 3.)  `younger`: mask and bias loads that this wave has issued behind the direct loads that must
    // have landed.
    int vote_at = 0;
    if (tid < 3) lds_st32(lds0 + SM::OFF_VOTE + 4 * tid, 0u);
    auto step_end = [&](bool any, int younger) -> bool {
        const uint32_t at = lds0 + SM::OFF_VOTE + 4 * vote_at;
        vote_at = vote_at == 2 ? 0 : vote_at + 1;
        if (__any(any)) lds_st32(at, 1u);
        if (tid == 0) lds_st32(lds0 + SM::OFF_VOTE + 4 * vote_at, 0u);
        if constexpr (DMA) {
            if (younger >= 2 * F_IT) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(2 * F_IT) : "memory");
            else if (younger >= F_IT) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(F_IT) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        } else {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
        }
        return __builtin_amdgcn_readfirstlane(lds_ld32(at)) != 0u;
    };
    const int n_mask = mbase ? F_IT : 0, n_bias = bbase ? F_IT : 0;

    // ---- main loop.  At the top of iteration j: tile j sits in LDS stage j&1 if it is active, `mreg` holds
    // the mask of tile j+1 and `act_next` says whether that tile has any kept element.
    // DEEP (head dims up to 64, and two waves per row block: where the registers are there): mask and bias -- the bytes that come from HBM -- stay in
    // flight for TWO iterations instead of one.  With one, every iteration contained a whole trip to memory (the mask
    // requested at its top decided, at its end, whether the tile after the next is fetched at all), and the launch moved
    // what it had in flight once per trip: 64 KB per CU every 3.5 us.  Now the mask of tile j+4 and the bias of tile
    // j+2 are requested at the top of iteration j, behind K / V of tile j+1 (cache hits; waiting for those must not
    // mean waiting for the younger requests: loads come back in the order they were issued).
    constexpr bool DEEP = D <= 64 || KSPLIT == 2;
    if (t_first < n_end && DEEP) {
        u32x2_t m1[F_IT], m2[F_IT], m3[F_IT];            // with mreg: the masks of tiles j .. j+3 at the top of iteration j
        u32x4_t b1[F_IT], b2[F_IT];                      // bias of tiles j+1 (requested an iteration ago), j+2
        load_mask(t_first, mreg);
        load_mask(t_first + 1, m1);
        load_mask(t_first + 2, m2);
        load_mask(t_first + 3, m3);
        bool act_cur = __syncthreads_or(finish_mask(t_first, mreg));
        if (act_cur) {
            load_rest(t_first);
            store_stage(t_first, mreg, breg);
        }
        if (DMA) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        bool act_1 = __syncthreads_or(t_first + 1 < n_end && finish_mask(t_first + 1, m1));
        if (act_1) load_bias(t_first + 1, b1);
        bool act_2 = __syncthreads_or(t_first + 2 < n_end && finish_mask(t_first + 2, m2));
        // one iteration; the register sets change roles from one iteration to the next (written out four iterations
        // at a time: a move between sets would have to wait for a load that is still in flight)
        auto step = [&](int j, u32x2_t (&ma)[F_IT], u32x2_t (&mc)[F_IT], u32x2_t (&md)[F_IT], u32x4_t (&ba)[F_IT], u32x4_t (&bb)[F_IT]) {
            // ma: mask of tile j+1 (finished); mc: of tile j+3 (in flight since the iteration before); md: receives tile j+4
            // ba: bias of tile j+1 (requested an iteration ago); bb: receives tile j+2
            const bool have_next = j + 1 < n_end && act_1;
            if (have_next) load_kv(j + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (j + 4 < n_end) load_mask(j + 4, md);
            __builtin_amdgcn_sched_barrier(0);
            if (j + 2 < n_end && act_2) load_bias(j + 2, bb);
            __builtin_amdgcn_sched_barrier(0);
            if (act_cur) compute(j, j & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (have_next) store_stage(j + 1, ma, ba);
            const bool act_3 = step_end(j + 3 < n_end && finish_mask(j + 3, mc), (j + 4 < n_end ? n_mask : 0) + (j + 2 < n_end && act_2 ? n_bias : 0));
            act_cur = have_next;
            act_1 = act_2;
            act_2 = act_3;
        };
#pragma unroll 1
        for (int j = t_first; j < n_end; j += 4) {
            step(j, m1, m3, mreg, b1, b2);  // (mreg, the set of tile j, is free: it receives tile j+4)
            if (j + 1 < n_end) step(j + 1, m2, mreg, m1, b2, b1);
            if (j + 2 < n_end) step(j + 2, m3, m1, m2, b1, b2);
            if (j + 3 < n_end) step(j + 3, mreg, m2, m3, b2, b1);
        }
    } else if (t_first < n_end) {
        load_mask(t_first, mreg);
        if (t_first + 1 < n_end) load_mask(t_first + 1, mnext);
        bool act_cur = __syncthreads_or(finish_mask(t_first, mreg));
        if (act_cur) {
            load_rest(t_first);
            store_stage(t_first, mreg, breg);
        }
        if (DMA) asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        bool act_next = __syncthreads_or(t_first + 1 < n_end && finish_mask(t_first + 1, mnext));
        // one iteration; `m_next` holds the (finished) mask of tile j+1, `m_new` receives the mask of tile j+2.
        // The scheduling barriers keep the loads at the top and their first use below the compute: their
        // latency is then covered by the MFMA work instead of being waited for right away.
        auto step = [&](int j, u32x2_t (&m_next)[F_IT], u32x2_t (&m_new)[F_IT]) {
            const bool have_next = j + 1 < n_end && act_next;
            if (have_next) load_rest(j + 1);
            if (j + 2 < n_end) load_mask(j + 2, m_new);
            __builtin_amdgcn_sched_barrier(0);
            if (act_cur) compute(j, j & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (have_next) store_stage(j + 1, m_next, breg);
            const bool act_nn = step_end(j + 2 < n_end && finish_mask(j + 2, m_new), 0);
            act_cur = have_next;
            act_next = act_nn;
        };
        for (int j = t_first; j < n_end; j += 2) {
            step(j, mnext, mreg);
            if (j + 1 < n_end) step(j + 1, mreg, mnext);
        }
    }

    // ---- epilogue: normalise, store O and LSE
    float total = xhalf_sum(row_sum);
    if constexpr (KSPLIT == 2) {
        // the upper key half hands over its sums and O (relative to its own maximum); the lower half merges and stores
        float *xm = (float *)smem + xw * 64 + lane;                                    // maximum, sum: 2 * RB * GH * 64 floats
        f32x4_t *xo = (f32x4_t *)(smem + 2 * (RB * GH) * 256) + xw * DB * 4 * 64 + lane;
        __syncthreads();  // (the tiles' last reads)
        if (kh == 1) {
            xm[0] = row_max;
            xm[(RB * GH) * 64] = total;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    xo[(db * 4 + q) * 64] = f32x4_t{o[db][4 * q], o[db][4 * q + 1], o[db][4 * q + 2], o[db][4 * q + 3]};
        }
        __syncthreads();
        if (!SHARES && kh == 1) return;
        const float m1 = xm[0], t1 = xm[(RB * GH) * 64];
        const float mx = fmaxf(row_max, m1), safe = mx == -INFINITY ? 0.f : mx;
        const float w0 = fast_exp2(row_max - safe), w1 = fast_exp2(m1 - safe);
        total = total * w0 + t1 * w1;
        row_max = mx;
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
    if constexpr (SHARES) {  // O in fp32 and its log2-sum-exp, which the last workgroup of the rows, or fwd_merge_kernel, adds up
        // (a sum that is no number has to reach the result: only an empty share is left out)
        const float l = total == 0.f ? -INFINITY : row_max + __builtin_amdgcn_logf(total);
        if (!p.dec_counter) {
            if (qrow < p.Lq && kh == 0) {
                const int64_t at = (((int64_t)blockIdx.y * p.B + b) * p.H + h) * p.Lq + qrow;
#pragma unroll
                for (int db = 0; db < DB; db++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int c = 32 * db + 16 * (q >> 1) + 8 * g + 4 * (q & 1);
                        if (c < p.d) *(f32x4_t *)(p.o_part + at * p.d + c) = f32x4_t{o[db][4 * q] * inv, o[db][4 * q + 1] * inv, o[db][4 * q + 2] * inv, o[db][4 * q + 3] * inv};
                    }
                if (g == 0) p.lse_part[at] = l;
            }
            return;
        }
        // (counters: [workgroup][share][wave of the lower half][32-wide block of O][quarter][lane] and [workgroup][share][row])
        constexpr int ROWS = 32 * RB * GH;
        const int64_t first = (int64_t)blockIdx.x * p.splits;
        float *o_lane = p.o_part + first * (ROWS * D) + xw * (32 * D) + lane * 2, *l_lane = p.lse_part + first * ROWS + xw * 32 + r;
        if (kh == 0) {
            float *at = o_lane + (int64_t)blockIdx.y * (ROWS * D);
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    share_store4(at + (db * 4 + q) * 256, f32x4_t{o[db][4 * q] * inv, o[db][4 * q + 1] * inv, o[db][4 * q + 2] * inv, o[db][4 * q + 3] * inv});
            if (g == 0) share_store(l_lane + (int64_t)blockIdx.y * ROWS, l);
        }
        if (!last_share(p.dec_counter + blockIdx.x, p.splits, (int *)(smem + SM::OFF_VOTE)) || kh || qrow >= p.Lq) return;
        bool on[MAX_KEY_SPLITS];
        const ShareWeights sw = lane_share_weights(l_lane, ROWS, p.splits, on);
        uint16_t *op = (uint16_t *)p.o + b * p.o_b + (int64_t)qrow * p.o_r + h * p.o_h;
#pragma unroll 1
        for (int i = 0; i < 2 * DB; i += 4) {
            u32x4_t y[4];
            lane_merged<T, 4>(sw, o_lane + i * 512, ROWS * D, p.splits, on, y);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int c = 16 * (i + u) + 8 * g;
                if (c < p.d) *(u32x4_t *)(op + c) = y[u];
            }
        }
        if (g == 0) p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = sw.lse;
        return;
    }
    if (qrow < p.Lq) {
        uint16_t *op = (uint16_t *)p.o + b * p.o_b + (int64_t)qrow * p.o_r + h * p.o_h;
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
            const float lse = total > 0.f ? (row_max + __builtin_amdgcn_logf(total)) * kLn2 : INFINITY;
            p.lse[((int64_t)b * p.H + h) * p.Lq + qrow] = lse;
        }
    }
}

template <typename T, int D, bool CAUSAL, int NW, int KSPLIT, int GH, bool ODD, bool SHARES = false>
hipError_t launch_fwd_o(const FwdParams &p, hipStream_t stream) {
    constexpr int BM = 32 * NW / KSPLIT / GH, NTHREADS = 64 * NW, BN = D > 128 ? 32 : BN_DEFAULT;
    if constexpr (!SHARES) {
        if (p.splits > 1) {
            if constexpr (KSPLIT == 2 || NW == 4) return launch_fwd_o<T, D, CAUSAL, NW, KSPLIT, GH, ODD, true>(p, stream);
            else return hipErrorInvalidValue;  // (general_key_shares plans none for the kernels of 256 rows)
        }
    }
    auto kern = fwd_kernel<T, D, CAUSAL, NW, BN, KSPLIT, GH, ODD, SHARES>;
    constexpr int merge = KSPLIT == 2 ? (NW / 2) * 512 + (NW / 2) * (D / 32) * 4096 : 0;  // the upper halves' sums
    constexpr int smem = FwdSmem<D, BM, BN>::TOTAL > merge ? FwdSmem<D, BM, BN>::TOTAL : merge;
    static DynSmemLimit smem_limit;
    hipError_t e = smem_limit.ensure((const void *)kern, (int)smem);
    if (e != hipSuccess) return e;
    dim3 grid(((p.Lq + BM - 1) / BM) * (p.H / GH) * p.B);
    if constexpr (SHARES) grid.y = p.splits;
    hipLaunchKernelGGL(kern, grid, dim3(NTHREADS), smem, stream, p);
    return hipGetLastError();
}

template <typename T, int D, bool CAUSAL, int NW, int KSPLIT = 1>
hipError_t launch_fwd_c(const FwdParams &p, hipStream_t stream) {
    const int gh = shared_rows(p);
    // (at d = 65 .. 128 whole aligned chunks / rows read where they lie, us: 2000 tokens x 16/8 heads 54.7 / 56.4, x 16/4 52.9 / 53.7,
    // 1024 x 16/8, causal 30.9 / 31.6)
    auto pick = [&](auto odd) -> hipError_t {
        constexpr bool O = decltype(odd)::value;
        if constexpr (D <= 128) if (gh == 4) return launch_fwd_o<T, D, CAUSAL, NW, KSPLIT, 4, O>(p, stream);
        if constexpr (D > 64) if (gh == 2) return launch_fwd_o<T, D, CAUSAL, NW, KSPLIT, 2, O>(p, stream);
        return launch_fwd_o<T, D, CAUSAL, NW, KSPLIT, 1, O>(p, stream);
    };
    if (D > 128 || odd_rows(p)) return pick(std::true_type());
    return pick(std::bool_constant<(D > 128)>());
}

template <typename T, int D>
hipError_t launch_fwd_t(const FwdParams &p, hipStream_t stream) {
    if constexpr (D > 64 && D <= 128) {
        if (general_rows_256(p))
            return p.causal ? launch_fwd_c<T, D, true, 8>(p, stream) : launch_fwd_c<T, D, false, 8>(p, stream);
        return p.causal ? launch_fwd_c<T, D, true, 8, 2>(p, stream) : launch_fwd_c<T, D, false, 8, 2>(p, stream);
    } else {
        return p.causal ? launch_fwd_c<T, D, true, 4>(p, stream) : launch_fwd_c<T, D, false, 4>(p, stream);
    }
}

}  // namespace

// Query heads per workgroup: 4 or 2 of a kv group, where they share mask and bias rows.  One head / four (us): 1999 x 16/4 heads, d = 128,
// fp16 70.8 / 57.3, 1231 x 8/2 44.8 / 34.8; d = 64, 4 x 724 x 32/8 39.5 / 28.8, 4096 x 8/2 120 / 107.  Two: d = 128, 2 x 2112 x 8/4
// 62.7 / 57.7, d = 256, 700 x 32/8 59.2 / 55.2 (four would leave each 32 rows); not at d <= 64 (1984 x 16/8 61.2 / 65.2).
int shared_rows(const FwdParams &p) {
    const int G = p.H / p.Hk;
    if (G > 1 && ((p.mask && p.Hm == p.H) || (p.bias && p.Hb == p.H))) return 1;
    if (p.d <= 128 && G % 4 == 0) return 4;
    return p.d > 64 && G % 2 == 0 ? 2 : 1;
}

// At head dims 65 to 128, forward and dQ: 256-row workgroups while the grid still covers the chip about twice
bool general_rows_256(const FwdParams &p) { return p.d > 64 && p.d <= 128 && (int64_t)p.B * p.H * ((p.Lq + 255) / 256) >= 512; }

int64_t general_share_units(const FwdParams &p) {
    const int gh = shared_rows(p), rows = 128 / gh;
    return (int64_t)((p.Lq + rows - 1) / rows) * (p.H / gh) * p.B;
}

// Shares that the key tiles of a row block are cut into, forward and dQ.  A workgroup's time is its chain of tiles (1.5 us each at head dims up
// to 128, 2.5 per 32 keys above), and few heads or short rows leave most CUs without one.
//   * As many as the chip holds workgroups at once (one per CU; d <= 64: two, three of 32-row ones), rounded DOWN: 64 blocks of 1000 rows,
//     d = 128: 4 shares 25.1 us, 5 31.5; 188 blocks 43.1 whole, 48.4 in three.
//   * Four tiles each at least, and at head dims 65 to 128, where a tile takes 1.1 us, twelve in all: below, the fp32 results, written and
//     read again, and the launch that adds them up cost more than the tiles (d = 128, whole / in two: 4 x 300 x 8/4 16.6 / 21.8,
//     4 x 478 x 8/4 19.8 / 23.3; d = 64, 2 x 704 x 16/16 25.8 / 23.5); above 128 twelve where there are more than CUs / 4 blocks (4 x 256
//     x 16/8 125 / 130 with the backward, 256 x 2/1 24.5 / 21.4).
//   * dQ from 24 tiles on (16 of 32 keys): below, a backward is bound by its launches, of which this is one more (1024 x 2/1,
//     d = 128: 66.9 and 69 to 72).
//   * None where the kernels of 256 rows take the call: they work on whole keys.
// (Up to head dim 128 the last workgroup of the rows adds the forward's shares up; a launch of its own: 3883 x 8/2, d = 64 66.7 / 55.9, 2 x 1198 x
// 8/4, d = 64 30.6 / 26.9, 2 x 1039 x 8/2 24.5 / 21.0.)
// Whole / shares, us (forward; backward with its other kernels): 2316 x 2/1 heads, d = 256 162 / 46, 323 / 180; 3000 x 2/1, d = 64 83 / 25,
// 141 / 75; 2240 x 2/1, d = 96 56 / 24, 107 / 72; 4096 x 2/1, d = 128 98 / 39, 172 / 106; 3000 x 8/2, d = 64 81 / 41, 198 / 171; 1999 x 8/4,
// not causal 61 / 43, 138 / 119.  Rows that are not whole chunks, in instantiations of their own (forward; backward without a bias): 2999 x 2/1, d = 64
// 101 / 28, 143 / 69; 2239 x 2/1, d = 96 60 / 28, 104 / 64; 4095 x 2/2, d = 128 130 / 48, 182 / 102; 3001 x 8/2, d = 64 85 / 45, 177 / 135.
int general_key_shares(const FwdParams &p, bool dq) {
    if (p.cu_q || p.Lq < 1 || p.Lk < 1) return 1;
    const int gh = shared_rows(p), tile = p.d > 128 ? 32 : 64, tiles = (p.Lk + tile - 1) / tile;
    if (general_rows_256(p) || (dq && tiles < (p.d > 128 ? 16 : 24))) return 1;
    const int64_t blocks = general_share_units(p);
    int64_t s = blocks > 0 ? device_cus() * (p.d > 64 ? 1 : (gh == 4 ? 3 : 2)) / blocks : 1;
    if (s > tiles / 4) s = tiles / 4;
    if (p.d > 64 && tiles < 12 && (p.d <= 128 || 4 * blocks > device_cus())) return 1;
    return s < 2 ? 1 : (s > MAX_KEY_SPLITS ? MAX_KEY_SPLITS : (int)s);
}

hipError_t launch_fwd(const FwdParams &p, int dtype, hipStream_t stream) {
    if (p.Lq <= 0 || p.B <= 0) return hipSuccess;
    if (fwd_colmask_applicable(p)) return launch_fwd_colmask(p, dtype, stream);
    // head dims up to 64 / 128 / 256 (a head dim in between runs in the next larger instantiation)
    const hipError_t e = dtype == 0 ? (p.d <= 64 ? launch_fwd_t<bf16_tag, 64>(p, stream) : p.d <= 128 ? launch_fwd_t<bf16_tag, 128>(p, stream) : launch_fwd_t<bf16_tag, 256>(p, stream))
                                    : (p.d <= 64 ? launch_fwd_t<fp16_tag, 64>(p, stream) : p.d <= 128 ? launch_fwd_t<fp16_tag, 128>(p, stream) : launch_fwd_t<fp16_tag, 256>(p, stream));
    return e != hipSuccess || p.splits <= 1 || p.dec_counter ? e : launch_fwd_merge(p, dtype, stream);
}

}  // namespace fdma
