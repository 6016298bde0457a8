// Backward dynamic-mask attention for gfx950, general form (mask and / or bias vary per query row), head dims 65 .. 128:
// the dK / dV / dBias kernel.
//
// Same math and reference counterparts as fdma_bwd.hip (compute_dq_dk_dv_1colblock,
// csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the reference), laid out for what a head dim of 128 costs: the
// dK / dV accumulators of 32 keys alone are 128 registers per lane, and the tiles leave room for one workgroup per CU.  With
// four waves (one per SIMD, nothing to hide behind) a step of 64 query rows x 128 keys took 4.9 us for 0.85 us of matrix
// work.
//
// Here a workgroup is 8 waves over 128 keys: wave (kw, qh) takes 32 keys and HALF of a step's 64 query rows.
//   * Q, dO and the row statistics go from global memory straight into LDS (global_load_lds, issued between the MFMAs a
//     step ahead): no staging registers.  K and V are parked in LDS for the whole launch.  What is left in registers --
//     accumulators, one score and one dP tile, fragments -- fits the 256 that two waves per SIMD have.
//   * The fused bias tile (bias where the mask keeps, -inf elsewhere, beyond Lq, beyond Lk and above the causal diagonal:
//     the inner loop has no selects) has ONE stage.  A thread fetches its 8-key chunks of the next step's bias and mask at
//     the top of a step; dS replaces the elements it was computed from; behind the step's first barrier the same thread
//     writes its chunk of dS to dBias and puts the next step's chunk in its place.
//   * At the end the two query halves exchange sums through LDS: wave (kw, 0) finishes dK, wave (kw, 1) dV.
// LDS: 2 x 32.5 KB of Q / dO, 64 KB of K / V, 17 KB fused bias.  Bound by LDS reads: 384 KB per step, 3000 clocks at 128
// bytes a clock, against 2050 of matrix work.
//
// A workgroup's work grows with Lq * G and there are only ceil(Lk / 128) * Hk * B of them: where they do not fill the chip
// the query blocks are cut into `kv_segs` segments (general_kv_segments), every segment a workgroup that leaves fp32 sums
// which bwd_dkdv_sum_kernel (fdma_bwd.hip) adds in segment order.
// B = 1, L = 1999, H = 16, Hk = 4, d = 128, fp16, mask and bias rows shared by the group: 630 us as 64 workgroups of four
// waves, 112 + 7 (sums) as 256 of eight; B = 1, L = 4096, H = Hk = 16, bf16, causal: 320 -> 210 us.
// Positions and bases are kept up from step to step and a lane's offsets are two registers: with divisions of the step's number and
// the addresses made from scratch a third of the vector instructions of a step were for that.  The first call 116 -> 103 us, 3000 x 8/8,
// d = 96 122 -> 111, 2048 x 16/4 83 -> 72, 2 x 700 x 8/2 with one bias value per key 49 -> 41.
// (Wave pairs that share keys by role, as at head dim 256, with P through LDS: 122 us, and 130 with a pair half a step apart: the 32
// rows of softmax per lane and the sums over heads want the registers that the roles free.)
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int D = 128;
constexpr int NT = 512;
constexpr int BM = 64;    // query rows per step
constexpr int BN = 128;   // keys per workgroup
constexpr int KS = D / 16, DB = D / 32;
using TL = LdsTile<D>;

constexpr int TILE = BM * TL::ROW_BYTES;              // a Q or dO tile
constexpr int STAGE = 2 * TILE + 2 * BM * 4;          // Q, dO, LSE, D
constexpr int OFF_K = 2 * STAGE;
constexpr int OFF_V = OFF_K + BN * TL::ROW_BYTES;
constexpr int OFF_FB = OFF_V + BN * TL::ROW_BYTES;
constexpr int SB = BN + 8;                            // row stride of the fused tile (elements)
constexpr int OFF_COL = OFF_FB + BM * SB * 2;
constexpr int SMEM = OFF_COL + 2 * 2 * BN * 4;        // dBias column sums: [step parity][query half][key]
static_assert(2 * BN * D * 4 <= OFF_COL, "the halves' sums are exchanged through the tiles' LDS");
static_assert(STAGE % 256 == 0, "stages keep the bank alignment the swizzle is made for");
static_assert(SMEM <= 160 * 1024, "one workgroup per CU");

template <typename T> struct NegInfPair;
template <> struct NegInfPair<bf16_tag> { static constexpr uint32_t value = 0xFF80FF80u; };
template <> struct NegInfPair<fp16_tag> { static constexpr uint32_t value = 0xFC00FC00u; };

template <typename T, bool CAUSAL, bool GSUM, bool ODD>
__global__ void __launch_bounds__(NT) bwd_dkdv_wide_kernel(const BwdParams p) {
    using E = Elem<T>;
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int kw = wave & 3, qh = wave >> 2;  // 32-key group and query half of this wave
    // linear workgroup id -> (key block, segment, kv head, batch), key block OUTERMOST and ascending: under causal masking
    // the low key blocks are seen by the most queries, so the heaviest workgroups of every head start first
    const int hb_count = f.Hk * f.B, segs = p.kv_segs, part_id = (int)blockIdx.x;
    const int n_block = part_id / (hb_count * segs), seg = (part_id / hb_count) % segs, hk = (part_id % hb_count) % f.Hk, b = (part_id % hb_count) / f.Hk;
    const int G = f.H / f.Hk;
    const int n0 = n_block * BN;
    const int key = n0 + kw * 32 + r;  // the key column this lane owns
    const int shift = f.Lk - f.Lq;

    const int M_blocks = (f.Lq + BM - 1) / BM;
    int m_start = 0;
    if (CAUSAL) {
        const int first_q = n0 - shift;  // first query row that sees key n0
        if (first_q > 0) m_start = first_q / BM;
        if (m_start > M_blocks) m_start = M_blocks;
    }
    // this workgroup's segment of the query blocks that see its keys, walked from the last one down so that neighbouring
    // workgroups stream the same tiles together
    const int m_lo = (M_blocks - m_start) * seg / segs, n_m = (M_blocks - m_start) * (seg + 1) / segs - m_lo;
    const int n_steps = n_m * G;

    const bool has_bias = f.bias != nullptr;
    const bool bias_rows = has_bias && f.bi_r != 0;   // per-query bias (and dbias) rows
    const bool use_accum = p.dbias_accum != nullptr;   // several workgroups share a dbias element
    // per-query dbias wants (m outer, g inner) to sum dS over the group in registers; row-broadcast dbias wants
    // (g outer, m inner) to keep one column sum per bias head: see `advance`
    // a fused tile that all query heads of the group share stays for its G steps: its inputs are fetched once, at the first
    // of them (G - 1 more steps until they are needed), and it is replaced -- by dS, then by the next tile -- at the last
    const bool hold = GSUM && bias_rows && f.Hb != f.H && (!f.mask || f.Hm != f.H);
    const int mi_last = M_blocks - m_lo - n_m;
    auto advance = [&](int &gi, int &mi) {  // (without branches: they would put the positions on the stack)
        const bool wrap = bias_rows ? gi == G - 1 : mi == mi_last;
        const int gt = bias_rows && wrap ? 0 : gi + (bias_rows || wrap ? 1 : 0);
        mi = !bias_rows && wrap ? M_blocks - 1 - m_lo : mi - (!bias_rows || wrap ? 1 : 0);
        gi = gt;
    };

    const bool per_head = f.Hb == f.H;
    // zero the part of a per-query dbias this workgroup owns but never visits (above the causal diagonal)
    if (bias_rows && !use_accum && m_start > 0 && seg == 0) {
        const int ngh = (f.Hb == f.H) ? G : 1;
        for (int gh = 0; gh < ngh; gh++) {
            const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
            uint16_t *dbp = (uint16_t *)p.dbias + b * p.db_b + hb * p.db_h;
            const int rows = m_start * BM < f.Lq ? m_start * BM : f.Lq;
            for (int idx = tid; idx < rows * 16; idx += NT) {
                const int row = idx >> 4, kk = n0 + (idx & 15) * 8;
                if (kk < f.Lk) *(u32x4_t *)(dbp + (int64_t)row * p.db_r + kk) = u32x4_t{0, 0, 0, 0};
            }
        }
    }

    // ---- K and V rows of the 128 keys -> LDS (chunks beyond d and rows beyond Lk as zeros: they meet clamped Q / dO
    // chunks and end in accumulators that are not stored)
    for (int i = tid; i < BN * 16; i += NT) {
        const int row = i >> 4, c = i & 15;
        u32x4_t kv = {0, 0, 0, 0}, vv = {0, 0, 0, 0};
        if (n0 + row < f.Lk && c * 8 < f.d) {
            kv = *(const u32x4_t *)((const uint16_t *)f.k + b * f.k_b + (int64_t)(n0 + row) * f.k_r + hk * f.k_h + c * 8);
            vv = *(const u32x4_t *)((const uint16_t *)f.v + b * f.v_b + (int64_t)(n0 + row) * f.v_r + hk * f.v_h + c * 8);
        }
        *(u32x4_t *)(smem + OFF_K + TL::chunk(row, c)) = kv;
        *(u32x4_t *)(smem + OFF_V + TL::chunk(row, c)) = vv;
    }

    // ---- direct loads of a step's tiles: load n = 2 * wave + i of a tile fills LDS bytes [1024 n, 1024 n + 1024), i.e.
    // rows 4n .. 4n+3, lane l the chunk POSITION l % 16 of row 4n + l / 16 -- which holds chunk position ^ swz(row) of the
    // global row.  One more 4-byte load per wave: the 64 LSE values (even waves) or D values (odd waves).
    // bases of the group's first head, and bytes from one head, and one row, to the next
    const int h0 = hk * G;
    const int64_t q_h2 = f.q_h * 2, do_h2 = p.do_h * 2;
    const char *q_base = (const char *)((const uint16_t *)f.q + b * f.q_b + h0 * f.q_h), *do_base = (const char *)((const uint16_t *)p.dout + b * p.do_b + h0 * p.do_h);
    const int st_h = wave & 1 ? p.Lq_rounded : f.Lq;
    const float *st_base = (wave & 1 ? p.softmax_d : f.lse) + ((int64_t)b * f.H + h0) * st_h;
    // offsets of this lane's pieces: its row (clamped per step: offsets grow with the row), its two columns
    const uint32_t q_r2 = (uint32_t)(f.q_r * 2), do_r2 = (uint32_t)(p.do_r * 2);
    uint32_t q_row, do_row, pcol[2];
    {
        const int row = 8 * wave + (lane >> 4);
        q_row = row * q_r2;
        do_row = row * do_r2;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int chunk = (lane & 15) ^ (int)TL::swz(row + 4 * i);
            pcol[i] = chunk * 8 < f.d ? chunk * 16 : 0;
        }
    }
    auto least = [](uint32_t x, uint32_t y) { return x < y ? x : y; };
    gptr_t ld_q = nullptr, ld_do = nullptr, ld_stat = nullptr;
    uint32_t ld_rows = 0;  // last existing row of the step being fetched
    uint32_t ld_dst = 0;
    auto dma_begin = [&](int gi, int m0, int buf) {
        ld_q = uniform_ptr(q_base + gi * q_h2 + (int64_t)m0 * q_r2);
        ld_do = uniform_ptr(do_base + gi * do_h2 + (int64_t)m0 * do_r2);
        ld_stat = uniform_ptr(st_base + gi * st_h + m0);
        const int left = f.Lq - 1 - m0;
        ld_rows = (uint32_t)(left < BM - 1 ? left : BM - 1);
        ld_dst = lds0 + buf * STAGE;
    };
    // (written in assembly and waited for by hand, as in fdma_bwd_colmask.hip: behind the compiler's builtin every LDS read
    // waits for all LDS operations in flight.  m0 carries the LDS address.)
    auto dma_piece = [&](int n) {
        if (n < 4) {
            const int i = n & 1;
            const uint32_t r2 = n < 2 ? q_r2 : do_r2;
            const uint32_t off = least((n < 2 ? q_row : do_row) + 4 * i * r2, ld_rows * r2) + pcol[i];
            load_lds16(off, n < 2 ? ld_q : ld_do, __builtin_amdgcn_readfirstlane(ld_dst + (n < 2 ? 0 : TILE) + (2 * wave + i) * 1024));
        } else {
            load_lds4(least((uint32_t)lane, ld_rows) * 4, ld_stat, __builtin_amdgcn_readfirstlane(ld_dst + 2 * TILE + (wave & 1) * BM * 4));
        }
    };

    // ---- this thread's chunks of the fused tile: keys n0 + 8 bc .. + 7 of rows br0 and br0 + 32
    // (row and key of the chunks; made opaque at every step, or the compiler keeps every address derived from them in
    // registers that the loop does not have)
    const int bc = tid & 15;
    int br0 = tid >> 4, kk = n0 + 8 * bc;
    u32x4_t braw[2];
    u32x2_t mraw[2];
    // Every load is unconditional and raw (clamped rows / keys; an absent mask or bias is read from K, any valid address,
    // and ignored later): nothing looks at a value before the step's first barrier.
    const int hm0 = f.Hm == 1 ? 0 : f.Hm == f.H ? h0 : hk, hb0 = f.Hb == 1 ? 0 : f.Hb == f.H ? h0 : hk;
    const uint8_t *m_base = !f.mask ? (const uint8_t *)f.k : f.mbits ? f.mbits + b * f.mb_b + hm0 * f.mb_h : f.mask + b * f.m_b + hm0 * f.m_h;
    const int64_t m_h1 = f.mask && f.Hm == f.H ? (f.mbits ? f.mb_h : f.m_h) : 0, m_r1 = f.mask ? (f.mbits ? f.mb_r : f.m_r) : 0;
    const uint16_t *bi_base = has_bias ? (const uint16_t *)f.bias + b * f.bi_b + hb0 * f.bi_h : (const uint16_t *)f.k;
    const int64_t bi_h1 = has_bias && per_head ? f.bi_h : 0, bi_r1 = has_bias ? f.bi_r : 0;
    auto fb_load = [&](int gi, int m0) {
        asm volatile("" : "+v"(br0), "+v"(kk));
        const int at = chunk8_at<ODD>(kk, f.Lk), m_at = !f.mask ? 0 : f.mbits ? ((kk < f.Lk ? kk : 0) >> 3) & ~7 : at, b_at = has_bias ? at : 0;
        const uint8_t *mp = m_base + gi * m_h1 + m0 * m_r1;
        const uint16_t *bp = bi_base + gi * bi_h1 + m0 * bi_r1;
#pragma unroll
        for (int it = 0; it < 2; it++) {
            int row = br0 + 32 * it;
            row = row < f.Lq - m0 ? row : f.Lq - 1 - m0;
            braw[it] = *(const u32x4_el_t *)(bp + (row * bi_r1 + b_at));
            mraw[it] = *(const u32x2_any_t *)(mp + (row * m_r1 + m_at));
        }
    };
    const uint32_t fb_chunk = lds0 + OFF_FB + (br0 * SB + 8 * bc) * 2;
    auto fb_store = [&](int m0) {
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int qq = m0 + br0 + 32 * it;
            u32x4_t bv = has_bias ? chunk8_fix<ODD>(braw[it], kk, f.Lk) : u32x4_t{0, 0, 0, 0};
            u32x2_t mv = f.mask ? (f.mbits ? mask_bits_to_bytes(mask_bits_byte(mraw[it], kk < f.Lk ? kk : 0)) : chunk8_fix_mask<ODD>(mraw[it], kk, f.Lk)) : u32x2_t{0x01010101u, 0x01010101u};
            // keys of the chunk this row may see
            int n = (CAUSAL && qq + shift + 1 < f.Lk ? qq + shift + 1 : f.Lk) - kk;
            n = qq < f.Lq ? n : 0;
            const uint64_t keepm = n >= 8 ? ~0ull : (n <= 0 ? 0ull : (1ull << (8 * n)) - 1ull);
            mv[0] &= (uint32_t)keepm;
            mv[1] &= (uint32_t)(keepm >> 32);
#pragma unroll
            for (int hlf = 0; hlf < 2; hlf++) {
                uint32_t x = mv[hlf];
                x = ((((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) >> 7) & 0x01010101u;  // nonzero byte -> 0x01
                const uint32_t z = (x << 8) - x;                                      // 0x01 -> 0xFF per byte
                const uint32_t m0w = __builtin_amdgcn_perm(0, z, 0x01010000u);        // [b0 b0 b1 b1]
                const uint32_t m1w = __builtin_amdgcn_perm(0, z, 0x03030202u);        // [b2 b2 b3 b3]
                bv[2 * hlf] = (bv[2 * hlf] & m0w) | (NegInfPair<T>::value & ~m0w);
                bv[2 * hlf + 1] = (bv[2 * hlf + 1] & m1w) | (NegInfPair<T>::value & ~m1w);
            }
            *(__attribute__((address_space(3))) u32x4_t *)(uintptr_t)(fb_chunk + 32 * it * SB * 2) = bv;
        }
    };

    f32x16_t dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) { dk[db][i] = 0.f; dv[db][i] = 0.f; }

    // fragment addresses (see LdsTile): Q / dO rows of this wave's half, K / V rows of its keys
    uint32_t a_off = lds0 + 32 * qh * TL::ROW_BYTES + TL::frag_base(pi_row(r), g);
    uint32_t kv_off = lds0 + OFF_K + TL::frag_base(kw * 32 + r, g);
    const TrLane tr = tr_lane(lane);
    uint32_t tr_off = lds0 + 32 * qh * TL::ROW_BYTES + TL::tr_base(g, tr);
    const uint32_t stat_off = lds0 + 2 * TILE + (32 * qh + 8 * g) * 4;
    // fused tile: rows 32 qh + 16 blk + 8 g + .., this lane's column.  Read through transposing reads (lane (te, tc) of 16
    // supplies four elements of row te, lane i receives rows 0 .. 3 of column i), written back element by element.
    const uint32_t fb_tr = lds0 + OFF_FB + ((32 * qh + 8 * g + tr.te) * SB + kw * 32 + 16 * tr.tdh + 4 * tr.tc) * 2;
    uint16_t *fb_col = (uint16_t *)(smem + OFF_FB) + (32 * qh + 8 * g) * SB + kw * 32 + r;
    float *s_col = (float *)(smem + OFF_COL);

    float colsum = 0.f;  // row-broadcast dbias: sum over queries of dS for this lane's key
    float dsum[GSUM ? 16 : 1];  // per-query dbias with bias heads < H: sum over the group
    if (GSUM) {
#pragma unroll
        for (int i = 0; i < 16; i++) dsum[GSUM ? i : 0] = 0.f;
    }

    int gi = 0, mi = M_blocks - 1 - m_lo;
    if (n_steps > 0) {
        fb_load(0, mi * BM);
        dma_begin(0, mi * BM, 0);
#pragma unroll
        for (int n = 0; n < 5; n++) dma_piece(n);
        fb_store(mi * BM);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __syncthreads();

    auto one_step = [&](auto buf_c, const int step) {
        constexpr int buf = decltype(buf_c)::value;
        const int m0 = mi * BM;
        const int hb = per_head ? h0 + gi : hb0;
        // the next step (past the last one its tiles are fetched again and dropped), and the step of the next fused tile
        int gn = gi, mn = mi;
        advance(gn, mn);
        gn = step + 1 < n_steps ? gn : gi;
        mn = step + 1 < n_steps ? mn : mi;
        // (the swizzled addresses are these constants XOR a compile-time value, recomputed where used: hoisted they would
        // cost registers)
        asm volatile("" : "+v"(a_off), "+v"(tr_off), "+v"(kv_off));
        const bool fb_in = !hold || gi == 0, fb_out = !hold || gi == G - 1;  // this step fetches / replaces a fused tile
        const int f_gi = hold ? 0 : gn, f_m0 = (hold ? (mi > mi_last ? mi - 1 : mi) : mn) * BM;
        if (fb_in) fb_load(f_gi, f_m0);
        dma_begin(gn, mn * BM, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);

        // ---- S = Q K^T and dP = dO V^T (M = query, N = key)
        f32x16_t s, dp;
#pragma unroll
        for (int i = 0; i < 16; i++) { s[i] = 0.f; dp[i] = 0.f; }
        {
            constexpr int FR = 1;  // k-steps whose four fragments are read ahead (two: 7 to 60 spilled registers)
            u32x4_t a[KS][2], w[KS][2];
            auto frags = [&](int ks) {
#pragma unroll
                for (int x = 0; x < 2; x++) {
                    a[ks][x] = lds_ld128(TL::frag_at(a_off, ks) + (uint32_t)(buf * STAGE + x * TILE));
                    w[ks][x] = lds_ld128(TL::frag_at(kv_off, ks) + (uint32_t)(x * (OFF_V - OFF_K)));
                }
            };
#pragma unroll
            for (int ks = 0; ks < FR; ks++) frags(ks);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                if (ks + FR < KS) frags(ks + FR);
                s = E::mfma(a[ks][0], w[ks][0], s);
                dp = E::mfma(a[ks][1], w[ks][1], dp);
                if (ks < 5) dma_piece(ks);
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // ---- P = exp2((S*scale + fused)*log2e - LSE*log2e) ; dS = P * (dP - D), 16 query rows (8 per lane) at a time
        if (GSUM && (f.Hb == f.H || gi == 0)) {                  // this step starts a sum over the group
#pragma unroll
            for (int i = 0; i < 16; i++) dsum[GSUM ? i : 0] = 0.f;
        }
        const bool dsum_last = f.Hb == f.H || gi == G - 1;       // ... ends one
        uint32_t ppk[8], dpk[8];
        float part = 0.f;
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
            const uint32_t so = buf * STAGE + 16 * blk * 4;
            const f32x4_t l0 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so)), l1 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + 16));
            const f32x4_t d0 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + BM * 4)), d1 = __builtin_bit_cast(f32x4_t, lds_ld128(stat_off + so + BM * 4 + 16));
            const u32x2_t fb0 = lds_ld_tr16(fb_tr + 16 * blk * SB * 2), fb1 = lds_ld_tr16(fb_tr + (16 * blk + 4) * SB * 2);
            float pv[8], dsv[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t fw = e < 4 ? fb0[(e >> 1) & 1] : fb1[(e >> 1) & 1];
                const float fb = (e & 1) ? E::hi(fw) : E::lo(fw);
                const float lse = e < 4 ? l0[e & 3] : l1[e & 3], dd = e < 4 ? d0[e & 3] : d1[e & 3];
                const float x = __builtin_fmaf(__builtin_fmaf(s[8 * blk + e], f.scale, fb), kLog2e, -lse * kLog2e);
                pv[e] = fast_exp2(x);
                dsv[e] = (dp[8 * blk + e] - dd) * pv[e];
            }
            if (GSUM && bias_rows) {
#pragma unroll
                for (int e = 0; e < 8; e++) dsum[GSUM ? 8 * blk + e : 0] += dsv[e];
            } else if (!bias_rows) {
#pragma unroll
                for (int e = 0; e < 8; e++) part += dsv[e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                ppk[4 * blk + e] = E::pack2(pv[2 * e], pv[2 * e + 1]);
                dpk[4 * blk + e] = E::pack2(dsv[2 * e], dsv[2 * e + 1]);
            }
            if (!GSUM && bias_rows && !use_accum) {  // dS replaces the fused elements this lane has just read
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    fb_col[(16 * blk + 2 * e) * SB] = (uint16_t)(dpk[4 * blk + e] & 0xffffu);
                    fb_col[(16 * blk + 2 * e + 1) * SB] = (uint16_t)(dpk[4 * blk + e] >> 16);
                }
            }
        }

        // ---- dV^T += dO^T P ; dK^T += Q^T dS (M = d, N = key, contraction = query): fragments one pair ahead
        {
            constexpr int NP = 2 * DB;
            u32x4_t a1[2], a2[2];
            auto tr_frag = [&](int idx, int slot) {
                const int qb = idx / DB, db = idx % DB;
                const uint32_t lo_a = TL::tr_at(tr_off, qb, db, 0) + buf * STAGE, hi_a = TL::tr_at(tr_off, qb, db, 1) + buf * STAGE;
                const u32x2_t lo = lds_ld_tr16(lo_a + TILE), hi = lds_ld_tr16(hi_a + TILE);
                const u32x2_t lo2 = lds_ld_tr16(lo_a), hi2 = lds_ld_tr16(hi_a);
                a1[slot] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
                a2[slot] = u32x4_t{lo2[0], lo2[1], hi2[0], hi2[1]};
            };
            tr_frag(0, 0);
#pragma unroll
            for (int idx = 0; idx < NP; idx++) {
                if (idx + 1 < NP) tr_frag(idx + 1, (idx + 1) & 1);
                const int qb = idx / DB, db = idx % DB;
                const u32x4_t pb = {ppk[4 * qb], ppk[4 * qb + 1], ppk[4 * qb + 2], ppk[4 * qb + 3]};
                const u32x4_t sb = {dpk[4 * qb], dpk[4 * qb + 1], dpk[4 * qb + 2], dpk[4 * qb + 3]};
                dv[db] = E::mfma(a1[idx & 1], pb, dv[db]);
                dk[db] = E::mfma(a2[idx & 1], sb, dk[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // ---- dBias, next fused tile
        if (GSUM && bias_rows && dsum_last) {  // (behind the matrix work: the registers of the scores are free again)
            if (use_accum) {
                int gg = g;
                asm volatile("" : "+v"(gg));
                float *ap = p.dbias_accum + b * p.dba_b + hb * p.dba_h + (int64_t)(m0 + 32 * qh + 8 * gg) * p.dba_r + key;
                const int rows = f.Lq - (m0 + 32 * qh + 8 * gg);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int row = 16 * (i >> 3) + (i & 7);
                    if (row < rows && key < f.Lk) atomicAdd(ap + row * p.dba_r, dsum[GSUM ? i : 0]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    const uint32_t wv = E::pack2(dsum[GSUM ? i : 0], dsum[GSUM ? i + 1 : 0]);
                    fb_col[(16 * (i >> 3) + (i & 7)) * SB] = (uint16_t)(wv & 0xffffu);
                    fb_col[(16 * (i >> 3) + (i & 7) + 1) * SB] = (uint16_t)(wv >> 16);
                }
            }
        }
        const bool tile_out = bias_rows && !use_accum && (!GSUM || dsum_last);
        const bool col_out = has_bias && !bias_rows && mi == mi_last && (f.Hb == f.H || gi == G - 1);
        if (has_bias && !bias_rows) {
            colsum += part;
            if (col_out) {
                const float tot = xhalf_sum(colsum);
                if (g == 0) s_col[((step & 1) * 2 + qh) * BN + kw * 32 + r] = tot;
                colsum = 0.f;
            }
        }
        // (every fused element has been read and every dS of the tile written; this wave's loads of the next step have
        // arrived -- waited for here, in front of the stores, so that the stores need not be waited for)
        __builtin_amdgcn_s_waitcnt(0x0070);
        if (fb_out) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (tile_out) {
            uint16_t *dbp = (uint16_t *)p.dbias + b * p.db_b + hb * p.db_h;
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const int qq = m0 + br0 + 32 * it;
                const u32x4_t v = lds_ld128(fb_chunk + 32 * it * SB * 2);
                if (qq < f.Lq && kk < f.Lk) *(u32x4_t *)(dbp + ((int64_t)qq * p.db_r + kk)) = v;
            }
        }
        if (fb_out) fb_store(f_m0);
        if (col_out && tid < BN) {  // (a step's sums are overwritten two steps later at the earliest)
            const float tot = s_col[(step & 1) * 2 * BN + tid] + s_col[((step & 1) * 2 + 1) * BN + tid];
            const int kc = n0 + tid;
            if (segs > 1) p.db_part[((int64_t)part_id * G + (f.Hb == f.H ? gi : 0)) * BN + tid] = tot;
            else if (kc < f.Lk) {
                if (use_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + kc, tot);
                else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + kc] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        gi = gn;
        mi = mn;
    };
    for (int step = 0; step < n_steps; step += 2) {
        one_step(std::integral_constant<int, 0>(), step);
        if (step + 1 < n_steps) one_step(std::integral_constant<int, 1>(), step + 1);
    }

    // a key block that no query (of this segment) can see still owns its dbias column (row-broadcast case)
    if (has_bias && !bias_rows && n_steps == 0 && tid < BN) {
        const int ngh = (f.Hb == f.H) ? G : 1;
        for (int gh = 0; gh < ngh; gh++) {
            const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
            if (segs > 1) p.db_part[((int64_t)part_id * G + gh) * BN + tid] = 0.f;
            else if (!use_accum && n0 + tid < f.Lk) ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + n0 + tid] = 0;
        }
    }

    // ---- the two query halves: wave (kw, 0) ends with dK, wave (kw, 1) with dV of the 32 keys
    {
        f32x4_t *give = (f32x4_t *)smem + (qh * 4 + kw) * DB * 4 * 64 + lane;
        const f32x4_t *take = (const f32x4_t *)smem + ((qh ^ 1) * 4 + kw) * DB * 4 * 64 + lane;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x16_t &v = qh ? dk[db] : dv[db];
                give[(db * 4 + q) * 64] = f32x4_t{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
            }
        __syncthreads();
        const float m = (qh || segs > 1) ? 1.f : f.scale;
        f32x4_t *dst = (f32x4_t *)p.dkv_part + ((int64_t)part_id * 2 + qh) * (BN * D / 4) + kw * DB * 4 * 64 + lane;
        uint16_t *out = qh ? (uint16_t *)p.dv + b * p.dv_b + (int64_t)key * p.dv_r + hk * p.dv_h
                           : (uint16_t *)p.dk + b * p.dk_b + (int64_t)key * p.dk_r + hk * p.dk_h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                f32x4_t w[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const f32x4_t o = take[(db * 4 + 2 * blk + q) * 64];
                    const f32x16_t &v = qh ? dv[db] : dk[db];
#pragma unroll
                    for (int e = 0; e < 4; e++) w[q][e] = (v[8 * blk + 4 * q + e] + o[e]) * m;
                }
                const int c = 32 * db + 16 * blk + 8 * g;
                if (segs > 1) {  // in the order the lanes hold them (1 KB per store)
                    dst[(db * 4 + 2 * blk) * 64] = w[0];
                    dst[(db * 4 + 2 * blk + 1) * 64] = w[1];
                } else if (key < f.Lk && c < f.d) {
                    *(u32x4_t *)(out + c) = u32x4_t{E::pack2(w[0][0], w[0][1]), E::pack2(w[0][2], w[0][3]), E::pack2(w[1][0], w[1][1]), E::pack2(w[1][2], w[1][3])};
                }
            }
    }
}

template <typename T, bool CAUSAL, bool GSUM, bool ODD>
hipError_t launch_wide_o(const BwdParams &p, hipStream_t stream) {
    auto kern = bwd_dkdv_wide_kernel<T, CAUSAL, GSUM, ODD>;
    static DynSmemLimit smem_limit;
    hipError_t e = smem_limit.ensure((const void *)kern, SMEM);
    if (e != hipSuccess) return e;
    const int units = ((p.f.Lk + BN - 1) / BN) * p.f.Hk * p.f.B;
    hipLaunchKernelGGL(kern, dim3(units * p.kv_segs), dim3(NT), SMEM, stream, p);
    return hipGetLastError();
}

template <typename T, bool CAUSAL, bool GSUM>
hipError_t launch_wide(const BwdParams &p, hipStream_t stream) {
    return odd_rows(p.f) ? launch_wide_o<T, CAUSAL, GSUM, true>(p, stream) : launch_wide_o<T, CAUSAL, GSUM, false>(p, stream);
}

}  // namespace

hipError_t launch_bwd_dkdv_wide(const BwdParams &p, int dtype, bool gsum, hipStream_t stream) {
    const bool c = p.f.causal != 0;
    if (dtype == 0) {
        if (gsum) return c ? launch_wide<bf16_tag, true, true>(p, stream) : launch_wide<bf16_tag, false, true>(p, stream);
        return c ? launch_wide<bf16_tag, true, false>(p, stream) : launch_wide<bf16_tag, false, false>(p, stream);
    }
    if (gsum) return c ? launch_wide<fp16_tag, true, true>(p, stream) : launch_wide<fp16_tag, false, true>(p, stream);
    return c ? launch_wide<fp16_tag, true, false>(p, stream) : launch_wide<fp16_tag, false, false>(p, stream);
}

}  // namespace fdma
