// Backward dynamic-mask attention for gfx950, column-mask specialisation at head dims 129 .. 256: the dK / dV / dBias kernel.
//
// Same math, work items and outputs as bwd_dkdv_colmask_kernel (fdma_bwd_colmask.hip; compute_dq_dk_dv_1colblock,
// csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the reference), laid out for what a head dim of 256 costs: dK and dV of
// 32 keys are 256 registers per lane, K and V of them another 128.  A wave that holds all of it (one per SIMD) spilled 200
// registers and took 5 us per step of 32 rows x 128 keys, for 0.85 us of matrix work.
//
// Here a workgroup is 8 waves over 128 keys, two to a SIMD, and a pair of waves shares 32 keys by ROLE: wave (kw, 0) has K,
// the scores, P and dV; wave (kw, 1) has V, dP, dS and dK.  Either is 16 + 16 MFMAs per step and fits 256 registers.  P passes from
// one to the other through LDS in fp32, once per step: a barrier in the middle of the step publishes it (the scores and dP in front of
// it, the dV and dK products behind it).
// Q, dO and the row statistics of a step come straight into LDS (global_load_lds), two steps ahead into three stages.
// LDS: 3 x 32 KB of Q / dO, 16 KB of P.  Bound by the chain of a step (two barriers, two waves per SIMD): 1.6 us.
// Before / now (us): 8192 tokens x 16/4 heads, 2048 kept: the call with its forward 2872 / 1049, this kernel 352; 1408 x 32/8, 439
// kept 268 / 70; ragged entries of 300 to 2000 x 8/2 1990 / 220 (in parts); 16 blocks of 256 rows, two heads each 137 / 38.
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_bwd_units.h"

namespace fdma {

namespace {

constexpr int D = 256;
constexpr int NT = 512;
constexpr int BM = 32;                 // query rows per step
constexpr int SUB = KV_BM / BM;        // steps per planning block
constexpr int KS = D / 16, DB = D / 32;
constexpr int ROW = D * 2;
constexpr int TILE = BM * ROW;         // a Q or dO tile
constexpr int NST = 3;
constexpr int STAGE = 2 * TILE;        // Q, dO
constexpr int OFF_STAT = NST * STAGE;  // per stage: 256 bytes of LSE (32 values, the last repeated), 256 of D
constexpr int OFF_P = OFF_STAT + NST * 512;
constexpr int SMEM = OFF_P + 4 * 4096;
constexpr int N_DMA = 5;               // direct loads of a wave per step: 2 of Q, 2 of dO, the statistics


template <typename T, bool CAUSAL, bool CMP>
__global__ void __launch_bounds__(NT) bwd_dkdv_256_kernel(const BwdParams p) {
    using E = Elem<T>;
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int kw = wave & 3, role = wave >> 2;
    const int G = f.H / f.Hk;
    const KvItem it = kv_item<CMP>(p, false);
    if (!it.valid) return;
    const int b = it.pair / f.Hk, hk = it.pair % f.Hk;
    const int n0 = it.n_block * KV_BN;
    const SeqInfo sq = seq_info(f, b);
    const int LqS = sq.Lq, LkS = sq.Lk;
    const int Lk = CMP ? f.cmp.count[it.pair] : LkS;
    if (n0 >= Lk) return;
    int slot = it.slot, first_step = 0, part_steps = 0;
    if (!CMP && p.kv_most > 1) {
        const int steps = G * kv_unit_steps(LqS, LkS, CAUSAL, n0, BM);
        const int n_parts = kv_parts_of(steps, p.kv_quota ? p.kv_quota : ragged_part_quota(f, BM), p.kv_most);
        if (it.part >= n_parts) return;
        if (n_parts > 1) {
            first_step = (int)((int64_t)steps * it.part / n_parts);
            part_steps = (int)((int64_t)steps * (it.part + 1) / n_parts) - first_step;
            slot = kv_unit_slot(p, b, hk, it.n_block) + it.part;
        }
    }
    const int key = n0 + kw * 32 + r;  // the key column this lane owns
    const int key_c = key < Lk ? key : Lk - 1;
    const int shift = LkS - LqS;
    const int32_t *cidx = CMP ? f.cmp.idx + (int64_t)it.pair * f.cmp.ld : nullptr;
    const int okey = CMP ? cidx[key_c] : key;
    const int okey_first = CMP ? cidx[n0] : n0;
    const int wlast = n0 + kw * 32 + 31;
    const int okey_wlast = CMP ? cidx[wlast < Lk ? wlast : Lk - 1] : wlast;

    // ---- this workgroup's steps: query blocks [s_lo, s_hi) of every head, the last block first, from step first_step on
    const int M_blocks = (LqS + KV_BM - 1) / KV_BM;
    const int m_start = M_blocks - dkdv_query_blocks(LqS, LkS, CAUSAL, okey_first);
    int m_lo = m_start, m_hi = M_blocks;
    if (CMP && slot >= 0) {
        const int n_seg = dkdv_segments(M_blocks - m_start, it.Q, it.Sm);
        if (it.seg >= n_seg) return;  // the reduce kernel knows that this slot stays unwritten
        const int len = (M_blocks - m_start + n_seg - 1) / n_seg;
        m_lo = m_start + it.seg * len;
        m_hi = m_lo + len < M_blocks ? m_lo + len : M_blocks;
    }
    const int S_blocks = (LqS + BM - 1) / BM;
    const int s_lo = m_lo * SUB, s_hi = m_hi * SUB < S_blocks ? m_hi * SUB : S_blocks;
    const int n_m = s_hi > s_lo ? s_hi - s_lo : 0;
    const int n_steps = !CMP && slot >= 0 ? part_steps : n_m * (it.g_hi - it.g_lo);
    const int gi0 = CMP || n_steps == 0 ? it.g_lo : first_step / n_m, mi0 = s_hi - 1 - (CMP || n_steps == 0 ? 0 : first_step % n_m);

    // ---- stationary fragment of this role: K (times softmax_scale * log2(e)) or V; lane holds row `key`, elements 16 ks + 8 g ..
    u32x4_t w[KS];
    {
        const uint16_t *kp = (const uint16_t *)f.k + b * f.k_b + (sq.k0 + key_c) * f.k_r + hk * f.k_h;
        const uint16_t *vp = (const uint16_t *)f.v + b * f.v_b + (sq.k0 + key_c) * f.v_r + hk * f.v_h;
        const uint16_t *src = role ? vp : kp;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            w[ks] = u32x4_t{0, 0, 0, 0};
            if (c < f.d) w[ks] = *(const u32x4_t *)(src + c);
        }
        if (role == 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int e = 0; e < 4; e++) w[ks][e] = E::pack2(E::lo(w[ks][e]) * f.scale_log2, E::hi(w[ks][e]) * f.scale_log2);
        }
    }

    const bool has_bias = f.bias != nullptr;
    // fused constant of this lane's key for query head h: bias * log2e, or -inf when the key is dropped
    // (the keys are opaque here and where sums leave: addresses derived from them would stay in registers that the loop lacks)
    auto column_const = [&](int h) -> float {
        int key_c = key < Lk ? key : Lk - 1;
        asm volatile("" : "+v"(key_c));
        if (key >= Lk) return -INFINITY;
        if (CMP) return f.cmp.fb[(int64_t)(b * f.cmp.Hfb + (f.cmp.Hfb == f.H ? h : hk)) * f.cmp.ld + key_c];
        if (f.mask) {
            const int hm = f.Hm == f.H ? h : (f.Hm == 1 ? 0 : hk);
            if (!f.mask[b * f.m_b + hm * f.m_h + key_c]) return -INFINITY;
        }
        if (!has_bias) return 0.f;
        const int hb = f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk);
        return E::lo((uint32_t)((const uint16_t *)f.bias)[b * f.bi_b + hb * f.bi_h + key_c]) * kLog2e;
    };

    // ---- direct loads of a step: piece i of a tile is rows 2 i, 2 i + 1; wave w fetches pieces w and w + 8 of Q and of dO.
    // A lane fills chunk position lane % 32 of its row, which holds chunk position ^ chunk_swz(row) of the global row.  Rows beyond the
    // queries repeat the last one (masked where used), chunks beyond d repeat chunk 0 (they meet zeros).
    const int prow = 2 * wave + (lane >> 5);
    const int pchunk = (lane & 31) ^ (int)chunk_swz<256>(prow);
    const uint32_t pcol = pchunk * 8 < f.d ? pchunk * 16 : 0;
    const uint32_t q_r2 = (uint32_t)(f.q_r * 2), do_r2 = (uint32_t)(p.do_r * 2);
    int dma_gi = gi0, dma_mi = mi0, dma_stage = 0;  // the step being fetched
    auto dma_step = [&](bool more) {  // all loads of that step; then on to the following one (past the last it is fetched again)
        const int h = hk * G + dma_gi, m0 = dma_mi * BM;
        const int left = LqS - 1 - m0, rows = left < BM - 1 ? left : BM - 1;
        const gptr_t qb = uniform_ptr((const uint16_t *)f.q + b * f.q_b + h * f.q_h + (sq.q0 + m0) * f.q_r);
        const gptr_t db = uniform_ptr((const uint16_t *)p.dout + b * p.do_b + h * p.do_h + (sq.q0 + m0) * p.do_r);
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(dma_stage * STAGE + wave * 1024));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = prow + 16 * i, row_c = row < rows ? row : rows;
            load_lds16((uint32_t)row_c * q_r2 + pcol, qb, dst + i * 8192);
            load_lds16((uint32_t)row_c * do_r2 + pcol, db, dst + TILE + i * 8192);
        }
        // (even waves fetch the LSE values, odd ones D, all the same)
        const gptr_t sp = uniform_ptr(wave & 1 ? p.softmax_d + b * p.sd_b + h * p.sd_h + sq.q0 + m0 : f.lse + b * f.lse_b + h * f.lse_h + sq.q0 + m0);
        load_lds4((uint32_t)(lane < rows ? lane : rows) * 4, sp, __builtin_amdgcn_readfirstlane(lds0 + OFF_STAT + dma_stage * 512 + (wave & 1) * 256));
        dma_stage = dma_stage == NST - 1 ? 0 : dma_stage + 1;
        if (more) {
            if (dma_mi == s_lo) { dma_mi = s_hi - 1; dma_gi++; } else dma_mi--;
        }
    };

    // fragment addresses (stage 0): rows of Q (scores) or dO (dP); transposing reads of dO (dV) or Q (dK)
    const int frow = pi_row(r);
    const uint32_t a_off = lds0 + (role ? TILE : 0) + (uint32_t)frow * ROW + (((uint32_t)g ^ chunk_swz<256>(frow)) << 4);
    const uint32_t tr_off = lds0 + (role ? 0 : TILE) + tr_chunk<256>(g, tr_lane(lane));
    const uint32_t stat_off = lds0 + OFF_STAT + role * 256 + 32 * g;
    const uint32_t p_off = lds0 + OFF_P + kw * 4096 + lane * 16;

    f32x16_t acc[DB];  // dV^T (role 0) or dK^T (role 1) of this wave's keys
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.f;
    float colsum = 0.f, cconst = 0.f;
    const bool use_accum = p.dbias_accum != nullptr;

    int gi = gi0, mi = mi0, stage = 0;
    if (n_steps > 0) {
        if (role == 0) cconst = column_const(hk * G + gi0);
        dma_step(n_steps > 1);
        dma_step(n_steps > 2);
        __builtin_amdgcn_s_waitcnt(0x0070 | N_DMA);
        __builtin_amdgcn_s_barrier();
    }
    for (int step = 0; step < n_steps; step++) {
        const int h = hk * G + gi, m0 = mi * BM;
        const uint32_t st = (uint32_t)stage * STAGE;  // (a multiple of 512: the swizzles stay XORs)
        uint32_t a_cur = a_off + st, tr_cur = tr_off + st;
        const uint32_t stat = stat_off + (uint32_t)stage * 512;
        asm volatile("" : "+v"(a_cur), "+v"(tr_cur));  // (the swizzled addresses are recomputed where used)
        dma_step(step + 3 < n_steps);  // (into the stage that the last step has left)

        // ---- S = Q K^T (role 0) or dP = dO V^T (role 1): M = query, N = key
        f32x16_t s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = cconst;  // (zero in role 1)
        {
            constexpr int FR = 4;
            u32x4_t a[KS];
            auto frag = [&](int ks) { return lds_ld128((a_cur ^ ((uint32_t)(ks & 7) << 5)) + (uint32_t)((ks >> 3) * 256)); };
#pragma unroll
            for (int ks = 0; ks < FR; ks++) a[ks] = frag(ks);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                if (ks + FR < KS) a[ks + FR] = frag(ks + FR);
                s = E::mfma(a[ks], w[ks], s);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // statistics of this lane's rows: register 8 blk + e <-> row 16 blk + 8 g + e
        f32x4_t st4[4];
#pragma unroll
        for (int q = 0; q < 4; q++) st4[q] = __builtin_bit_cast(f32x4_t, lds_ld128(stat + 64 * (q >> 1) + 16 * (q & 1)));
        uint32_t pk[8];
        if (role == 0) {
            // ---- P = exp2(S - LSE * log2e), scores already scaled and offset by the column constant
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = fast_exp2(__builtin_fmaf(st4[i >> 2][i & 3], -kLog2e, s[i]));
            if ((CAUSAL && okey_wlast > m0 + shift) || m0 + BM > LqS) {  // rows above the diagonal, or beyond the queries
                asm volatile("" ::: "memory");
                const int lim = CAUSAL ? okey - shift - m0 - 8 * g : -64, lim_hi = LqS - m0 - 8 * g;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int row = 16 * (i >> 3) + (i & 7);
                    s[i] = (row >= lim && row < lim_hi) ? s[i] : 0.f;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(__attribute__((address_space(3))) f32x4_t *)(uintptr_t)(p_off + q * 1024) = f32x4_t{s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]};
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // P is there
        if (role != 0) {
            // ---- dS = P * (dP - D)
            float part = 0.f;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4_t pv = __builtin_bit_cast(f32x4_t, lds_ld128(p_off + q * 1024));
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    s[4 * q + e] = (s[4 * q + e] - st4[q][e]) * pv[e];
                    part += s[4 * q + e];
                }
            }
            colsum += part;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) pk[i] = E::pack2(s[2 * i], s[2 * i + 1]);
        __builtin_amdgcn_sched_barrier(0);
        // ---- dV^T += dO^T P or dK^T += Q^T dS (M = d, N = key, contraction = query)
        {
            constexpr int NG = 2 * DB, FR2 = 3;
            u32x2_t tl[NG], th[NG];
            auto tr_read = [&](int gi_) {
                const int qb = gi_ / DB, db = gi_ % DB;
                const uint32_t lo = tr_cur ^ ((uint32_t)(db & 3) << 6), hi = tr_cur ^ (((uint32_t)(db & 3) << 6) | 16u);
                const uint32_t c = (uint32_t)(qb * 16 * ROW + (db >> 2) * 256);
                tl[gi_] = lds_ld_tr16(lo + c);
                th[gi_] = lds_ld_tr16(hi + c + 4 * ROW);
            };
#pragma unroll
            for (int x = 0; x < FR2; x++) tr_read(x);
#pragma unroll
            for (int x = 0; x < NG; x++) {
                if (x + FR2 < NG) tr_read(x + FR2);
                const int qb = x / DB, db = x % DB;
                const u32x4_t bop = {pk[4 * qb], pk[4 * qb + 1], pk[4 * qb + 2], pk[4 * qb + 3]};
                const u32x4_t av = {tl[x][0], tl[x][1], th[x][0], th[x][1]};
                acc[db] = E::mfma(av, bop, acc[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- dBias column sums: flushed when the bias head changes (a part: at its own last step too, one sum for all its
        // heads where they share the bias)
        if (has_bias && role != 0) {
            const bool part_end = !CMP && slot >= 0 && step == n_steps - 1;
            if ((mi == s_lo && ((CMP && slot >= 0) || f.Hb == f.H || (gi == G - 1 && slot < 0))) || part_end) {
                const float tot = xhalf_sum(colsum);
                int kk = kw * 32 + r, ok = okey;
                asm volatile("" : "+v"(kk), "+v"(ok));
                const int hb = f.Hb == f.H ? h : (f.Hb == 1 ? 0 : hk);
                if (slot >= 0) {
                    if (g == 0) p.db_part[((int64_t)slot * G + (CMP || f.Hb == f.H ? gi - it.g_lo : 0)) * KV_BN + kk] = tot;
                } else if (g == 0 && key < Lk) {
                    if (use_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + ok, tot);
                    else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + ok] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
                }
                colsum = 0.f;
            }
        }
        if (mi == s_lo) {
            mi = s_hi - 1;
            gi++;
            if (role == 0 && step + 1 < n_steps) cconst = column_const(hk * G + gi);
        } else {
            mi--;
        }
        stage = stage == NST - 1 ? 0 : stage + 1;
        // the next step's loads have landed (the N_DMA of the one after it stay in flight), everybody is done with this stage and P
        __builtin_amdgcn_s_waitcnt(0x0070 | N_DMA);
        __builtin_amdgcn_s_barrier();
    }
    // (direct loads still in flight must not land in LDS that belongs to the next workgroup by then)
    __builtin_amdgcn_s_waitcnt(0x0070);

    // a key block that no query can see still owns its dbias column
    if (has_bias && role != 0 && n_steps == 0 && g == 0) {
        if (slot >= 0) {
            for (int gl = 0; gl < it.g_hi - it.g_lo; gl++) p.db_part[((int64_t)slot * G + gl) * KV_BN + (key - n0)] = 0.f;
        } else if (!use_accum && key < Lk) {
            const int ngh = (f.Hb == f.H) ? G : 1;
            for (int gh = 0; gh < ngh; gh++) {
                const int hb = f.Hb == f.H ? hk * G + gh : (f.Hb == 1 ? 0 : hk);
                ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + okey] = 0;
            }
        }
    }

    // ---- a part: fp32 sums in the order the lanes hold them (1 KB per store); heads without a step in it have zero columns
    if (!CMP && slot >= 0) {
        if (has_bias && role != 0 && f.Hb == f.H && g == 0) {
            const int g_end = (first_step + part_steps - 1) / n_m;
            for (int gh = 0; gh < G; gh++)
                if (gh < gi0 || gh > g_end) p.db_part[((int64_t)slot * G + gh) * KV_BN + (key - n0)] = 0.f;
        }
        f32x4_t *dst = (f32x4_t *)p.dkv_part + (int64_t)slot * (2 * KV_BN * D / 4) + (role ? 0 : KV_BN * D / 4) + kw * DB * 4 * 64 + lane;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) dst[(db * 4 + q) * 64] = f32x4_t{acc[db][4 * q], acc[db][4 * q + 1], acc[db][4 * q + 2], acc[db][4 * q + 3]};
        return;
    }
    // ---- shared block of compacted keys: fp32 partial dK^T / dV^T, [which][d][key] so that a wave writes 128-byte runs
    if (CMP && slot >= 0) {
        float *dst = p.dkv_part + ((int64_t)slot * 2 + (role ? 0 : 1)) * D * KV_BN + (key - n0);
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) dst[(32 * db + 16 * (i >> 3) + 8 * g + (i & 7)) * KV_BN] = acc[db][i];
        return;
    }
    // ---- dK (scaled) or dV
    if (key < Lk) {
        int okey_s = okey;
        asm volatile("" : "+v"(okey_s));
        const float m = role ? f.scale : 1.f;
        uint16_t *out = role ? (uint16_t *)p.dk + b * p.dk_b + (sq.k0 + okey_s) * p.dk_r + hk * p.dk_h
                             : (uint16_t *)p.dv + b * p.dv_b + (sq.k0 + okey_s) * p.dv_r + hk * p.dv_h;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const int c = 32 * db + 16 * blk + 8 * g;
                u32x4_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = E::pack2(acc[db][8 * blk + 2 * e] * m, acc[db][8 * blk + 2 * e + 1] * m);
                if (c < f.d) *(u32x4_t *)(out + c) = v;
            }
    }
}

template <typename T, bool CAUSAL, bool CMP> hipError_t launch_one(const BwdParams &p, int grid, hipStream_t stream) {
    auto kern = bwd_dkdv_256_kernel<T, CAUSAL, CMP>;
    static DynSmemLimit smem_limit;
    const hipError_t e = smem_limit.ensure((const void *)kern, SMEM);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), SMEM, stream, p);
    return hipGetLastError();
}
template <typename T> hipError_t launch_t(const BwdParams &p, int grid, hipStream_t stream) {
    if (p.f.cmp.on) return p.f.causal ? launch_one<T, true, true>(p, grid, stream) : launch_one<T, false, true>(p, grid, stream);
    return p.f.causal ? launch_one<T, true, false>(p, grid, stream) : launch_one<T, false, false>(p, grid, stream);
}

}  // namespace

hipError_t launch_bwd_dkdv_256(const BwdParams &p, int dtype, int grid, hipStream_t stream) {
    return dtype == 0 ? launch_t<bf16_tag>(p, grid, stream) : launch_t<fp16_tag>(p, grid, stream);
}

}  // namespace fdma
