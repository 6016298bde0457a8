// Backward dynamic-mask attention for gfx950, column-mask specialisation at head dims 129 .. 256: the dQ kernel.
//
// Same math, inputs and outputs as bwd_dq_colmask_kernel (fdma_bwd_colmask.hip; compute_dq_dk_dv_1colblock,
// csrc/flash_sparse_attn/src/flash_bwd_kernel.h:79-1142 of the reference), laid out for what a head dim of 256 costs: dQ, Q and dO of
// 32 rows are 256 registers per lane.  A wave that held them (one per SIMD) took 4 us per step of 128 rows x 32 keys, for 0.43 us of
// matrix work.
//
// Here a workgroup is 8 waves over 128 query rows, two to a SIMD, and a pair of waves shares 32 rows by ROLE (as in
// fdma_bwd_dkdv_256.hip): wave (rw, 0) has Q, the scores and P, wave (rw, 1) dO, dP and dS; either then adds K^T dS to its half of
// dQ's head dim.  P passes through LDS in fp32 (a barrier), dS in the 16 bits that the product takes (another).
// K, V and the fused bias column of a 32-key tile come straight into LDS (global_load_lds), requested a tile and a half ahead, behind
// the first barrier of a step, into the stage that the step before has left: two barriers per step are all there are.
// LDS: 3 x 32 KB of K / V, 24 KB of P and dS.  Bound by the chain of a step (two barriers, two waves per SIMD): 1.7 us.
// Before / now (us): 8192 tokens x 16/4 heads, 2048 kept (sums of dK / dV parts carried along) 528 / 482; 1408 x 32/8, 439 kept
// 88 / 73; 4096 x 8/2, 1024 kept 85 / 70; 600 x 16/4, all kept 47.5 / 44; a ragged entry of 3000 x 2/1 168 / 162.
#include <type_traits>

#include "fdma_bwd_reduce.h"
#include "fdma_bwd_units.h"
#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int D = 256;
constexpr int NT = 512;
constexpr int BM = 128;                // query rows per workgroup
constexpr int BN = 32;                 // keys per tile
constexpr int KS = D / 16, DH = D / 64;  // 16-wide steps of the head dim; 32-wide blocks of a role's half of dQ
constexpr int ROW = D * 2;
constexpr int TILE = BN * ROW;
constexpr int NST = 3;
constexpr int STAGE = 2 * TILE;        // K, V
constexpr int OFF_COL = NST * STAGE;   // per stage: 32 floats, twice (what a direct load of a wave fills)
constexpr int OFF_P = OFF_COL + NST * 256;
constexpr int OFF_DS = OFF_P + 4 * 4096;
constexpr int OFF_BITS = OFF_DS + 4 * 2048;
static_assert(OFF_BITS >= 2 * RED_LDS, "the workgroups that sum parts use it");
constexpr int SMEM = OFF_BITS + (1 << 20) / BN / 8;  // (bwd_colmask_applicable: 2^20 keys at most)


template <typename T, bool CAUSAL, bool CMP>
__global__ void __launch_bounds__(NT) bwd_dq_256_kernel(const BwdParams p) {
    using E = Elem<T>;
    constexpr int N_DMA = 4 + (CMP ? 1 : 0);  // direct loads of a wave per tile: 2 of K, 2 of V, the column
    extern __shared__ __attribute__((aligned(256))) char smem[];
    const uint32_t lds0 = lds_addr(smem);  // (a multiple of 256)
    uint32_t *sBits = (uint32_t *)(smem + OFF_BITS);

    const FwdParams &f = p.f;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int rw = wave & 3, role = wave >> 2;
    int lid = blockIdx.x;  // index among the dQ workgroups
    if (CMP) {  // some workgroups sum partial results of the dK/dV kernel instead (see place_reduction, fdma_bwd_colmask.hip)
        const int at = lid - p.red_first;
        if (at >= 0 && at < p.red_count) {
            dkdv_reduce_blocks<T, D>(kernel_args_apart<BwdParams>(), at * 2 + (wave >> 2), p.red_count * 2, tid & 255, (float *)(smem + (wave >> 2) * RED_LDS));
            return;
        }
        if (at >= 0) lid -= p.red_count;
    }
    const RowUnit ru = row_unit(f, lid, BM);  // (heaviest first under causal)
    if (ru.block < 0) return;
    const int b = ru.b, hk = ru.hk, h = ru.h;
    const int m0 = ru.block * BM;
    const SeqInfo sq = seq_info(f, b);
    const int LqS = sq.Lq, LkS = sq.Lk;
    if (m0 >= LqS) return;
    const int qrow = m0 + rw * 32 + r;
    const int qrow_c = qrow < LqS ? qrow : LqS - 1;
    const int shift = LkS - LqS;

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
    const int vis_wave = CAUSAL ? visible_columns<CMP>(m0 + rw * 32, LqS, LkS, ccnt) : 0;
    const int vis_block = CAUSAL ? visible_columns<CMP>(m0 + BM - 1, LqS, LkS, ccnt) : 0;
    int n_end = (Lk + BN - 1) / BN;
    if (CAUSAL) {
        const int ne = ((vis_block < 0 ? 0 : vis_block) + BN - 1) / BN;
        if (ne < n_end) n_end = ne;
    }

    // ---- active-tile bitmap (tiles with at least one kept key)
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
        if (lane == 0) {
            const int w0 = (base + wave * 64) >> 5;
            sBits[w0] = (uint32_t)ball;
            sBits[w0 + 1] = (uint32_t)(ball >> 32);
        }
    }
    if (!CMP) __syncthreads();
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

    // ---- stationary fragments of this role (B operands): Q, times softmax_scale * log2(e) (it only feeds the scores), or dO
    u32x4_t w[KS];
    {
        const uint16_t *qp = (const uint16_t *)f.q + b * f.q_b + (sq.q0 + qrow_c) * f.q_r + h * f.q_h;
        const uint16_t *dp = (const uint16_t *)p.dout + b * p.do_b + (sq.q0 + qrow_c) * p.do_r + h * p.do_h;
        const uint16_t *src = role ? dp : qp;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            w[ks] = u32x4_t{0, 0, 0, 0};
            if (qrow < LqS && c < f.d) w[ks] = *(const u32x4_t *)(src + c);
        }
        if (role == 0) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int e = 0; e < 4; e++) w[ks][e] = E::pack2(E::lo(w[ks][e]) * f.scale_log2, E::hi(w[ks][e]) * f.scale_log2);
        }
    }
    // what the accumulators of this role start from, negated: LSE * log2(e) or D
    float stat = role ? 0.f : INFINITY;
    if (role == 0) {
        if (qrow < LqS) stat = f.lse[b * f.lse_b + h * f.lse_h + sq.q0 + qrow] * kLog2e;
    } else if (CMP) {
        if (qrow < LqS) stat = p.softmax_d[b * p.sd_b + h * p.sd_h + sq.q0 + qrow];
    } else {  // D = rowsum(dO * O), left for the dK/dV kernel (see bwd_dq_colmask_kernel)
        const uint16_t *op = (const uint16_t *)f.o + b * f.o_b + (sq.q0 + qrow_c) * f.o_r + h * f.o_h;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = ks * 16 + g * 8;
            const u32x4_t ov = *(const u32x4_t *)(op + (c < f.d ? c : 0));  // (dO is zero beyond d and beyond Lq)
#pragma unroll
            for (int e = 0; e < 4; e++) stat += E::lo(ov[e]) * E::lo(w[ks][e]) + E::hi(ov[e]) * E::hi(w[ks][e]);
        }
        stat = xhalf_sum(stat);
        if (qrow >= LqS) stat = 0.f;
        // (fixed lengths: padded rows are zero)
        if (g == 0 && (qrow < LqS || (!f.cu_q && qrow < p.Lq_rounded))) p.softmax_d[b * p.sd_b + h * p.sd_h + sq.q0 + qrow] = stat;
    }

    // ---- staging: piece i of a tile is rows 2 i, 2 i + 1; wave w fetches pieces w and w + 8 of K and of V (see
    // fdma_bwd_dkdv_256.hip).  The column: with compacted keys as it is in memory, else made by wave 0 from mask and bias.
    const int prow = 2 * wave + (lane >> 5);
    const int pchunk = (lane & 31) ^ (int)chunk_swz<256>(prow);
    const uint32_t pcol = pchunk * 8 < f.d ? pchunk * 16 : 0;
    const uint32_t k_r2 = (uint32_t)(f.k_r * 2), v_r2 = (uint32_t)(f.v_r * 2);
    auto load_tile = [&](int j, int stage) {
        const gptr_t kb = uniform_ptr(kbase + (int64_t)j * BN * f.k_r), vb = uniform_ptr(vbase + (int64_t)j * BN * f.v_r);
        const int left = Lk - 1 - j * BN, rows = left < BN - 1 ? left : BN - 1;
        if (!CMP && wave == 0) {
            const int col = j * BN + r;
            const int cc = col < Lk ? col : 0;
            const bool keep = col < Lk && (!mrow || mrow[cc]);  // (a dropped key's bias is not looked at: it need not be a number)
            const float v = brow ? E::lo((uint32_t)brow[cc]) * kLog2e : 0.f;
            lds_st32(lds0 + OFF_COL + (uint32_t)stage * 256 + 4 * lane, __float_as_uint(keep ? v : -INFINITY));
        }
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(stage * STAGE + wave * 1024));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = prow + 16 * i, row_c = row < rows ? row : rows;
            load_lds16((uint32_t)row_c * k_r2 + pcol, kb, dst + i * 8192);
            load_lds16((uint32_t)row_c * v_r2 + pcol, vb, dst + TILE + i * 8192);
        }
        if (CMP)  // (columns beyond the kept keys repeat the last one: masked where used)
            load_lds4((uint32_t)(r < rows ? r : rows) * 4, uniform_ptr(fbrow + j * BN), __builtin_amdgcn_readfirstlane(lds0 + OFF_COL + (uint32_t)stage * 256));
    };

    // fragment addresses (stage 0): rows of K or V; transposing reads of K, this role's half of the head dim
    const int frow = pi_row(r);
    const uint32_t a_off = lds0 + (role ? TILE : 0) + (uint32_t)frow * ROW + (((uint32_t)g ^ chunk_swz<256>(frow)) << 4);
    const uint32_t tr_off = lds0 + (uint32_t)role * 256 + tr_chunk<256>(g, tr_lane(lane));
    const uint32_t col_off = lds0 + OFF_COL + 32 * g;
    const uint32_t p_off = lds0 + OFF_P + rw * 4096 + lane * 16, ds_off = lds0 + OFF_DS + rw * 2048 + lane * 16;

    f32x16_t dq[DH];
#pragma unroll
    for (int db = 0; db < DH; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dq[db][i] = 0.f;

    int jc = next_active(0), jn = n_end, stage = 0;
    if (jc < n_end) {
        jn = next_active(jc + 1);
        load_tile(jc, 0);
        load_tile(jn < n_end ? jn : jc, 1);  // (past the last tile it is fetched again and dropped)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N_DMA) : "memory");
    }
    while (jc < n_end) {
        const int n0 = jc * BN;
        const int jnn = next_active(jn + 1);
        const uint32_t st = (uint32_t)stage * STAGE;  // (a multiple of 512: the swizzles stay XORs)
        uint32_t a_cur = a_off + st, tr_cur = tr_off + st;
        asm volatile("" : "+v"(a_cur), "+v"(tr_cur));  // (the swizzled addresses are recomputed where used)

        // ---- S^T = K Q^T on top of the column and minus the row's LSE (role 0), or dP^T = V dO^T on top of minus D (role 1)
        f32x16_t s;
        if (role == 0) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4_t c = __builtin_bit_cast(f32x4_t, lds_ld128(col_off + (uint32_t)stage * 256 + 64 * (q >> 1) + 16 * (q & 1)));
#pragma unroll
                for (int e = 0; e < 4; e++) s[4 * q + e] = c[e] - stat;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = -stat;
        }
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
        if (role == 0) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = fast_exp2(s[i]);
            if ((CAUSAL && n0 + BN > vis_wave) || (CMP && n0 + BN > Lk)) {  // keys above the diagonal, or beyond the kept ones
                asm volatile("" ::: "memory");
                int lim = CAUSAL ? vis_lane - 1 - n0 - 8 * g : BN;
                const int last = Lk - 1 - n0 - 8 * g;
                lim = lim < last ? lim : last;
#pragma unroll
                for (int i = 0; i < 16; i++) s[i] = 16 * (i >> 3) + (i & 7) <= lim ? s[i] : 0.f;
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                *(__attribute__((address_space(3))) f32x4_t *)(uintptr_t)(p_off + q * 1024) = f32x4_t{s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]};
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // P is there, and everybody has left the stage before this one
        load_tile(jnn < n_end ? jnn : jc, stage == 0 ? NST - 1 : stage - 1);
        uint32_t pk[8];
        if (role != 0) {
            // ---- dS^T = P^T * (dP^T - D)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4_t pv = __builtin_bit_cast(f32x4_t, lds_ld128(p_off + q * 1024));
                pk[2 * q] = E::pack2(s[4 * q] * pv[0], s[4 * q + 1] * pv[1]);
                pk[2 * q + 1] = E::pack2(s[4 * q + 2] * pv[2], s[4 * q + 3] * pv[3]);
            }
#pragma unroll
            for (int q = 0; q < 2; q++)
                *(__attribute__((address_space(3))) u32x4_t *)(uintptr_t)(ds_off + q * 1024) = u32x4_t{pk[4 * q], pk[4 * q + 1], pk[4 * q + 2], pk[4 * q + 3]};
        }
        // dS is there, and so is the next tile (the loads of the one after it stay in flight)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N_DMA) : "memory");
        if (role == 0) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const u32x4_t v = lds_ld128(ds_off + q * 1024);
#pragma unroll
                for (int e = 0; e < 4; e++) pk[4 * q + e] = v[e];
            }
        }
        // ---- dQ^T += K^T dS^T, this role's half of the head dim
        {
            constexpr int NG = 2 * DH, FR2 = 3;
            u32x2_t tl[NG], th[NG];
            auto tr_read = [&](int x) {
                const int kb = x / DH, db = x % DH;
                const uint32_t c = (uint32_t)(kb * 16 * ROW);
                tl[x] = lds_ld_tr16((tr_cur ^ ((uint32_t)db << 6)) + c);
                th[x] = lds_ld_tr16((tr_cur ^ (((uint32_t)db << 6) | 16u)) + c + 4 * ROW);
            };
#pragma unroll
            for (int x = 0; x < FR2; x++) tr_read(x);
#pragma unroll
            for (int x = 0; x < NG; x++) {
                if (x + FR2 < NG) tr_read(x + FR2);
                const int kb = x / DH, db = x % DH;
                const u32x4_t bop = {pk[4 * kb], pk[4 * kb + 1], pk[4 * kb + 2], pk[4 * kb + 3]};
                const u32x4_t av = {tl[x][0], tl[x][1], th[x][0], th[x][1]};
                dq[db] = E::mfma(av, bop, dq[db]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        stage = stage == NST - 1 ? 0 : stage + 1;
        jc = jn;
        jn = jnn;
    }
    // (direct loads still in flight must not land in LDS that belongs to the next workgroup by then)
    __builtin_amdgcn_s_waitcnt(0x0070);
    if (qrow < LqS) {
        uint16_t *dqp = (uint16_t *)p.dq + b * p.dq_b + (sq.q0 + qrow) * p.dq_r + h * p.dq_h;
#pragma unroll
        for (int db = 0; db < DH; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const int c = 128 * role + 32 * db + 16 * blk + 8 * g;
                u32x4_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = E::pack2(dq[db][8 * blk + 2 * e] * f.scale, dq[db][8 * blk + 2 * e + 1] * f.scale);
                if (c < f.d) *(u32x4_t *)(dqp + c) = v;
            }
    }
}

template <typename T, bool CAUSAL, bool CMP> hipError_t launch_one(const BwdParams &p, int grid, hipStream_t stream) {
    auto kern = bwd_dq_256_kernel<T, CAUSAL, CMP>;
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

hipError_t launch_bwd_dq_256(const BwdParams &p, int dtype, int grid, hipStream_t stream) {
    return dtype == 0 ? launch_t<bf16_tag>(p, grid, stream) : launch_t<fp16_tag>(p, grid, stream);
}

}  // namespace fdma
