// Sums of the parts that the compacted dK/dV kernels leave, as device code of the dQ launches (fdma_bwd_colmask.hip,
// fdma_bwd_dq_256.hip), some of whose workgroups do this instead of dQ work.
#pragma once

#include "fdma_bwd_units.h"
#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int RED_THREADS = 256;  // threads that share an item (a workgroup, or half of one)

// Sums the partial results of one unit that the compacted dK/dV kernel split over several workgroups, in a fixed
// order, and writes dK (scaled), dV and dBias to the original rows / columns of the kept keys.  `y` picks a pair of
// 8-wide head-dim chunks (0 .. D/16 - 1), so that few units still give many work items; item y == 0 also folds the
// unit's dBias columns.  Called by the workgroups that the dQ launch sets aside for it (see bwd_dq_colmask_kernel).
template <typename T, int D>
__device__ __forceinline__ void dkdv_reduce_item(const BwdParams &p, const int unit, const int y, const int tid) {
    using E = Elem<T>;
    const FwdParams &f = p.f;
    const int32_t *plan = f.cmp.plan;
    const int Gs = plan[1], Sm = plan[2], Q = plan[4], per = Gs * Sm;
    // a plan whose lists overflowed left parts uncomputed: every sum starts from NaN then
    const float start = plan[6] != 0 ? __builtin_nanf("") : 0.f;
    int lo = 0, hi = f.B * f.Hk;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (plan[DKDV_PLAN_HDR + mid] <= unit) lo = mid;
        else hi = mid;
    }
    const int pair = lo, b = pair / f.Hk, hk = pair % f.Hk;
    const int n0 = (unit - plan[DKDV_PLAN_HDR + pair]) * KV_BN;
    const int Lk = f.cmp.count[pair];
    const int G = f.H / f.Hk;
    const int kk = tid % KV_BN, half = tid / KV_BN;
    const bool live = n0 + kk < Lk;
    const int okey = live ? f.cmp.idx[(int64_t)pair * f.cmp.ld + n0 + kk] : 0;
    // segments of this unit that were written (same rule as in the main kernel)
    const int n_seg = dkdv_segments(dkdv_query_blocks(f.Lq, f.Lk, f.causal, f.cmp.idx[(int64_t)pair * f.cmp.ld + n0]), Q, Sm);
    const float *base = p.dkv_part + (int64_t)unit * per * 2 * D * KV_BN + kk;
    for (int c = 2 * y + half; c == 2 * y + half && c * 8 < f.d; c += RED_THREADS / KV_BN) {
        float ak[8], av[8];
#pragma unroll
        for (int e = 0; e < 8; e++) { ak[e] = start; av[e] = start; }
        // written slots in a fixed order, four at a time: a workgroup here sits beside the dQ workgroups and should
        // give its place back soon, so the loads of four slots are in flight together (slots past the end repeat
        // the last one and are not added)
        const int n_w = Gs * n_seg;
        for (int j = 0; j < n_w; j += 4) {
            float kq[4][8], vq[4][8];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int jt = j + t < n_w ? j + t : n_w - 1;
                const float *pt = base + (int64_t)((jt / n_seg) * Sm + jt % n_seg) * 2 * D * KV_BN;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    kq[t][e] = pt[(c * 8 + e) * KV_BN];
                    vq[t][e] = pt[(D + c * 8 + e) * KV_BN];
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++)
                if (j + t < n_w) {
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        ak[e] += kq[t][e];
                        av[e] += vq[t][e];
                    }
                }
        }
        if (live) {
            u32x4_t wk, wv;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                wk[e] = E::pack2(ak[2 * e] * f.scale, ak[2 * e + 1] * f.scale);
                wv[e] = E::pack2(av[2 * e], av[2 * e + 1]);
            }
            *(u32x4_t *)((uint16_t *)p.dk + b * p.dk_b + (int64_t)okey * p.dk_r + hk * p.dk_h + c * 8) = wk;
            *(u32x4_t *)((uint16_t *)p.dv + b * p.dv_b + (int64_t)okey * p.dv_r + hk * p.dv_h + c * 8) = wv;
        }
    }
    if (f.bias && live && y == 0) {
        const int gper = G / Gs;
        const float *dbp = p.db_part + (int64_t)unit * per * G * KV_BN + kk;  // [part][local head][key]
        auto emit = [&](int hb, float tot) {
            if (p.dbias_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + okey, tot);
            else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + okey] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
        };
        if (f.Hb == f.H) {
            for (int gi = half; gi < G; gi += RED_THREADS / KV_BN) {
                float tot = start;
                for (int sg = 0; sg < n_seg; sg++) tot += dbp[((int64_t)((gi / gper) * Sm + sg) * G + gi % gper) * KV_BN];
                emit(hk * G + gi, tot);
            }
        } else if (half == 0) {
            float tot = start;
            for (int gs = 0; gs < Gs; gs++)
                for (int sg = 0; sg < n_seg; sg++)
                    for (int gl = 0; gl < gper; gl++) tot += dbp[((int64_t)(gs * Sm + sg) * G + gl) * KV_BN];
            emit(f.Hb == 1 ? 0 : hk, tot);
        }
    }
}

// Workgroup `rb` of `nrb` reducing workgroups takes every nrb-th of the U units x D/16 chunk pairs.
template <typename T, int D>
__device__ __forceinline__ void dkdv_reduce_blocks(const BwdParams &p, const int rb, const int nrb, const int tid) {
    const int32_t *plan = p.f.cmp.plan;
    const int U = plan[0];
    if (plan[1] * plan[2] == 1) return;  // no unit was split: the dK/dV kernel wrote the results itself
    for (int item = rb; item < U * (D / 16); item += nrb) dkdv_reduce_item<T, D>(p, item / (D / 16), item % (D / 16), tid);
}

}  // namespace

}  // namespace fdma
