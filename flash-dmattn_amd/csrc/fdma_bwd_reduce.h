// Sums of the parts that the compacted dK/dV kernels leave, as device code of the dQ launches (fdma_bwd_colmask.hip,
// fdma_bwd_dq_256.hip), some of whose workgroups do this instead of dQ work.
#pragma once

#include "fdma_bwd_units.h"
#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int RED_THREADS = 256;            // threads that share an item (a workgroup, or half of one)
constexpr int RED_PITCH = 136;              // floats of an LDS row: 128 keys, and rows four apart lie half the banks apart
constexpr int RED_LDS = 64 * RED_PITCH * 4;  // LDS of an item

// Sums the partial results of one unit that the compacted dK/dV kernel split over several workgroups, in a fixed
// order, and writes dK (scaled), dV and dBias to the original rows / columns of the kept keys.  `y` picks a pair of
// 8-wide head-dim chunks (0 .. D/16 - 1), so that few units still give many work items; item y == 0 also folds the
// unit's dBias columns.
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
#pragma unroll 4
                for (int sg = 0; sg < n_seg; sg++) tot += dbp[((int64_t)((gi / gper) * Sm + sg) * G + gi % gper) * KV_BN];
                emit(hk * G + gi, tot);
            }
        } else if (half == 0) {
            float tot = start;
            const int n = Gs * n_seg * gper;
            int gs = 0, sg = 0, gl = 0;  // of the next column: group of heads, segment, local head
            for (int j = 0; j < n; j += 8) {
                float v[8];
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    v[t] = j + t < n ? dbp[((int64_t)(gs * Sm + sg) * G + gl) * KV_BN] : 0.f;
                    if (++gl == gper) {
                        gl = 0;
                        if (++sg == n_seg) { sg = 0; gs++; }
                    }
                }
#pragma unroll
                for (int t = 0; t < 8; t++) tot += v[t];
            }
            emit(f.Hb == 1 ? 0 : hk, tot);
        }
    }
}

// Sum of `n_w` slots of eight head-dim rows of a unit's partial dK or dV (128 keys each), into LDS as S sums per row, which the
// caller adds up.  Thread (row = tid / 32, quad = tid % 32) has four keys, every S-th slot from row % S on and S of the eight rows.  Slots
// are taken in a fixed order, 8 to 16 loads in flight (slots past the end repeat the last one and are not added).
template <int S, int D>
__device__ __forceinline__ void dkdv_reduce_rows(const float *base, const int n_w, const int n_seg, const int Sm, const int tid, float *lds) {
    constexpr int U = S == 8 ? 2 : 8 / S;  // slots in flight
    const int row = tid >> 5, quad = tid & 31, first = row % S, d0 = row / S * S;
    const float *src = base + d0 * KV_BN + 4 * quad;
    f32x4_t acc[S];
#pragma unroll
    for (int x = 0; x < S; x++) acc[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int j = first; j < n_w; j += U * S) {
        f32x4_t v[U][S];
#pragma unroll
        for (int t = 0; t < U; t++) {
            const int jt = j + t * S < n_w ? j + t * S : n_w - 1;
            const float *pt = src + (int64_t)(jt / n_seg * Sm + jt % n_seg) * 2 * D * KV_BN;
#pragma unroll
            for (int x = 0; x < S; x++) v[t][x] = *(const f32x4_t *)(pt + x * KV_BN);
        }
#pragma unroll
        for (int t = 0; t < U; t++)
            if (j + t * S < n_w) {
#pragma unroll
                for (int x = 0; x < S; x++) acc[x] += v[t][x];
            }
    }
#pragma unroll
    for (int x = 0; x < S; x++) *(f32x4_t *)(lds + (first * 8 + d0 + x) * RED_PITCH + 4 * quad) = acc[x];
}

// Sums the partial results of the units that the compacted dK/dV kernel split over several workgroups, in a fixed
// order, and writes dK (scaled), dV and dBias to the original rows / columns of the kept keys.  Called by the workgroups that the
// dQ launch sets aside for it: share `rb` of `nrb`.  All threads of the workgroup call it together (it has barriers); `lds`:
// RED_LDS bytes of this share's own.
// Items of 16 columns of dK and dV: 64 loads in flight per thread and no barrier (bound by memory).  But a unit has up to 16 slots per
// query head of its group, and a thread that walks them waits for memory again and again on few CUs (3968 tokens x 8/2 heads, d = 64, 320
// kept: 6 units, 24 items, and their dBias slot by slot, 46 us the launch, 13.7 now).  Where that is longer than dQ beside it (plan[7]),
// an item is eight columns of dK or of dV, or dBias, the slots are spread over the threads, and the sums are added up through LDS.
// That keeps a third as many bytes in flight and more workgroups busy.  One thread / side by side, the dQ launch of 2048 tokens (us):
// d = 64: 16/8 heads, 256 kept 19.3 / 13.2, 16/4, 640 kept 20.7 / 19.2, 2 x 16/8, 384 kept 20.6 / 22.3, 4 x 16/8, 384 kept 33.2 / 35.3, 6 x 16/8, 640
// kept 60.8 / 66.6; d = 128: 16/4, 384 kept 28.3 / 21.8, 32/8, 384 kept 27.7 / 29.8, 4652 x 8/1, 1000 kept 57.9 / 35.7; d = 256: 8/2, 100 kept
// 30.0 / 17.8, 16/8, 384 kept 38.6 / 40.8, 2 x 16/8, 640 kept 83.4 / 93.3, 4 x 16/16, 256 kept 118 / 129.  Of 956 backward calls (256 to 8000 rows, 64
// to 2048 kept) the rule of sums_by_chains costs more than 3 % over the better way on 27, 9 % at most (3001 x 8/4, d = 256, 1024 kept, the launch 65.2 /
// 60.9); all by one thread 230 and 76 %, all side by side 173 and 16 %.
template <typename T, int D>
__device__ __forceinline__ void dkdv_reduce_blocks(const BwdParams &p, const int rb, const int nrb, const int tid, float *lds) {
    using E = Elem<T>;
    const FwdParams &f = p.f;
    const int32_t *plan = f.cmp.plan;
    const int U = plan[0], Gs = plan[1], Sm = plan[2], Q = plan[4], per = Gs * Sm;
    if (per == 1) return;  // no unit was split: the dK/dV kernel wrote the results itself
    if (!plan[7]) {
        for (int item = rb; item < U * (D / 16); item += nrb) dkdv_reduce_item<T, D>(p, item / (D / 16), item % (D / 16), tid);
        return;
    }
    // a plan whose lists overflowed left parts uncomputed: every sum starts from NaN then
    const float start = plan[6] != 0 ? __builtin_nanf("") : 0.f;
    // (what the items need of the launch's arguments is read here, and what their results need at the head of an item: read where it is
    // used, behind barriers, it was a trip to memory each time)
    const int Hk = f.Hk, G = f.H / Hk, gper = G / Gs, n_pairs = f.B * Hk, Lq = f.Lq, Lk = f.Lk, causal = f.causal, ld = f.cmp.ld;
    const int32_t *idx0 = f.cmp.idx, *counts = f.cmp.count;
    const float *dkv_part = p.dkv_part, *db_part = p.db_part;
    const bool with_bias = f.bias != nullptr, per_head = f.Hb == f.H, one_row = f.Hb == 1;
    const int n_ch = (f.d + 7) / 8, ipu = 2 * n_ch + (with_bias ? 1 : 0);  // items per unit
    const int total = U * ipu, share = (total + nrb - 1) / nrb;
    const int kk = tid >> 1, hf = tid & 1;  // the key, and half of the eight columns, that this thread writes
    int unit = -1, b = 0, hk = 0, n_seg = 1, okey = 0;
    bool live = false;
    for (int i = 0; i < share; i++) {
        const int item = rb * share + i, y = item % ipu;
        const bool ok = item < total;
        if (ok && item / ipu != unit) {
            unit = item / ipu;
            int lo = 0, hi = n_pairs;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (plan[DKDV_PLAN_HDR + mid] <= unit) lo = mid;
                else hi = mid;
            }
            b = lo / Hk;
            hk = lo % Hk;
            const int n0 = (unit - plan[DKDV_PLAN_HDR + lo]) * KV_BN;
            const int32_t *idx = idx0 + (int64_t)lo * ld + n0;
            live = n0 + kk < counts[lo];
            okey = live ? idx[kk] : 0;
            // segments of this unit that were written (same rule as in the main kernel)
            n_seg = dkdv_segments(dkdv_query_blocks(Lq, Lk, causal, idx[0]), Q, Sm);
        }
        const int n_w = Gs * n_seg, mat = y >= n_ch ? 1 : 0, c = y - mat * n_ch;
        const bool cols = y == 2 * n_ch;
        const int slots = n_w >= 16 ? 8 : (n_w >= 8 ? 4 : (n_w >= 4 ? 2 : 1));
        const float *dbp = db_part + (int64_t)unit * per * G * KV_BN;  // [part][local head][key]
        uint16_t *dst = mat == 0 ? (uint16_t *)p.dk + b * p.dk_b + hk * p.dk_h : (uint16_t *)p.dv + b * p.dv_b + hk * p.dv_h;
        const int64_t dst_r = mat == 0 ? p.dk_r : p.dv_r;
        const float m = mat == 0 ? f.scale : 1.f;
        if (ok && !cols) {
            const float *base = dkv_part + ((int64_t)unit * per * 2 * D + mat * D + c * 8) * KV_BN;
            if (slots == 8) dkdv_reduce_rows<8, D>(base, n_w, n_seg, Sm, tid, lds);
            else if (slots == 4) dkdv_reduce_rows<4, D>(base, n_w, n_seg, Sm, tid, lds);
            else if (slots == 2) dkdv_reduce_rows<2, D>(base, n_w, n_seg, Sm, tid, lds);
            else dkdv_reduce_rows<1, D>(base, n_w, n_seg, Sm, tid, lds);
        } else if (ok && !per_head) {  // every eighth (part, local head) to a row of threads
            const int row = tid >> 5, quad = tid & 31, n = n_w * gper;
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
            for (int j = row; j < n; j += 32) {
                f32x4_t v[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const int jt = j + 8 * t < n ? j + 8 * t : n - 1, pt = jt / gper;
                    v[t] = *(const f32x4_t *)(dbp + ((int64_t)(pt / n_seg * Sm + pt % n_seg) * G + jt % gper) * KV_BN + 4 * quad);
                }
#pragma unroll
                for (int t = 0; t < 4; t++)
                    if (j + 8 * t < n) acc += v[t];
            }
            *(f32x4_t *)(lds + row * RED_PITCH + 4 * quad) = acc;
        }
        __syncthreads();
        auto emit = [&](int hb, float tot) {
            if (p.dbias_accum) atomicAdd(p.dbias_accum + b * p.dba_b + hb * p.dba_h + okey, tot);
            else ((uint16_t *)p.dbias)[b * p.db_b + hb * p.db_h + okey] = (uint16_t)(E::pack2(tot, 0.f) & 0xffffu);
        };
        if (ok && live && !cols) {
            float a[4];
#pragma unroll
            for (int e = 0; e < 4; e++) a[e] = start;
            for (int s = 0; s < slots; s++)
#pragma unroll
                for (int e = 0; e < 4; e++) a[e] += lds[(s * 8 + 4 * hf + e) * RED_PITCH + kk];
            *(u32x2_t *)(dst + (int64_t)okey * dst_r + c * 8 + 4 * hf) = u32x2_t{E::pack2(a[0] * m, a[1] * m), E::pack2(a[2] * m, a[3] * m)};
        } else if (ok && live && per_head) {
            for (int gi = hf; gi < G; gi += 2) {
                float tot = start;
#pragma unroll 4
                for (int sg = 0; sg < n_seg; sg++) tot += dbp[((int64_t)((gi / gper) * Sm + sg) * G + gi % gper) * KV_BN + kk];
                emit(hk * G + gi, tot);
            }
        } else if (ok && live && hf == 0) {
            float tot = start;
#pragma unroll
            for (int s = 0; s < 8; s++) tot += lds[s * RED_PITCH + kk];
            emit(one_row ? 0 : hk, tot);
        }
        __syncthreads();
    }
}

}  // namespace

}  // namespace fdma
