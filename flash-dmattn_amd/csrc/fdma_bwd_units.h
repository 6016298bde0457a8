// Work items of the column-form dK/dV kernels (fdma_bwd_colmask.hip, fdma_bwd_dkdv_256.hip): which 128 keys, query heads and query
// blocks a workgroup has, from its id.
#pragma once

#include "fdma_params.h"

namespace fdma {

namespace {

// XCD-aware work distribution shared by both kernels: `pairs` independent (batch, kv head) pairs with
// `n_units` units of work each (heaviest first), `k_split` lists of units per pair; see the forward column-mask kernel for the rationale.
struct XcdMap {
    int pair, unit;
    bool valid;
};
__host__ __device__ __forceinline__ int xcd_lists_per_pair(int pairs) {
    const int gcd8 = (pairs % 8 == 0) ? 8 : ((pairs % 4 == 0) ? 4 : ((pairs % 2 == 0) ? 2 : 1));
    return 8 / gcd8;
}
__device__ __forceinline__ XcdMap xcd_map(int lid, int k_split, int n_units, int per_unit) {
    const int list_len = ((n_units + k_split - 1) / k_split) * per_unit;
    const int xcd = lid % 8, slot = lid / 8;
    const int vlist = xcd + 8 * (slot / list_len);
    const int pos = slot % list_len;
    XcdMap m;
    m.pair = vlist / k_split;
    m.unit = (pos / per_unit) * k_split + vlist % k_split;
    m.valid = m.unit < n_units;
    return m;
}
inline int xcd_grid(int pairs, int k_split, int n_units, int per_unit) {
    return pairs * k_split * ((n_units + k_split - 1) / k_split) * per_unit;
}

constexpr int KV_BM = 64;   // query rows per planning block (the work split counts these)
constexpr int KV_BN = 128;  // key columns per workgroup (32 per wave)


// Unit `u` of a kv head's units in a ragged batch: the blocks of 128 keys of its entries, the entry with the most query rows
// first, equal ones in their order.  A block of keys walks the rows of its entry; workgroups start in the order of their ids, and
// one of a long entry that starts last runs on alone.  16384 tokens in entries of 1 to 5394, the longest last, 32 heads over 8,
// head dim 128: 1396 -> 1247 us.  Ranks and first units come from one comparison per entry and lane; a batch of more entries than a
// wave has lanes keeps its order (its units are many and small enough to even out).  Units beyond the last: block < 0.
struct RaggedUnit {
    int entry, block;
};
__device__ inline RaggedUnit ragged_unit(const FwdParams &p, int u) {
    const int lane = (int)(threadIdx.x & 63);
    if (p.B > 64) {  // (entry b's units start at cu_k[b] / 128 + b: kv_unit_slot)
        int e = -1;
        for (int base = 0; base < p.B; base += 64) {
            const int b = base + lane;
            e += __popcll(__ballot(b < p.B && p.cu_k[b] / KV_BN + b <= u));
        }
        const int len = p.cu_k[e + 1] - p.cu_k[e], n = u - (p.cu_k[e] / KV_BN + e);
        return {e, n * KV_BN < len ? n : -1};
    }
    const int b = lane < p.B ? lane : 0, len = lane < p.B ? p.cu_q[b + 1] - p.cu_q[b] : -1;
    const int n = lane < p.B ? (p.cu_k[b + 1] - p.cu_k[b] + KV_BN - 1) / KV_BN : 0;
    int first = 0;
    for (int t = 0; t < p.B; t++) {
        const int other = __builtin_amdgcn_readlane(len, t), nt = __builtin_amdgcn_readlane(n, t);
        first += (other > len || (other == len && t < lane)) ? nt : 0;
    }
    const uint64_t at = __ballot(u >= first && u < first + n);
    if (!at) return {0, -1};
    const int e = __builtin_ctzll(at);
    return {e, u - __builtin_amdgcn_readlane(first, e)};
}

// Steps per part of a ragged batch (kv_part_quota of all its units' steps): every lane takes entries, the wave adds up.
__device__ inline int ragged_part_quota(const FwdParams &p, int bm) {
    int64_t sum = 0;
    for (int b = (int)(threadIdx.x & 63); b < p.B; b += 64)
        sum += kv_head_steps(p.cu_q[b + 1] - p.cu_q[b], p.cu_k[b + 1] - p.cu_k[b], p.causal, bm);
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) sum += __shfl_xor((long long)sum, m);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)sum), hi = __builtin_amdgcn_readfirstlane((uint32_t)(sum >> 32));
    return kv_part_quota((int64_t)(((uint64_t)hi << 32) | lo) * p.H);
}
// Where the sums of a unit's parts lie: unit number within the call (times kv_most).  Ragged: entry b's blocks start at
// cu_k[b] / 128 + b, which leaves every entry the blocks it has.
__device__ inline int kv_unit_slot(const BwdParams &p, int b, int hk, int n_block) {
    const int u = p.f.cu_q ? hk * p.kv_units + p.f.cu_k[b] / KV_BN + b + n_block : (b * p.f.Hk + hk) * p.kv_units + n_block;
    return u * p.kv_most;
}

// Work item of a dK/dV workgroup: a 128-key block of one (batch, kv head) pair, over query heads [g_lo, g_hi) and segment `seg` of
// `Sm` of the query range (compacted keys, from the device-made plan) or part `part` of its steps (original key axis); `slot` >= 0
// when the block is shared by several workgroups.  turns: the entries of a ragged batch longest first (ragged_unit).
struct KvItem {
    int pair, n_block, g_lo, g_hi, seg, Sm, Q, slot, part;
    bool valid;
};
template <bool CMP> __device__ __forceinline__ KvItem kv_item(const BwdParams &p, bool turns) {
    const FwdParams &f = p.f;
    const int G = f.H / f.Hk;
    KvItem w = {0, 0, 0, G, 0, 1, 1 << 30, -1, 0, false};
    if (CMP) {
        const int32_t *plan = f.cmp.plan;
        const int Gs = plan[1];
        w.Sm = plan[2];
        w.Q = plan[4];
        const int per = Gs * w.Sm;
        int sub;
        const int x = blockIdx.x % 8, l = blockIdx.x / 8;
        if (per > 1) {
            // Split units: the plan holds, per XCD, the list of the parts that exist -- (pair, unit, part of the
            // unit), longest parts first.  Workgroup l of an XCD takes entry l; consecutive workgroups of an XCD go
            // to its shader engines in turn, and with the existing parts side by side every engine gets its share.
            const int cap = gridDim.x / 8;
            const int32_t *lists = plan + plan[5];
            if (l >= lists[x]) return w;
            const int32_t *e = lists + 8 + 2 * ((int64_t)x * cap + l);
            w.pair = e[0];
            w.n_block = e[1] & 0xffff;
            sub = e[1] >> 16;
        } else {
            // unit lists per XCD: the units of a pair are dealt to its k lists, the lists to the XCDs
            const int P = f.B * f.Hk, k = dkdv_lists_per_pair(P);
            const int list_len = plan[3];
            if (list_len == 0) return w;
            const int ls = l / list_len, pos = l % list_len;
            if (ls >= P * k / 8) return w;
            const int vlist = x + 8 * ls, fold = vlist % k;
            w.pair = vlist / k;
            w.n_block = dkdv_unit_at(pos, fold, k);
            if (w.n_block >= plan[DKDV_PLAN_HDR + w.pair + 1] - plan[DKDV_PLAN_HDR + w.pair]) return w;
            sub = 0;
        }
        const int unit = plan[DKDV_PLAN_HDR + w.pair] + w.n_block;
        const int gper = G / Gs;
        w.g_lo = (sub / w.Sm) * gper;
        w.g_hi = w.g_lo + gper;
        w.seg = sub % w.Sm;
        if (per > 1) w.slot = unit * per + sub;
    } else {
        const int n_nb = (f.Lk + KV_BN - 1) / KV_BN;
        const bool ragged = turns && f.cu_q;
        const int k = ragged ? ragged_lists_per_pair(f) : xcd_lists_per_pair(f.B * f.Hk), n_units = ragged ? p.kv_units : n_nb;
        XcdMap wm;
        if (ragged) {
            // All lists of an XCD side by side: the long entries of all its heads are under way before the short ones start.
            // One list after the other / side by side, forward + backward (us): 4000, 3000, 700, 1 x 16/16 heads, d = 64 386 / 355;
            // 900, 6000, 30 x 48/12, d = 64 1443 / 1332; six entries up to 4000 x 32/32, d = 128 1250 / 1207.  (Up to 8 lists: alike.)
            // The last parts first, see below.
            const int per_list = (n_units + k - 1) / k, nl = f.Hk * k / 8, at = (int)(blockIdx.x / 8), pos = at % (per_list * nl);
            w.part = p.kv_most - 1 - at / (per_list * nl);
            const int vlist = (int)(blockIdx.x % 8) + 8 * (pos % nl);
            wm.pair = vlist / k;
            wm.unit = pos / nl * k + vlist % k;
            wm.valid = wm.unit < n_units;
        } else if (p.kv_most > 1) {
            // A list holds its units once per part, the LAST parts first: those exist for the longest units only.  Workgroups
            // side by side go to the shader engines of an XCD in turn, whether they stay or return at once: with the parts of
            // a unit side by side instead, the engines that got the missing ones idled (ragged, 16384 tokens, two parts at
            // most: 1966 us instead of 1224 without parts).
            const int per_list = (n_units + k - 1) / k, pos = (int)(blockIdx.x / 8) % (per_list * p.kv_most);
            w.part = p.kv_most - 1 - pos / per_list;
            const int vlist = (int)(blockIdx.x % 8) + 8 * ((int)(blockIdx.x / 8) / (per_list * p.kv_most));
            wm.pair = vlist / k;
            wm.unit = pos % per_list * k + vlist % k;
            wm.valid = wm.unit < n_units;
        } else {
            wm = xcd_map(blockIdx.x, k, n_units, 1);
        }
        if (!wm.valid) return w;
        w.n_block = wm.unit;  // low key blocks are seen by the most queries under causal: heaviest first
        w.pair = wm.pair;
        if (ragged) {
            const RaggedUnit ru = ragged_unit(f, w.n_block);
            if (ru.block < 0 || ru.block >= n_nb) return w;  // (rows beyond the longest length that the caller names: not computed)
            w.n_block = ru.block;
            w.pair = ru.entry * f.Hk + wm.pair;
        }
    }
    w.valid = true;
    return w;
}

}  // namespace

}  // namespace fdma
