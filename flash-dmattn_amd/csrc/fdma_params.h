// Kernel argument blocks (device side) and the launch functions each .hip file exports to the
// C-ABI layer in fdma_api.cpp.  Plays the role of the reference's Flash_fwd_params /
// Flash_bwd_params (csrc/flash_sparse_attn/src/flash.h:20-198) without any torch types.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <cmath>

namespace fdma {

// Column compaction for keep-masks that are broadcast over queries: the kept keys of every
// (batch, kv head) pair are gathered, in ascending column order, into dense copies of K and V, and the
// main kernels then run over `count` keys instead of Lk.  Causal masking compares against the number of
// kept columns a query can see (`cnt`), and gradients are written back through `idx`.
struct Compact {
    const int32_t *idx;    // (B*Hk, ld): original column of compacted key c, c < count
    const int32_t *cnt;    // (B*Hk, ld): kept keys among the original columns 0..j (inclusive)
    const int32_t *count;  // (B*Hk): kept keys
    const float *fb;       // (B*Hfb, ld): bias * log2(e) of compacted key c (0 without a bias)
    const int32_t *plan;   // backward only: work split of the dK/dV kernel, see DkdvPlan
    int32_t ld;            // row stride of the arrays above (Lk rounded up to 16)
    int32_t Hfb;           // heads of fb: Hk, or H when the bias differs per query head
    int32_t on;            // 0 = no compaction: k / v are the caller's tensors
    // Tile images (forward at head dim 128 on large grids, see fwd_stream_applicable): instead of row-major copies the
    // pre-pass writes, per 64-key tile of the compacted key axis, exactly the bytes the forward kernel keeps in LDS --
    // the K tile with padded rows (times softmax_scale * log2(e)) followed by V already transposed (img_kv, IMG_KV_BYTES per tile, img_tiles tiles per
    // (batch, kv head) pair) and the 16-element side rows of the keys (img_x, IMG_X_BYTES per tile, per (batch, fb
    // head)) -- so that the forward fetches a tile with contiguous global->LDS loads.  nullptr = row-major copies.
    const char *img_kv;
    const char *img_x;
    int32_t img_tiles;
};
constexpr int IMG_BN = 64;                                // keys per tile image
constexpr int IMG_SK = 128 + 8, IMG_SVT = IMG_BN + 8;     // row strides (elements) of the K tile and of V^T
constexpr int IMG_K_BYTES = IMG_BN * IMG_SK * 2;          // 17408
constexpr int IMG_VT_BYTES = 128 * IMG_SVT * 2;           // 18432
constexpr int IMG_KV_BYTES = IMG_K_BYTES + IMG_VT_BYTES;  // 35840 = 35 pieces of 1 KB
constexpr int IMG_X_BYTES = IMG_BN * 32;                  // 2048

// Work split of the compacted dK/dV kernel, made on the device once the kept-key counts are known.
// A unit is one 128-key block of one (batch, kv head) pair; U = number of units.  With few units the
// chip would idle (the kernel keeps K / V stationary and loops over query heads and query blocks), so
// every unit is split over `Gs` groups of query heads and, once every head has its own group, over
// segments of at most `Q` query blocks (a unit that fewer queries see gets fewer segments, so that parts
// are of similar size); each part writes fp32 partial results that a reduce kernel sums in a fixed order.
// Units go to the 8 XCDs (workgroup id % 8) pair by pair so that workgroups sharing an L2 stream the same
// Q / dO tiles; with fewer than 8 pairs (or a pair count that 8 does not divide) a pair is folded into
// k = 8 / gcd(pairs, 8) lists, unit u going to list snake(u mod 2k) -- low key blocks see the most queries
// under a causal mask, and the fold gives every list the same mix of heavy and light units.
//   plan[0] = U, plan[1] = Gs, plan[2] = Sm (segment slots per unit and head group), plan[3] = list length
//   bound (units), plan[4] = Q, plan[5] = where the lists begin, plan[6] = 1 when a per-XCD list overflowed (the
//   reduce kernel then writes NaN gradients), plan[7] = how the parts are summed (sums_by_chains), plan[8 + i] = first unit of pair i (i = 0..pairs)
constexpr int DKDV_PLAN_HDR = 8;
#ifndef FDMA_DKDV_TARGET
#define FDMA_DKDV_TARGET 768
#endif
constexpr int DKDV_TARGET_PARTS = FDMA_DKDV_TARGET;   // parts wanted (3 per CU, two of them resident at a time: measured best)
constexpr int DKDV_ENOUGH_UNITS = 384;    // from here on the units alone fill the chip
__host__ __device__ inline void dkdv_split(int U, int G, int &Gs, int &Sm) {
    Gs = 1;
    Sm = 1;
    if (U <= 0 || U >= DKDV_ENOUGH_UNITS) return;
    const int want = (DKDV_TARGET_PARTS + U - 1) / U;
    for (int c = 2; c <= G && c <= want; c++)
        if (G % c == 0) Gs = c;  // query heads first: largest divisor of G not above `want`
    if (Gs == G) {  // upper bound of the segments per unit: twice the even split, units differ in length
        Sm = 2 * want / G;
        Sm = Sm < 1 ? 1 : (Sm > 16 ? 16 : Sm);
    }
}
// How the parts of the units are summed (plan[7], see dkdv_reduce_blocks): by several chains of loads side by side, or every sum by
// one thread, whose trips to memory for four slots follow each other.  `nwg`: workgroups (halves of one at head dims above 128) that
// sum; wait: how much of dQ waits for a CU, from 0 (at most one workgroup per CU) to 1.  One thread is enough while its trips hide
// behind the longest row block's own chain of key tiles: about 0.8 / 1 / 4 trips' time (1.9 us) per unit of a pair at d = 64 / 128 / 256 (head dims in
// between: the next larger), and 2 / 4 / 8 where dQ goes on behind it anyway.
__host__ __device__ inline bool sums_by_chains(int U, int per, int pairs, int d, int nwg, float wait) {
    const int dpad = d <= 64 ? 64 : (d <= 128 ? 128 : 256), trips = (U * (dpad / 16) + nwg - 1) / nwg * ((per + 3) / 4);
    const float alone = d <= 64 ? 0.8f : (d <= 128 ? 1.f : 4.f), beside = d <= 64 ? 2.f : (d <= 128 ? 4.f : 8.f);
    return (float)trips > 2.f + (alone + (beside - alone) * wait) * (float)U / (float)pairs;
}
// query blocks (of 64 rows) that see a key block whose first key sits at original column `okey_first`
__host__ __device__ inline int dkdv_query_blocks(int Lq, int Lk, int causal, int okey_first) {
    const int M_blocks = (Lq + 63) / 64;
    int m_start = 0;
    if (causal) {
        const int first_q = okey_first - (Lk - Lq);
        if (first_q > 0) m_start = first_q / 64;
        if (m_start > M_blocks) m_start = M_blocks;
    }
    return M_blocks - m_start;
}
// segments a unit with n_tot query blocks is cut into
__host__ __device__ inline int dkdv_segments(int n_tot, int Q, int Sm) {
    const int s = (n_tot + Q - 1) / Q;
    return s < Sm ? s : Sm;
}

__host__ __device__ inline int dkdv_lists_per_pair(int pairs) {
    return pairs % 8 == 0 ? 1 : (pairs % 4 == 0 ? 2 : (pairs % 2 == 0 ? 4 : 8));
}
// The units of a pair are dealt to its k lists in a snake (0 .. k-1, k-1 .. 0, ...): position `pos` of list `fold`
// holds unit dkdv_unit_at(pos, fold, k); unit u sits in list dkdv_list_of(u, k).
__host__ __device__ inline int dkdv_unit_at(int pos, int fold, int k) {
    return 2 * k * (pos >> 1) + ((pos & 1) ? 2 * k - 1 - fold : fold);
}
__host__ __device__ inline int dkdv_list_of(int u, int k) {
    const int rem = u & (2 * k - 1);  // (k is 1, 2, 4 or 8)
    return rem < k ? rem : 2 * k - 1 - rem;
}
__host__ __device__ inline int dkdv_list_len(int units_in_largest_pair, int k) {
    return 2 * ((units_in_largest_pair + 2 * k - 1) / (2 * k));
}

constexpr int KV_PART_MIN = 4, KV_PART_TRADE = 18;  // see plan_kv_parts
// dK/dV kernel on the original key axis (no compaction; ragged batches): a unit is one 128-key block of a (batch, kv head) pair,
// its steps are the query blocks of `bm` rows that see it, query head after query head.  A unit of many steps is cut into parts of
// about `quota` steps, which leave fp32 sums that a launch of its own adds up in part order.
__host__ __device__ inline int kv_step_rows(int d) { return d <= 64 ? 64 : 32; }
// steps per query head of the unit whose first key is n0 (the kernel walks planning blocks of 64 rows from the first that sees it)
__host__ __device__ inline int kv_unit_steps(int Lq, int Lk, int causal, int n0, int bm) {
    const int blocks = (Lq + 63) / 64, first = blocks - dkdv_query_blocks(Lq, Lk, causal, n0);
    const int steps = (Lq + bm - 1) / bm - first * (64 / bm);
    return steps > 0 ? steps : 0;
}
// all steps of one query head's units (exact without a causal mask and for Lq == Lk up to the rounding of blocks)
__host__ __device__ inline int64_t kv_head_steps(int Lq, int Lk, int causal, int bm) {
    if (Lq <= 0 || Lk <= 0) return 0;  // (what a ragged batch has beside its longest entry, when the caller names more than there is)
    const int64_t n = (Lk + 127) / 128, most = kv_unit_steps(Lq, Lk, causal, 0, bm), least = n > 0 ? kv_unit_steps(Lq, Lk, causal, (int)(n - 1) * 128, bm) : 0;
    return n * (most + least) / 2;
}
// Steps per part when a call's units have `total` steps together: the square root of total / KV_PART_TRADE, rounded up.
__host__ __device__ inline int kv_part_quota(int64_t total) {
    const int64_t x = (total + KV_PART_TRADE - 1) / KV_PART_TRADE;
    int64_t q = (int64_t)sqrtf((float)x);
    while (q * q < x) q++;
    while (q > 1 && (q - 1) * (q - 1) >= x) q--;  // (the same on the host and on the device, whatever their square roots round to)
    return (int)(q < KV_PART_MIN ? KV_PART_MIN : q);
}
__host__ __device__ inline int kv_parts_of(int steps, int quota, int most) {
    if (steps <= quota + (quota >> 2)) return 1;
    const int n = (steps + quota - 1) / quota;
    return n < most ? n : most;
}

// Row `i` of the piece of 16 rows that starts at row `first` of a matrix of `rows` (the last one where it has fewer), in bytes: where
// the piece starts, the same for all lanes and of any size (a per-query dBias of 46352 keys has 4 GiB), and a lane's way from there
// (rows below 2^25 bytes).
struct RowPiece {
    int64_t base;
    uint32_t off;
};
__host__ __device__ inline RowPiece row_piece(int first, int rows, int i, uint32_t row_bytes) {
    const int last = rows - 1 - first;
    return {(int64_t)first * row_bytes, (uint32_t)(i < last ? i : last) * row_bytes};
}

// The key that an 8-key chunk of a mask or bias row is fetched from, for the chunk that starts at key kk (a multiple of 8): one that keeps
// the load inside a row of at least 8 keys (shorter rows are readable up to 8: fdma.h).  ODD = false: rows of whole chunks.
template <bool ODD> __host__ __device__ inline int chunk8_at(int kk, int Lk) {
    if (!ODD) return kk < Lk ? kk : 0;
    const int last = Lk >= 8 ? Lk - 8 : 0;
    return kk < last ? kk : last;
}
// Where the 8 bytes lie that hold this chunk of a mask row: its mask bytes or, of a mask packed to bits, the aligned piece of the bit row
// with the chunk's byte.  (One form for both: a choice between two addresses becomes two loads.)
__host__ __device__ inline int mask_piece_at(bool bits, int kk, int Lk) {
    const int last = bits ? Lk - 1 : (Lk >= 8 ? Lk - 8 : 0), k = kk < last ? kk : last;
    return (k >> (bits ? 3 : 0)) & (bits ? ~7 : ~0);
}

// Division by a number that the launch knows, of anything below 2^31: two products and a shift on the scalar unit where the general one
// is thirty vector instructions and a reciprocal.  (mul = ceil(2^(31 + shift) / by) with 2^shift >= by is off by less than
// by / 2^(31 + shift) of the quotient's step.)
struct Divisor {
    uint32_t by, mul, shift;
};
inline Divisor divisor(uint32_t by) {
    uint32_t s = 0;
    while (s < 31 && (1u << s) < by) s++;
    return {by, (uint32_t)((((uint64_t)1 << (31 + s)) + by - 1) / by), 31 + s};
}
__host__ __device__ inline int quotient(int n, const Divisor &d) { return (int)(((uint64_t)(uint32_t)n * d.mul) >> d.shift); }

struct FwdParams {
    const void *q, *k, *v;
    const uint8_t *mask;  // nullptr = absent
    const void *bias;     // nullptr = absent
    void *o;
    float *lse;           // element (b, h, row) at b * lse_b + h * lse_h + first row of b + row
    int64_t lse_b, lse_h; // (B, H, Lq): H * Lq, Lq; ragged batch (H, total_q): 0, total_q
    // Ragged batch (the reference's "varlen" layout, csrc/flash_sparse_attn/flash_api.cpp:556-790): q / k / v hold the
    // sequences back to back, (total rows, heads, d), batch entry b owns rows cu[b] .. cu[b + 1] - 1 and the batch
    // strides are 0.  Lq / Lk below are then the longest sequences (they size the grids).  nullptr = fixed lengths.
    const int32_t *cu_q, *cu_k;
    int32_t total_q, total_k;  // rows of the ragged q / k tensors
    int64_t q_b, q_r, q_h;
    int64_t k_b, k_r, k_h;
    int64_t v_b, v_r, v_h;
    int64_t o_b, o_r, o_h;
    int64_t m_b, m_h, m_r;  // mask strides (batch, head, row); 0 = broadcast
    int64_t bi_b, bi_h, bi_r;
    int32_t B, Lq, Lk, H, Hk, Hm, Hb, d;
    int32_t causal;
    float scale;        // softmax scale
    float scale_log2;   // scale * log2(e)
    // split-KV decode
    float *o_part;      // (splits, B, H, Lq, d) fp32
    float *lse_part;    // (splits, B, H, Lq) fp32, natural log, -inf for an empty split
    int32_t splits;
    // split-KV decode in one launch: one arrival counter per (batch entry, workgroup row of the grid), zero on entry and
    // left zero (fdma_fwd_args.counters of the C ABI); nullptr = the merge is a launch of its own
    int32_t *dec_counter;
    int32_t compact_mode;  // FDMA_COMPACT_* of the C ABI: 0 = decide from the problem, 1 = never, 2 = whenever the mask form allows
    Compact cmp;        // when cmp.on, k / v (and their strides) describe the compacted copies
    // kept-column lists handed over by the caller (fdma_kept_keys of the C ABI; nullptr = scan the mask): one row per
    // (mask batch entry, mask head)
    const int32_t *kept_idx, *kept_cnt, *kept_count;
    int32_t kept_ld;
    // Forward compaction for a query-broadcast mask with one row per QUERY head (Hm == H > kv heads): every query head
    // keeps its own keys, so the heads of a kv group share no compacted K / V.  The compaction layer then sees H "kv
    // heads" (Hk == H above, one compacted copy per query head) and finds the caller's K / V / bias head of such a head
    // by dividing by kv_share (= query heads per real kv head).  0 or 1: heads are what they say.
    int32_t kv_share;
    // the mask packed to one bit per key (fdma_mask_bits of the C ABI; nullptr = read the bool mask): strides in bytes,
    // broadcast like the mask
    const uint8_t *mbits;
    int64_t mb_b, mb_h, mb_r;
    // set by row_grid for row_unit: log2 of the lists that the row blocks of a pair are dealt to, -1: whole ragged entries; query heads
    // per kv head; workgroups of a turn of lists, lists side by side in it, kv heads
    int32_t row_lists;
    Divisor row_group, row_turn, row_side, row_heads;
};

// the caller's kv head behind head `hk` of the compaction layer (see FwdParams::kv_share)
__host__ __device__ inline int kv_head(const FwdParams &p, int hk) { return p.kv_share > 1 ? hk / p.kv_share : hk; }

// lengths and first rows of batch entry b
struct SeqInfo {
    int32_t Lq, Lk;
    int64_t q0, k0;
};
__device__ inline SeqInfo seq_info(const FwdParams &p, int b) {
    SeqInfo s;
    if (p.cu_q) {
        const int32_t q0 = p.cu_q[b], k0 = p.cu_k[b];
        s.q0 = q0;
        s.k0 = k0;
        s.Lq = p.cu_q[b + 1] - q0;
        s.Lk = p.cu_k[b + 1] - k0;
    } else {
        s.q0 = 0;
        s.k0 = 0;
        s.Lq = p.Lq;
        s.Lk = p.Lk;
    }
    return s;
}

// Workgroup -> (batch, kv head) pair and block of `bm` query rows, for the kernels that walk the keys of their rows (G workgroups per
// block: the query heads of the group), heaviest block first.  The blocks of a pair are dealt to k lists, the lists go to the XCDs in
// turn (a workgroup's XCD is its id % 8).  k is as small as it can be with all lists coming out even, which keeps a pair's K / V in few
// L2s: over all pairs where they have one length, over the kv heads of an entry where the batch is ragged -- otherwise the XCD
// that has the longest entry works alone.  The lists of a ragged entry go on where the blocks of those in front of it have ended.
// Over all pairs / over the heads, forward (us): entries of 18, 256, 1774, 4, 2696, 73, 22, 2677 x 2/1 heads, d = 128 60.0 / 39.3; 1000,
// 300, 500, 2000 x 8/2, d = 256 82 / 59; 4000, 100, 30, 200, 5, 60 x 8/2, d = 64 63.8 / 39.8; eight of 600 x 16/4, d = 256 57.9 / 62.1.
// Where the longest entry has fewer blocks than there are lists, most lists of an entry would be empty, and a workgroup without a block
// holds its place on a CU until it has seen that: whole entries go to the XCDs in turn there, eight pairs a turn, each turn from the
// next XCD on.  Lists of every entry / whole entries, forward (us): 64 entries of 60 to 128 rows x 8/1 heads, d = 128 41 / 22, d = 64 20.2 /
// 10.4; 256 of 64 x 16/2 178 / 129; 33 of 100 x 6/3, d = 96 14.2 / 9.8; 13 of 300 to 700 x 12/3 33.6 / 29.8.  (Whole entries up to 32
// workgroups each in batches of eight times the longest: 8 of 600 x 16/4 36.3 / 32.0, 16 of 2000 x 8/2 181 / 160, but 9 of 900 x 16/16 71 /
// 86, 200 of 20 to 400 x 8/4 137 / 165, 20 of 100 to 600 x 16/4, d = 256 78 / 88.)
inline int row_grid(FwdParams &p, int bm) {
    const int n = p.cu_q ? p.Hk : p.B * p.Hk, n_mb = (p.Lq + bm - 1) / bm;
    const int log_k = n % 8 == 0 ? 0 : (n % 4 == 0 ? 1 : (n % 2 == 0 ? 2 : 3)), k = 1 << log_k;
    const bool whole = p.cu_q && n_mb < k;
    p.row_lists = whole ? -1 : log_k;
    const int G = p.H / p.Hk, list_len = (whole ? n_mb : (n_mb + k - 1) / k) * G, side = p.cu_q && !whole ? p.Hk * k / 8 : 1;
    p.row_group = divisor(G);
    p.row_turn = divisor(list_len > 0 ? list_len * side : 1);
    p.row_side = divisor(side);
    p.row_heads = divisor(p.Hk);
    return (whole ? (p.B * p.Hk + 7) / 8 * 8 * n_mb : p.B * p.Hk * k * ((n_mb + k - 1) / k)) * G;
}
struct RowUnit {
    int pair, block;  // block < 0: none
    int b, hk, h;     // of the pair: batch entry and kv head; this workgroup's query head
};
__host__ __device__ inline RowUnit row_unit(const FwdParams &p, int id, int bm) {
    const bool whole = p.row_lists < 0;
    const int log_k = whole ? 0 : p.row_lists, k = 1 << log_k, n_mb = (p.Lq + bm - 1) / bm;
    // Of a ragged batch an XCD's lists of one entry run side by side, heaviest blocks first (more than 8 kv heads; one after the other /
    // side by side, forward: seven entries of 300 and one of 2000 x 12/12, d = 128 78 / 56; 2500 and 2500 x 24/12, d = 96 114 / 102).
    const int slot = id / 8, turn = quotient(slot, p.row_turn), in_turn = slot - turn * (int)p.row_turn.by;
    const int at = quotient(in_turn, p.row_group), g = in_turn - at * (int)p.row_group.by;
    const int pos = quotient(at, p.row_side), vlist = id % 8 + 8 * (turn * (int)p.row_side.by + at - pos * (int)p.row_side.by);
    int pair = vlist >> log_k;
    if (whole) {
        pair = (pair & ~7) | ((pair - (pair >> 3)) & 7);
        if (pair >= p.B * p.Hk) return {0, -1, 0, 0, 0};
    }
    const int b = quotient(pair, p.row_heads), hk = pair - b * p.Hk;
    int blocks = n_mb, fold = vlist & (k - 1);  // of this pair; this list
    if (p.cu_q) {
        const int q0 = p.cu_q[b], own = (p.cu_q[b + 1] - q0 + bm - 1) / bm;
        blocks = own < n_mb ? own : n_mb;  // (rows beyond the longest length that the caller names are not computed)
        fold = (fold - q0 / bm - b) & (k - 1);
    }
    const int rank = (pos << log_k) + fold;  // from the last block down
    return {pair, rank < blocks ? blocks - 1 - rank : -1, b, hk, hk * (int)p.row_group.by + g};
}

// Lists of units per (batch, kv head) pair, so that the lists of a ragged batch fill the 8 XCDs: the heads of ONE entry go to
// all of them (8 entries with one kv head each would otherwise put an entry on each XCD, and the call takes as long as the
// longest entry needs on 32 CUs).
__host__ __device__ inline int ragged_lists_per_pair(const FwdParams &p) {
    return p.Hk % 8 == 0 ? 1 : (p.Hk % 4 == 0 ? 2 : (p.Hk % 2 == 0 ? 4 : 8));
}

struct BwdParams {
    FwdParams f;  // f.o = forward output (read), f.lse = forward LSE (read)
    const void *dout;
    void *dq, *dk, *dv, *dbias;
    int64_t do_b, do_r, do_h;
    int64_t dq_b, dq_r, dq_h;
    int64_t dk_b, dk_r, dk_h;
    int64_t dv_b, dv_r, dv_h;
    int64_t db_b, db_h, db_r;  // dbias strides (batch, head, row); 0 = broadcast
    float *softmax_d;          // laid out like lse: b * sd_b + h * sd_h + first row of b + row
    int64_t sd_b, sd_h;        // (B, H, Lq_rounded): H * Lq_rounded, Lq_rounded; ragged batch: 0, total_q
    int32_t Lq_rounded;
    float *dbias_accum;        // fp32 scratch at the dbias shape when several workgroups share an element
    int64_t dba_b, dba_h, dba_r;
    int32_t kv_segs;           // general dK/dV kernel: segments of the query blocks (1 = no split; see general_kv_segments)
    // general dK/dV kernel with segments: per part [2][128][Dpad] fp32 (dK, dV, in register order) and [G][128] fp32 (dBias
    // columns).  Compacted dK/dV kernel, split mode: per part [2][Dpad][128] fp32 (dK^T, dV^T) and [G][128] fp32 (dBias)
    float *dkv_part;
    float *db_part;
    // dK/dV on the original key axis, cut into parts: most parts of a unit (1 = no cut), steps per part (0: ragged, from the
    // lengths on the device), units per (batch, kv head) pair -- ragged: per kv head.  Per part [2][Dpad][128] fp32 (dK, dV, in
    // register order) in dkv_part and [G][128] fp32 (dBias columns) in db_part
    int32_t kv_most, kv_quota, kv_units;
    // general form, dQ: shares that the key tiles of a row block are cut into (1: none), and their fp32 sums (shares, B, H, Lq, d)
    int32_t dq_shares;
    float *dq_part;
    int32_t dot_done;          // softmax_d has been computed by an earlier launch of this call
    int32_t red_first, red_count;  // compacted backward: workgroups of the dQ launch that sum the dK/dV partials (see place_reduction)
    float red_wait;                // how much of dQ waits for a CU beside them, 0 .. 1
};

// Keep-mask builder (fdma_mask.hip): one row of `Lk` 16-bit bias values per (batch, head, row).
struct MaskParams {
    const void *bias;
    const uint8_t *mask_in;  // nullptr = absent; 0 strides broadcast
    uint8_t *mask_out;
    int64_t bi_b, bi_h, bi_r;
    int64_t mi_b, mi_h, mi_r;
    int64_t mo_b, mo_h, mo_r;
    int32_t batch, heads, rows, Lk;
    int32_t window;      // top-k: entries kept per row
    int32_t block_size;  // > 1: majority vote inside aligned key blocks afterwards
    int32_t type;        // 0 = top-k, 1 = relu
    int32_t dtype;       // 0 = bf16, 1 = fp16
    uint32_t min_bits;   // the fill value for entries the incoming mask excludes, as bits of the bias type
    int32_t *kept_idx, *kept_cnt, *kept_count;  // optional second output (nullptr = not wanted): see scan_mask_row
    int32_t kept_ld;
    uint8_t *bits;           // optional third output (nullptr = not wanted): the mask packed to one bit per key
    int64_t bits_row_bytes;
};
hipError_t launch_make_mask(const MaskParams &p, hipStream_t stream);

// Bias producer (fdma_bias.hip): bias[b, j, 0, l] = A[j] * softplus(V_flat[b, l, :] . W[j, :] + pb[j]).
struct DynBiasParams {
    const void *v;        // (B, L, Hk, d): strides batch / row / head in elements, d contiguous
    const void *w;        // (Hk, Hk * d) row-major
    const void *pb;       // (Hk) or nullptr
    const void *a;        // (Hk)
    void *bias;           // out (forward): element (b, j, l) at b * bias_b + j * bias_h + l
    float *dt;            // (B * L, Hk) fp32: written by forward, read by backward
    int64_t v_b, v_r, v_h;
    int64_t bias_b, bias_h;
    int32_t B, L, Hk, d;
    // backward
    const void *dbias;    // (b, j, l) at b * dbias_b + j * dbias_h + l
    int64_t dbias_b, dbias_h;
    void *dv;             // (B, L, Hk, d), strides below
    int64_t dv_b, dv_r, dv_h;
    void *dw, *da, *dpb;  // (Hk, Hk * d), (Hk), (Hk) or nullptr
    float *part;          // n_wg partials of part_stride floats: dW (Hk * Hk * d), dA (Hk), dpb (Hk)
    int64_t part_stride;
    int32_t n_wg, rows_per_wg, col_waves;
};
hipError_t launch_dyn_bias_fwd(const DynBiasParams &p, int dtype, hipStream_t stream);
hipError_t launch_dyn_bias_bwd(const DynBiasParams &p, int dtype, hipStream_t stream);
int dyn_bias_bwd_workgroups(int64_t n_rows, int Hk, int d, int *rows_per_wg, int *col_waves);
int dyn_bias_bwd_parts(int64_t n_rows, int Hk, int d);  // partial results that a caller makes room for: at least as many

// Dynamic-LDS limit of a kernel, raised once per device (and again only for a larger request) instead of on every
// launch: one `static DynSmemLimit` per launch site.  Later launches make no runtime call besides the launch itself.
struct DynSmemLimit {
    static constexpr int kDevices = 16;
    std::atomic<int> set_bytes[kDevices] = {};
    hipError_t ensure(const void *kernel, int bytes) {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const bool tracked = dev >= 0 && dev < kDevices;
        if (tracked && set_bytes[dev].load(std::memory_order_acquire) >= bytes) return hipSuccess;
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e == hipSuccess && tracked) {
            int seen = set_bytes[dev].load(std::memory_order_relaxed);
            while (seen < bytes && !set_bytes[dev].compare_exchange_weak(seen, bytes, std::memory_order_release)) {}
        }
        return e;
    }
};

// dtype: 0 = bf16, 1 = fp16.  All launches are asynchronous on `stream`; return hipError_t.
hipError_t launch_fwd(const FwdParams &p, int dtype, hipStream_t stream);
// column-mask specialisation (mask / bias absent or broadcast over queries); nq = 32-row blocks per wave
bool fwd_colmask_applicable(const FwdParams &p);
bool fwd_from_lists(const FwdParams &p);
hipError_t launch_fwd_colmask(const FwdParams &p, int dtype, hipStream_t stream);
hipError_t launch_fwd_wide(const FwdParams &p, int dtype, hipStream_t stream);  // head dims 129 .. 256 (fdma_fwd_wide.hip)
int64_t fwd_blocks64(const FwdParams &p);  // 64-row blocks of all heads (ragged batches: at most)
// compacted forward: shares the keys of a row block are cut into (1: none); p.o_part / p.lse_part then hold
// splits * B * H * Lq rows of d / 1 floats
int fwd_key_splits(const FwdParams &p);
constexpr int MAX_KEY_SPLITS = 8;
// adds the shares of a forward call up
// (without arrival counters; with them, FwdParams::dec_counter, the last workgroup of a row block does it)
hipError_t launch_fwd_merge(const FwdParams &p, int dtype, hipStream_t stream);
// general form (mask or bias per query): shares that the key tiles of a row block are cut into (1: none), forward or dQ; what
// they leave lies in o_part / lse_part or BwdParams::dq_part
int general_key_shares(const FwdParams &p, bool dq);
int64_t general_share_units(const FwdParams &p);  // row blocks of a forward in shares, a counter each
// compacted forward in shares (fwd_key_splits): row blocks, a counter each
int64_t fwd_share_units(const FwdParams &p);
int fwd_share_block(const FwdParams &p);  // rows of a row block
int key_shares(const FwdParams &p);  // ... as far as the sizes go: what they would be if the keys were compacted
// compacted forward on tile images (fdma_fwd_stream.hip): resident workgroups that walk their share of the
// (query block, head) items with the tiles of the next item already on their way.  `fwd_stream_applicable` decides from
// the problem alone (the pre-pass, the forward and the backward of a problem must agree on the workspace layout).
bool fwd_stream_applicable(const FwdParams &p);
// smallest number of (256-row query block, head) items for which it is taken (process-wide; default 512)
void set_stream_min_items(int n);
int get_stream_min_items();
hipError_t launch_fwd_stream(const FwdParams &p, int dtype, hipStream_t stream);
hipError_t launch_fwd_decode(const FwdParams &p, int dtype, hipStream_t stream);
hipError_t launch_bwd(const BwdParams &p, int dtype, hipStream_t stream);
// column-mask specialisations of the two main backward kernels
bool bwd_colmask_applicable(const BwdParams &p);
hipError_t launch_bwd_dkdv_colmask(const BwdParams &p, int dtype, hipStream_t stream);
hipError_t launch_bwd_dkdv_256(const BwdParams &p, int dtype, int grid, hipStream_t stream);  // its kernel at head dims 129 .. 256 (fdma_bwd_dkdv_256.hip)
void place_reduction(BwdParams &p);  // compacted: which workgroups of the dQ launch sum the dK/dV partials
hipError_t launch_bwd_dq_colmask(const BwdParams &p, int dtype, hipStream_t stream);
hipError_t launch_bwd_dq_256(const BwdParams &p, int dtype, int grid, hipStream_t stream);  // its kernel at head dims 129 .. 256 (fdma_bwd_dq_256.hip)
// parts the units of the dK/dV kernel on the original key axis are cut into: fills kv_most / kv_quota / kv_units and returns the
// bytes of their sums (0: whole); *db_bytes: of their dBias columns
size_t plan_kv_parts(BwdParams &p, size_t *db_bytes);
// dQ from the dS tiles that the general dK/dV kernel has written as dBias (a per-query bias with a row per query head
// and batch entry, dBias written directly): one tile GEMM and no second pass over mask, bias, Q, V, dO
bool bwd_dq_from_ds_applicable(const BwdParams &p);
hipError_t launch_bwd_dq_from_ds(const BwdParams &p, int dtype, hipStream_t stream);
// dK / dV / dBias of the general form at head dims 65 .. 128 (fdma_bwd_dkdv_wide.hip); gsum: a per-query dBias element is
// shared by several query heads
hipError_t launch_bwd_dkdv_wide(const BwdParams &p, int dtype, bool gsum, hipStream_t stream);
bool bwd_dkdv_64_applicable(const BwdParams &p);  // general form, head dims up to 64, aligned rows (fdma_bwd_dkdv_64.hip)
hipError_t launch_bwd_dkdv_64(const BwdParams &p, int dtype, hipStream_t stream);
// general forward and dQ kernels: query heads to a workgroup (fdma_fwd.hip)
int shared_rows(const FwdParams &p);
bool general_rows_256(const FwdParams &p);  // whether those of 256 rows take the call, which do not work on shares of the keys
// general dQ kernel (mask / bias per query row), fdma_bwd_dq.hip
hipError_t launch_bwd_dq(const BwdParams &p, int dtype, hipStream_t stream);

// Column compaction: use_compact() decides from the problem alone (no device data), compact_bytes() is
// the scratch it needs, compact_setup() launches the gather pre-pass into `ws` and rewrites p.k / p.v /
// p.cmp; for a backward call (bp given) the same launch zero-fills the gradient rows / columns of dropped keys
// and makes the dK/dV plan.
bool use_compact(const FwdParams &p);
// ... and does so for the length of the key axis alone (few query rows): without scratch the call can skip tiles instead
bool compact_for_long_keys(const FwdParams &p);
// forward only: `p` has a query-broadcast mask with a row per query head and grouped kv heads, and `pv` -- the same
// problem as the compaction layer takes it (see FwdParams::kv_share) -- is one that use_compact() accepts
bool compact_per_query_head(const FwdParams &p, FwdParams &pv);
size_t compact_bytes(const FwdParams &p, bool backward, bool reuse_fwd = false);
// bp != nullptr: backward -- also plans the dK/dV split and sets bp->dkv_part / bp->db_part
// `fwd_ws` (backward only): the workspace a forward call of the same problem filled; its lists and copies are used
// instead of being made again, and `ws` then holds the backward's plan and partial sums alone.
hipError_t compact_setup(FwdParams &p, void *ws, int dtype, hipStream_t stream, BwdParams *bp = nullptr,
                         const void *fwd_ws = nullptr);
// host-side bounds over every possible unit count 1..U_max: workgroups to launch, partial slots to hold
// (n_max = units of one pair at most)
inline void dkdv_split_bounds(int pairs, int n_max, int G, int &grid, int &slots) {
    const int k = dkdv_lists_per_pair(pairs);
    const int lists_per_xcd = pairs * k / 8;
    // n = units of the largest pair; the total U is then between n and pairs * n, and the split factor does
    // not grow with U: the split of U = n bounds the workgroups, U * split(U) bounds the partial slots
    int64_t items = 1, sl = 1;
    for (int n = 1; n <= n_max; n++) {
        int Gs, Sm;
        dkdv_split(n, G, Gs, Sm);
        const int64_t it = (int64_t)dkdv_list_len(n, k) * Gs * Sm;
        if (it > items) items = it;
        if (n >= DKDV_ENOUGH_UNITS) {  // no split from here on: the bound grows with n alone
            const int64_t last = dkdv_list_len(n_max, k);
            if (last > items) items = last;
            break;
        }
    }
    const int U_max = pairs * n_max < DKDV_ENOUGH_UNITS ? pairs * n_max : DKDV_ENOUGH_UNITS - 1;
    for (int U = 1; U <= U_max; U++) {
        int Gs, Sm;
        dkdv_split(U, G, Gs, Sm);
        if (Gs * Sm > 1 && (int64_t)U * Gs * Sm > sl) sl = (int64_t)U * Gs * Sm;
    }
    grid = (int)(8 * lists_per_xcd * items);
    slots = (int)sl;
}

// general dK/dV kernel: segments its query blocks are cut into, and the bytes of the segments' fp32 sums (and of their dBias
// columns) the call must provide
int general_kv_segments(const FwdParams &f);
size_t general_kv_part_bytes(const FwdParams &f, size_t *db_bytes);
// general kernels: mask or bias rows that are not made of whole, aligned 8-key chunks (see chunk8_at in fdma_common.h)
inline bool odd_rows(const FwdParams &f) {
    if (f.Lk % 8 != 0) return true;
    const bool m = f.mask && !f.mbits && (((uintptr_t)f.mask | (uintptr_t)f.m_b | (uintptr_t)f.m_h | (uintptr_t)f.m_r) & 7) != 0;
    const bool b = f.bias && (((uintptr_t)f.bias & 15) != 0 || ((f.bi_b | f.bi_h | f.bi_r) & 7) != 0);
    return m || b;
}
// compute units of the current device (256 where there is none)
int device_cus();

// number of KV splits the decode path uses for this shape, with a mask or without (1 = no workspace needed)
int decode_num_splits(int B, int H, int Hk, int Lk, int d, bool masked);
int decode_splits_at_most(int splits, int Lk);
// arrival counters the one-launch decode needs for this shape (0 without splits)
int64_t decode_num_counters(int B, int H, int Hk, int Lk, int d);
bool use_decode_path(int Lq, int H, int Hk);

}  // namespace fdma
