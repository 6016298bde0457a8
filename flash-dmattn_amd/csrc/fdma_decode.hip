// Single-token decode (seqlen_q == 1) for gfx950: split-KV partial attention + LSE-weighted combine -- in ONE launch
// when the caller provides arrival counters (the last workgroup of a (batch entry, head chunk) to finish merges the
// splits), otherwise as a second launch.
//
// Replaces the reference's decode route: the `seqlenq_ngroups_swapped` reshaping of mha_fwd
// (csrc/flash_sparse_attn/flash_api.cpp:443-475, 541-551), num_splits_heuristic (:275-349),
// compute_attn_1rowblock_splitkv (csrc/flash_sparse_attn/src/flash_fwd_kernel.h:808-1587) and
// combine_attn_seqk_parallel (:1618-1813).
//
// The path is bound by HBM reads of K and V.  A key/value row of one KV head is d*2 contiguous bytes,
// so skipping can be done per KEY instead of per 64-key tile: each workgroup first compacts the
// keys of its range that any query head of the group keeps (ordered, by prefix sums), then gathers
// only those rows.  With a top-W mask that reads W rows instead of every 64-key tile that holds one.
// The query heads of a KV group are the 32 columns of an MFMA tile (unused columns carry zeros), so
// every gathered row is used by all of them: a wave stages 32 gathered K and V rows in its own
// piece of LDS (no barrier: nobody else reads it), S^T = K Q^T and O^T += V^T P^T run on the matrix
// pipe, and the vector ALU is left with one exp2 per (key, column).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"

namespace fdma {

namespace {

constexpr int DEC_THREADS = 256;
constexpr int DEC_RANGE = 16 * DEC_THREADS;  // keys compacted per pass (16 per thread)
constexpr int DEC_NJ = 4;                    // sub-ranges per pass: the mask of 4 x 4096 keys is fetched in one go
constexpr int DEC_SUPER = DEC_NJ * DEC_RANGE;
static_assert(DEC_NJ == 4, "the list builder selects among four mask words");
constexpr int DEC_LIST = DEC_RANGE / 2;       // LISTS: keys per pass (whole column numbers in the same LDS)
constexpr int DEC_TILE = 32;                 // gathered keys per wave and step
constexpr int DEC_COLS = 32;                 // query heads per workgroup (columns of the MFMA tile)

template <int D> struct DecSmem {
    static constexpr int S = D + 8;  // row stride of a staged tile in elements (16 bytes of padding)
    static constexpr int TILE_BYTES = DEC_TILE * S * 2;
    static constexpr int WAVE_BYTES = 2 * TILE_BYTES + DEC_TILE * 4;  // K rows, V rows, fused bias
    static constexpr int OFF_IDX = 4 * WAVE_BYTES;
    static constexpr bool Q_LDS = D > 128;  // the Q fragments are kept here, see decode_kernel
    static constexpr int OFF_Q = OFF_IDX + DEC_RANGE * 2;
    static constexpr int TOTAL = OFF_Q + (Q_LDS ? D / 16 * 1024 : 0);
    static constexpr int SO = D + 4;  // row stride of a wave's partial output in floats (rows fall into different banks)
    static_assert(DEC_COLS * SO * 4 <= WAVE_BYTES, "a wave's partial output must fit its own piece");
};

// nonzero bytes of x -> bit k of the result is set iff byte k of x != 0
__device__ __forceinline__ uint32_t nz_bytes_to_bits(uint32_t x) {
    uint32_t y = (((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u;
    return ((y >> 7) * 0x10204080u) >> 28;
}

// COHERENT: the partials were written by other workgroups of the SAME launch (possibly on another XCD, behind another L2):
// they are fetched with device-scope loads.
template <bool COHERENT> __device__ __forceinline__ float part_load(const float *ptr) {
    if (COHERENT) return __uint_as_float(__hip_atomic_load((const uint32_t *)ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    return *ptr;
}

template <bool COHERENT> __device__ __forceinline__ f32x2_t part_load2(const float *ptr) {  // (8-byte aligned)
    union { uint64_t u; f32x2_t f; } x;
    if (COHERENT) x.u = __hip_atomic_load((const uint64_t *)ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else x.f = *(const f32x2_t *)ptr;
    return x.f;
}

__device__ __forceinline__ void part_store(float *ptr, float v) {
    __hip_atomic_store((uint32_t *)ptr, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// out[b,h,:] = sum_s exp(lse_s - lse) * o_s ;  lse = logsumexp_s lse_s  (empty everywhere: 0 / +inf) for one (b, h) row,
// by ONE wave: lane s (and s + 64) fetches lse_s and holds the weight of split s, then lane i sums its head-dim elements 2 i,
// 2 i + 1 (and + 128) over the splits.  Bound by trips to memory: up to CMB_FLIGHT splits are requested together, the first of
// them beside the LSEs.  Eight at a time, an element a lane, weights through LDS / now, us: 2049 keys x 32 / 8 heads, 9 splits 10.0 / 9.3; 512 kept
// of 16384 x 4 / 1, 64 splits d = 64 10.5 / 11.1 (half of the lanes have no element), 128 14.0 / 11.9, 256 25.1 / 19.3; of 65537 in 86
// 12.8 / 12.8, 18.2 / 13.7, 33.8 / 22.6.
// Both users of this function sum in the same order, so their results agree bit for bit.
constexpr int CMB_FLIGHT = 32;
constexpr int CMB_GROUP = 8;  // requested and added without a branch between them

template <typename T, bool COHERENT, bool PAIRS>
__device__ __forceinline__ void combine_row_as(const FwdParams &p, int64_t row, int lane) {
    using E = Elem<T>;
    const int64_t rows = (int64_t)p.B * p.H;
    const float lv0 = lane < p.splits ? part_load<COHERENT>(p.lse_part + (int64_t)lane * rows + row) : -INFINITY;
    const float lv1 = lane + 64 < p.splits ? part_load<COHERENT>(p.lse_part + (int64_t)(lane + 64) * rows + row) : -INFINITY;
    const int64_t step = rows * p.d;
    f32x2_t v[CMB_FLIGHT];
    auto fetch = [&](int e0, int s0) {
        const int n = p.splits - s0, e = e0 + 2 * lane;
        const float *op = p.o_part + row * p.d + (e < p.d ? e : 0) + s0 * step;
#pragma unroll
        for (int u = 0; u < CMB_FLIGHT; u += CMB_GROUP) {
            if (u < n) {  // (beyond the last split: that one again, dropped below)
#pragma unroll
                for (int q = u; q < u + CMB_GROUP; q++) {
                    const float *src = op + (q < n ? q : n - 1) * step;
                    v[q] = PAIRS ? part_load2<COHERENT>(src) : f32x2_t{part_load<COHERENT>(src), part_load<COHERENT>(src + 1)};
                }
            }
        }
    };
    fetch(0, 0);
    const float mx = wave_max(fmaxf(lv0, lv1));
    const float w0 = mx == -INFINITY ? 0.f : __expf(lv0 - mx), w1 = mx == -INFINITY ? 0.f : __expf(lv1 - mx);  // exp(-inf) = 0 for empty splits
    const float sum = wave_sum(w0 + w1);
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    if (lane == 0) p.lse[row] = mx == -INFINITY ? INFINITY : mx + __logf(sum);
    f32x2_t acc = {0.f, 0.f};
    for (int e0 = 0, s0 = 0;;) {
        const int n = p.splits - s0;
        const int w = __float_as_int(s0 < 64 ? w0 : w1);
#pragma unroll
        for (int u = 0; u < CMB_FLIGHT; u += CMB_GROUP) {  // (the splits in ascending order: sums do not depend on how they were fetched)
            if (u < n) {
#pragma unroll
                for (int q = u; q < u + CMB_GROUP; q++) {
                    const float wq = __int_as_float(__builtin_amdgcn_readlane(w, (s0 & 63) + q));
                    acc[0] = fmaf(wq, q < n ? v[q][0] : 0.f, acc[0]);
                    acc[1] = fmaf(wq, q < n ? v[q][1] : 0.f, acc[1]);
                }
            }
        }
        s0 += CMB_FLIGHT;
        if (s0 >= p.splits) {
            const int e = e0 + 2 * lane;
            if (e < p.d)  // (rows of whole 16-byte chunks)
                *(uint32_t *)((uint16_t *)p.o + (row / p.H) * p.o_b + (row % p.H) * p.o_h + e) = E::pack2(acc[0] * inv, acc[1] * inv);
            e0 += 128;
            if (e0 >= p.d) break;
            s0 = 0;
            acc = f32x2_t{0.f, 0.f};
        }
        fetch(e0, s0);
    }
}

template <typename T, bool COHERENT>
__device__ __forceinline__ void combine_row(const FwdParams &p, int64_t row, int lane) {
    // (the caller's workspace need not be aligned beyond its floats)
    if (((uintptr_t)p.o_part & 7) == 0) combine_row_as<T, COHERENT, true>(p, row, lane);
    else combine_row_as<T, COHERENT, false>(p, row, lane);
}

// LISTS: the caller has handed over the ordered list of kept keys (fdma_kept_keys: the mask builder writes it).  A
// workgroup then takes its share of the LIST instead of a range of keys and builds nothing: one trip to memory less in a
// chain of six, and every split has the same number of rows whatever the mask looks like.
// PERHEAD: mask or bias differ between the query heads of a group, so a lane fetches the mask byte and the
// bias of its own (key, head) pairs; otherwise one fused value per key serves all columns.
template <typename T, int D, bool PERHEAD, bool WIDE, bool LISTS>
__global__ void __launch_bounds__(DEC_THREADS, D <= 128 ? 2 : 1) decode_kernel(const FwdParams p, int keys_per_split) {
    using E = Elem<T>;
    using SM = DecSmem<D>;
    constexpr int CH = D / 8;         // 16-byte chunks per row
    constexpr int RPI = 64 / CH;      // rows covered by one load instruction of a wave
    constexpr int NI = DEC_TILE / RPI;
    constexpr int KS = D / 16, DB = D / 32;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ int s_wcount[DEC_NJ][4];
    __shared__ float s_m[4][DEC_COLS], s_l[4][DEC_COLS];

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, g = lane >> 5;
    const int split = blockIdx.x, b = blockIdx.z;
    const int G = p.H / p.Hk;
    const int chunks = (G + DEC_COLS - 1) / DEC_COLS;
    const int hk = blockIdx.y / chunks;
    const int g0 = (blockIdx.y % chunks) * DEC_COLS;  // first query head (within the group) of this workgroup
    const int ncol = G - g0 < DEC_COLS ? G - g0 : DEC_COLS;
    const bool col_ok = r < ncol;
    const int h = hk * G + g0 + (col_ok ? r : 0);     // this lane's query head
    const int nchunk = p.d / 8;

    using Idx = std::conditional_t<LISTS, uint32_t, uint16_t>;
    Idx *s_idx = (Idx *)(smem + SM::OFF_IDX);  // kept keys of the current pass, relative to its first key (LISTS: absolute)
    char *sK = smem + wave * SM::WAVE_BYTES;
    char *sV = sK + SM::TILE_BYTES;
    float *sB = (float *)(sV + SM::TILE_BYTES);

    int lo = split * keys_per_split, hi = lo + keys_per_split;
    if (hi > p.Lk) hi = p.Lk;
    const int32_t *list = nullptr;
    if (LISTS) {  // this workgroup's share of the list
        const int srow = (p.m_b == 0 ? 0 : b) * p.Hm + (p.Hm == 1 ? 0 : hk);
        int n = p.kept_count[srow];  // (lists are device data the host cannot check: held inside the key axis)
        n = n < 0 ? 0 : (n < p.Lk ? n : p.Lk);
        list = p.kept_idx + (int64_t)srow * p.kept_ld;
        const int per = (n + p.splits - 1) / p.splits;
        lo = split * per < n ? split * per : n;
        hi = lo + per < n ? lo + per : n;
    }

    // B operands of S^T = K Q^T: lane supplies Q[head r][16 ks + 8 g .. + 7]; columns without a head are zero
    // (d > 128: in LDS, the same for all waves and a quarter made by each; the barriers in front of a list's first batch publish
    // them.  In registers, beside the accumulators and a batch of rows in flight, they cost 6 to 40 registers spilled to scratch:
    // d = 256, us, 16384 keys x 16 / 4 heads, 4096 kept 20.8 -> 20.1, all kept 30.4 -> 29.2; 65537 x 2 / 1 all kept 48.0 -> 46.4.)
    u32x4_t qf[SM::Q_LDS ? 1 : KS];
    {
        const uint16_t *qp = (const uint16_t *)p.q + b * p.q_b + (int64_t)h * p.q_h;
        auto q_frag = [&](int ks) { return col_ok && 2 * ks + g < nchunk ? *(const u32x4_t *)(qp + 16 * ks + 8 * g) : u32x4_t{0, 0, 0, 0}; };
        if constexpr (SM::Q_LDS) {
            for (int ks = wave; ks < KS; ks += 4) *(u32x4_t *)(smem + SM::OFF_Q + (ks * 64 + lane) * 16) = q_frag(ks);
        } else {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) qf[ks] = q_frag(ks);
        }
    }
    const int hm = p.Hm == p.H ? h : (p.Hm == 1 ? 0 : hk);
    const int hb = p.Hb == p.H ? h : (p.Hb == 1 ? 0 : hk);
    const uint8_t *mrow = p.mask ? p.mask + b * p.m_b + hm * p.m_h : nullptr;
    const uint16_t *brow = p.bias ? (const uint16_t *)p.bias + b * p.bi_b + hb * p.bi_h : nullptr;

    float m = -INFINITY, l = 0.f;  // running maximum of the column (log2 domain), sum over this lane's keys
    f32x16_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.f;

    const uint16_t *kbase = (const uint16_t *)p.k + b * p.k_b + hk * p.k_h;
    const uint16_t *vbase = (const uint16_t *)p.v + b * p.v_b + hk * p.v_h;

    // fragment addresses inside a staged tile (see fdma_common.h)
    const uint32_t a_off = (uint32_t)((pi_row(r) * SM::S + g * 8) * 2);
    const TrLane tr = tr_lane(lane);
    const uint32_t tr_off = (uint32_t)(((8 * g + tr.te) * SM::S + 16 * tr.tdh + 4 * tr.tcp) * 2);
    // staging: this lane's row within a load instruction and its chunk
    const int srow = lane / CH, sc = lane % CH;
    const uint32_t st_off = (uint32_t)((srow * SM::S + sc * 8) * 2);
    const bool pad_lane = sc >= nchunk;             // head dimension below D: these lanes stage zeros
    const int scl = pad_lane ? nchunk - 1 : sc;


    // phase 1: the ordered list of the kept keys of a pass
    uint32_t bits[DEC_NJ];
    auto scan_pass = [&](int r0, int nj) {
        // the keys of [r0, r0 + DEC_SUPER): a thread tests 16 keys of each of the DEC_NJ sub-ranges (one 16-byte mask load
        // per mask row, all of them in flight together); wave scans and one barrier order the output, relative to r0
        u32x4_t mv[DEC_NJ];
        int key0[DEC_NJ];
#pragma unroll
        for (int j = 0; j < DEC_NJ; j++) {
            key0[j] = r0 + j * DEC_RANGE + 16 * tid;
            mv[j] = p.mask ? u32x4_t{0, 0, 0, 0} : u32x4_t{~0u, ~0u, ~0u, ~0u};
        }
        if (p.mask && p.Lk >= 16 && (!PERHEAD || p.Hm != p.H)) {
            // ld_row16, with nothing fetched beyond the range and, in a wave without a piece that crosses the end of the row,
            // no shifts behind the loads: what shifts in every wave cost beside aligned rows, which were all the kernel took once
            // (8 x 32 heads over 65536 keys 22.79 with them, 22.37 without and with aligned rows alone)
            const uint8_t *row = p.mask + b * p.m_b + (int64_t)(p.Hm == 1 ? 0 : hk) * p.m_h;
            bool cross = false;
#pragma unroll
            for (int j = 0; j < DEC_NJ; j++) {
                if (key0[j] < hi) mv[j] = *(const u32x4_any_t *)(row + (key0[j] + 16 <= p.Lk ? key0[j] : p.Lk - 16));
                cross = cross || (key0[j] < hi && key0[j] + 16 > p.Lk);
            }
            if (__any(cross)) {
#pragma unroll
                for (int j = 0; j < DEC_NJ; j++) mv[j] = shift_row16(mv[j], key0[j] + 16 - p.Lk);
            }
        } else if (p.mask) {  // union of the mask rows of this workgroup's columns
#pragma unroll
            for (int j = 0; j < DEC_NJ; j++) key0[j] = key0[j] < hi ? key0[j] : lo;  // (beyond the range: any piece of it, dropped below)
            for (int q = 0; q < (PERHEAD && p.Hm == p.H ? ncol : 1); q++) {
                u32x4_t x[DEC_NJ];
                const int hq = PERHEAD && p.Hm == p.H ? hk * G + g0 + q : (p.Hm == 1 ? 0 : hk);
                ld_row16(p.mask + b * p.m_b + (int64_t)hq * p.m_h, key0, p.Lk, x);
#pragma unroll
                for (int j = 0; j < DEC_NJ; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) mv[j][e] |= x[j][e];
            }
        }
#pragma unroll
        for (int j = 0; j < DEC_NJ; j++) {
            const int nval = hi - (r0 + j * DEC_RANGE + 16 * tid);  // keys of this thread inside the range
            const uint32_t inrange = nval >= 16 ? 0xffffu : (nval <= 0 ? 0u : ((1u << nval) - 1u));
            bits[j] = (nz_bytes_to_bits(mv[j][0]) | (nz_bytes_to_bits(mv[j][1]) << 4) | (nz_bytes_to_bits(mv[j][2]) << 8) |
                       (nz_bytes_to_bits(mv[j][3]) << 12)) & inrange;
        }
        // bits[j] also carries, in its upper half, the kept keys of the lower lanes of this wave in sub-range j
#pragma unroll
        for (int j = 0; j < DEC_NJ; j++) {
            if (j < nj) {
                const int cnt = __popc(bits[j]);
                int wave_total;
                const int incl = wave_scan(cnt, lane, wave_total);
                if (lane == 0) s_wcount[j][wave] = wave_total;
                bits[j] |= (uint32_t)(incl - cnt) << 16;
            }
        }
        __syncthreads();
    };

    for (int r0 = lo; r0 < hi; r0 += LISTS ? DEC_LIST : DEC_SUPER) {
        const int nj = (hi - r0 + DEC_RANGE - 1) / DEC_RANGE < DEC_NJ ? (hi - r0 + DEC_RANGE - 1) / DEC_RANGE : DEC_NJ;
        if (!LISTS) scan_pass(r0, nj);
        const int key_base = LISTS ? 0 : r0;  // what the list's entries are relative to

        // ---- phase 2 (called once the list is complete): a wave takes every fourth batch of 32 kept keys.  The
        // rows of the next batch are in flight (in registers) while the current one is worked on from LDS.
        const gptr_t kb0 = uniform_ptr(kbase + (int64_t)key_base * p.k_r), vb0 = uniform_ptr(vbase + (int64_t)key_base * p.v_r);
        const gptr_t bb0 = uniform_ptr(brow ? brow + key_base : kbase);
        auto process = [&](int total) {
            u32x4_t kreg[NI], vreg[NI];
            uint32_t braw = 0;
            bool bvalid = false;
            auto load_batch = [&](int t0) {
                // rows beyond the list repeat its last row (their scores are dropped below); lanes beyond the head
                // dimension fetch its last chunk and are cleared when the batch is staged
#pragma unroll
                for (int j = 0; j < NI; j++) {
                    const int t = t0 + j * RPI + srow;
                    const uint32_t rel = s_idx[t < total ? t : total - 1];
                    if (WIDE || LISTS) {
                        kreg[j] = *(const __attribute__((address_space(1))) u32x4_t *)(kb0 + ((int64_t)rel * p.k_r + scl * 8) * 2);
                        vreg[j] = *(const __attribute__((address_space(1))) u32x4_t *)(vb0 + ((int64_t)rel * p.v_r + scl * 8) * 2);
                    } else {
                        kreg[j] = *(const __attribute__((address_space(1))) u32x4_t *)(kb0 + (rel * (uint32_t)p.k_r + scl * 8) * 2u);
                        vreg[j] = *(const __attribute__((address_space(1))) u32x4_t *)(vb0 + (rel * (uint32_t)p.v_r + scl * 8) * 2u);
                    }
                }
                if (!PERHEAD) {  // one fused value per key: lane i < 32 fetches the bias of the batch's key i
                    bvalid = lane < DEC_TILE && t0 + lane < total;
                    braw = 0;
                    if (bvalid && brow) braw = *(const __attribute__((address_space(1))) uint16_t *)(bb0 + 2u * s_idx[t0 + lane]);
                }
            };
            int t0 = wave * DEC_TILE;
            if (t0 < total) load_batch(t0);
            while (t0 < total) {
                // stage the batch (LDS operations of one wave execute in order: the reads of the previous batch are done)
#pragma unroll
                for (int j = 0; j < NI; j++) {
                    *(u32x4_t *)(sK + st_off + j * RPI * SM::S * 2) = pad_lane ? u32x4_t{0, 0, 0, 0} : kreg[j];
                    *(u32x4_t *)(sV + st_off + j * RPI * SM::S * 2) = pad_lane ? u32x4_t{0, 0, 0, 0} : vreg[j];
                }
                if (!PERHEAD && lane < DEC_TILE) sB[lane] = bvalid ? E::lo(braw) * kLog2e : -INFINITY;
                // additive term of this lane's 16 (key, column) pairs: register 8 blk + e <-> key 16 blk + 8 g + e of the batch
                float badd[16];
                if (PERHEAD) {
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const int t = t0 + 16 * (i >> 3) + 8 * g + (i & 7);
                        badd[i] = -INFINITY;
                        if (t < total) {
                            const int key = key_base + (int)s_idx[t];
                            const bool keep = !mrow || mrow[key];
                            const float bv = brow ? E::lo((uint32_t)brow[key]) * kLog2e : 0.f;
                            badd[i] = keep ? bv : -INFINITY;
                        }
                    }
                }
                const int tn = t0 + 4 * DEC_TILE;
                if (tn < total) load_batch(tn);

                // S^T = K Q^T
                f32x16_t s;
#pragma unroll
                for (int i = 0; i < 16; i++) s[i] = 0.f;
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const u32x4_t a = *(const u32x4_t *)(sK + a_off + ks * 32);
                    s = E::mfma(a, SM::Q_LDS ? *(const u32x4_t *)(smem + SM::OFF_Q + (ks * 64 + lane) * 16) : qf[SM::Q_LDS ? 0 : ks], s);
                }
                if (!PERHEAD) {
#pragma unroll
                    for (int blk = 0; blk < 2; blk++) {
                        const f32x4_t b0 = *(const f32x4_t *)(sB + 16 * blk + 8 * g);
                        const f32x4_t b1 = *(const f32x4_t *)(sB + 16 * blk + 8 * g + 4);
#pragma unroll
                        for (int e = 0; e < 4; e++) { badd[8 * blk + e] = b0[e]; badd[8 * blk + 4 + e] = b1[e]; }
                    }
                }
                float mt = -INFINITY;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    s[i] = fmaf(s[i], p.scale_log2, badd[i]);
                    mt = fmaxf(mt, s[i]);
                }
                mt = xhalf_max(mt);
                const float mn = fmaxf(m, mt);
                const float ms = mn == -INFINITY ? 0.f : mn;
                if (__any(mn > m)) {
                    const float alpha = fast_exp2(m - ms);
                    l *= alpha;
#pragma unroll
                    for (int db = 0; db < DB; db++)
#pragma unroll
                        for (int i = 0; i < 16; i++) o[db][i] *= alpha;
                }
                m = mn;
                uint32_t pk[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float p0 = fast_exp2(s[2 * e] - ms), p1 = fast_exp2(s[2 * e + 1] - ms);
                    l += p0 + p1;
                    pk[e] = E::pack2(p0, p1);
                }
                // O^T += V^T P^T (V^T through transposing LDS reads of the row-major rows)
#pragma unroll
                for (int kb = 0; kb < 2; kb++) {
                    const u32x4_t bop = {pk[4 * kb], pk[4 * kb + 1], pk[4 * kb + 2], pk[4 * kb + 3]};
#pragma unroll
                    for (int db = 0; db < DB; db++) {
                        const uint32_t off = tr_off + (uint32_t)((16 * kb * SM::S + 32 * db) * 2);
                        const u32x2_t lo_ = lds_read_tr16(sV, off), hi_ = lds_read_tr16(sV, off + 4 * SM::S * 2);
                        const u32x4_t a = {lo_[0], lo_[1], hi_[0], hi_[1]};
                        o[db] = E::mfma(a, bop, o[db]);
                    }
                }
                t0 = tn;
            }
        };

        if (LISTS) {
            const int total = hi - r0 < DEC_LIST ? hi - r0 : DEC_LIST;
            for (int i = tid; i < total; i += DEC_THREADS) {
                const int32_t key = list[r0 + i];
                s_idx[i] = (Idx)(key < 0 ? 0 : (key < p.Lk ? key : p.Lk - 1));
            }
            __syncthreads();
            process(total);
            __syncthreads();
            continue;
        }
        // append sub-ranges to the list while they fit, work the list off, go on with the rest (dense masks only)
        for (int j = 0; j < nj;) {
            int total = 0;
            for (; j < nj; j++) {
                const int wg_cnt = s_wcount[j][0] + s_wcount[j][1] + s_wcount[j][2] + s_wcount[j][3];
                if (total + wg_cnt > DEC_RANGE) break;
                const uint32_t bj = j == 0 ? bits[0] : (j == 1 ? bits[1] : (j == 2 ? bits[2] : bits[3]));
                int pos = total + (int)(bj >> 16);
                for (int w = 0; w < wave; w++) pos += s_wcount[j][w];
                uint32_t u = bj & 0xffffu;
                while (u) {
                    const int k = __builtin_ctz(u);
                    u &= u - 1;
                    s_idx[pos++] = (Idx)(j * DEC_RANGE + 16 * tid + k);
                }
                total += wg_cnt;
            }
            __syncthreads();
            process(total);
            __syncthreads();  // the list (and, after the last round, the counts) are rebuilt next
        }
    }

    // ---- phase 3: every wave leaves its partial result in its own piece of LDS, then the four are merged
    l = xhalf_sum(l);
    if (g == 0 && col_ok) { s_m[wave][r] = m; s_l[wave][r] = l; }
    if (col_ok) {
        float *so = (float *)sK + r * SM::SO;  // [column][d]
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                const int c = 32 * db + 16 * blk + 8 * g;
                *(f32x4_t *)(so + c) = f32x4_t{o[db][8 * blk], o[db][8 * blk + 1], o[db][8 * blk + 2], o[db][8 * blk + 3]};
                *(f32x4_t *)(so + c + 4) = f32x4_t{o[db][8 * blk + 4], o[db][8 * blk + 5], o[db][8 * blk + 6], o[db][8 * blk + 7]};
            }
    }
    __syncthreads();
    for (int idx = tid; idx < ncol * D; idx += DEC_THREADS) {
        const int col = idx / D, e = idx % D;
        if (e >= p.d) continue;
        float mx = -INFINITY;
#pragma unroll
        for (int q = 0; q < 4; q++) mx = fmaxf(mx, s_m[q][col]);
        // (a wave without keys has sums of 0 and a maximum of -inf; one whose scores are all NaN has that maximum too, and its
        // sums have to reach the result)
        const float ms = mx == -INFINITY ? 0.f : mx;
        float lt = 0.f, ot = 0.f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float w = fast_exp2(s_m[q][col] - ms);
            lt += w * s_l[q][col];
            ot += w * ((const float *)(smem + q * SM::WAVE_BYTES))[col * SM::SO + e];
        }
        const int hh = hk * G + g0 + col;
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
        if (p.splits > 1) {
            // (device-scope stores: written through to where every XCD sees them, so that the merging workgroup of
            // this launch -- or the merge launch -- reads them whichever L2 it sits behind)
            const int64_t row = ((int64_t)split * p.B + b) * p.H + hh;
            part_store(p.o_part + row * p.d + e, ot * inv);
            if (e == 0) part_store(p.lse_part + row, lt > 0.f ? (mx + __builtin_amdgcn_logf(lt)) * kLn2 : -INFINITY);
        } else {
            uint16_t *op = (uint16_t *)p.o + b * p.o_b + hh * p.o_h;
            op[e] = (uint16_t)(E::pack2(ot * inv, 0.f) & 0xffffu);
            if (e == 0) p.lse[(int64_t)b * p.H + hh] = lt > 0.f ? (mx + __builtin_amdgcn_logf(lt)) * kLn2 : INFINITY;
        }
    }
    // ---- phase 4 (arrival counters given): the workgroup that finishes last among the splits of its (batch entry,
    // head chunk) merges their partial results, so the call is one launch.  The partials above are device-scope
    // stores; every wave waits until its own have been acknowledged, the barrier collects the waves, and one thread
    // then counts the workgroup in with a device-scope atomic (no cache write-back or invalidate is involved: a fence
    // would walk the whole L2 in every workgroup, which made this launch four times longer than the two it replaces).
    // The counter starts at zero, and the last arrival puts it back to zero for the next call.  Nothing waits for
    // another workgroup: one that is not last just ends.
    if (p.splits > 1 && p.dec_counter) {
        __shared__ int s_last;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            int32_t *cnt = p.dec_counter + ((int64_t)b * gridDim.y + blockIdx.y);
            const int old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int last = old == p.splits - 1;
            if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = last;
        }
        __syncthreads();
        if (s_last) {
            for (int col = wave; col < ncol; col += 4)
                combine_row<T, true>(p, (int64_t)b * p.H + hk * G + g0 + col, lane);
        }
    }
}

// The merge as a launch of its own (no arrival counters given): one wave per (b, h) row, four rows per workgroup.
constexpr int CMB_THREADS = 256;
constexpr int CMB_MAX_SPLITS = 128;  // >= the largest number of splits (decode_num_splits): a lane holds two of them

template <typename T>
__global__ void __launch_bounds__(CMB_THREADS) decode_combine_kernel(const FwdParams p) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (CMB_THREADS / 64) + wave;
    if (row < (int64_t)p.B * p.H) combine_row<T, false>(p, row, lane);
}

template <typename T, int D, bool PERHEAD, bool WIDE, bool LISTS>
hipError_t launch_decode_w(const FwdParams &p, int keys_per_split, hipStream_t stream) {
    const int G = p.H / p.Hk;
    const int chunks = (G + DEC_COLS - 1) / DEC_COLS;
    dim3 grid(p.splits, p.Hk * chunks, p.B);
    auto kern = decode_kernel<T, D, PERHEAD, WIDE, LISTS>;
    static DynSmemLimit smem_limit;
    hipError_t e = smem_limit.ensure((const void *)kern, DecSmem<D>::TOTAL);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, grid, dim3(DEC_THREADS), DecSmem<D>::TOTAL, stream, p, keys_per_split);
    return hipGetLastError();
}

template <typename T, int D, bool PERHEAD>
hipError_t launch_decode_d(const FwdParams &p, int keys_per_split, hipStream_t stream) {
    // byte offsets of a gathered row relative to the first row of a pass fit 32 bits unless the row stride is huge
    if (p.kept_idx && p.mask && p.Hm != p.H) return launch_decode_w<T, D, PERHEAD, true, true>(p, keys_per_split, stream);
    if (p.kept_idx && p.mask && p.H == p.Hk) return launch_decode_w<T, D, false, true, true>(p, keys_per_split, stream);
    const int64_t rmax = p.k_r > p.v_r ? p.k_r : p.v_r;
    const bool wide = ((int64_t)DEC_SUPER * rmax + D) * 2 >= ((int64_t)1 << 32);
    return wide ? launch_decode_w<T, D, PERHEAD, true, false>(p, keys_per_split, stream) : launch_decode_w<T, D, PERHEAD, false, false>(p, keys_per_split, stream);
}

template <typename T>
hipError_t launch_decode_t(const FwdParams &p, hipStream_t stream) {
    const int G = p.H / p.Hk;
    const int keys_per_split = ((p.Lk + p.splits - 1) / p.splits + DEC_THREADS - 1) / DEC_THREADS * DEC_THREADS;
    const bool perhead = G > 1 && ((p.mask && p.Hm == p.H) || (p.bias && p.Hb == p.H));
    hipError_t e;
    if (p.d <= 64) e = perhead ? launch_decode_d<T, 64, true>(p, keys_per_split, stream) : launch_decode_d<T, 64, false>(p, keys_per_split, stream);
    else if (p.d <= 128) e = perhead ? launch_decode_d<T, 128, true>(p, keys_per_split, stream) : launch_decode_d<T, 128, false>(p, keys_per_split, stream);
    else e = perhead ? launch_decode_d<T, 256, true>(p, keys_per_split, stream) : launch_decode_d<T, 256, false>(p, keys_per_split, stream);
    if (e != hipSuccess) return e;
    if (p.splits > 1 && !p.dec_counter) {  // (with arrival counters the decode launch has merged its splits itself)
        const int64_t rows = (int64_t)p.B * p.H;
        hipLaunchKernelGGL((decode_combine_kernel<T>), dim3((unsigned)((rows + CMB_THREADS / 64 - 1) / (CMB_THREADS / 64))), dim3(CMB_THREADS), 0, stream, p);
        e = hipGetLastError();
    }
    return e;
}

}  // namespace

// Decode route: one query token and a head dimension one lane-group can hold (16 lanes x 8).
bool use_decode_path(int Lq, int H, int Hk) {
    (void)H; (void)Hk;
    return Lq == 1;
}

// Workgroups have a fixed cost of several microseconds (mask fetch, list, arrival, merge), so few fat ones win: as many as there are CUs,
// rounded DOWN.  A few more than that and CUs work two of them off (together; at head dims above 128 one after the other): d = 256,
// 48 pairs, 1000 kept of 30000 keys, 5 splits (240) 20.5 us, 6 (288) 31.0; d = 128, 80 pairs, 2000 of 9000, 3 (240) 21.0, 4 (320) 24.0.
//   * Up to head dim 128 a CU holds two (three at 64), and where a split then still spans 8192 keys that many are taken, rounded
//     down too; also two per CU beyond 16384 keys (8192 at 64) where a CU's one would leave a fifth of them idle (88 pairs of 13235 keys,
//     all kept, d = 64: 2 splits 73.2, 3 62.0, 5 59.4), and at 64 where a CU's one is two splits: 104 to 127 pairs, 220
//     calls of 8192 to 65536 keys, by length and share kept: 2 are 0.87 to 1.04 times as fast as the number rounded up, 4 1.01 to 1.08
//     (108 pairs of 11806, all kept, 3 / 2 / 4: 67.2 / 71.8 / 64.8).
// Against the same numbers rounded up, 2400 calls of 12 to 256 pairs over 1024 to 65536 keys, 128 to all of them kept, whose number differs: 1.18
// times as fast, 26 of them more than 3 % slower and three more than 10 (192 pairs, d = 64: 12 x 26023 x 32/16, all kept 256 / 294,
// 24 x 27510 x 8/8, half 144 / 164; d = 128: 18 x 53394 x 4/4, 128 kept 10.8 / 12.4).
// Few (batch entry, kv head) pairs do not take the whole chip: every split adds some 60 ns of arrival and merge, so there are at
// most 32, or one for 1280 keys beyond 32768 keys.  Sparse masks are served best by few splits, masks that keep every key by
// many, and the host does not know which it is.  us, spans of 768 / 1024 / 1280 / 2048 keys, one pair of four heads, d = 64 | 128 | 256:
// 33001 keys, 512 kept 10.4 / 9.6 / 9.2 / 8.8 | 11.0 / 10.0 / 9.7 / 9.3 | 17.6 / 16.4 / 15.3 / 14.6; 65537, 512 kept
// 13.0 / 11.8 / 10.7 / 9.8 | 13.8 / 12.5 / 11.6 / 10.3 | 23.2 / 20.9 / 18.5 / 16.4; 4096 kept 13.3 / 11.9 / 10.8 / 10.7 | 14.0 / 12.8 /
// 11.8 / 11.8 | 23.5 / 21.2 / 19.1 / 20.2; all 33001 kept 14.9 / 16.1 / 16.8 / 21.1 | 19.0 / 20.8 / 22.4 / 29.4 | 36.7 / 42.0 / 45.8 / 61.7; all
// 65537 18.0 / 18.3 / 18.8 / 22.4 | 22.0 / 23.3 / 24.4 / 30.4 | 43.3 / 47.3 / 49.6 / 64.3.  (64 splits of 256 keys instead of
// 32 of 512: 16384 keys x 8 / 4 heads, d = 128, 512 kept 13.3 / 9.6, all kept 15.7 / 14.8.)
// A call without a mask keeps every key, and the host does know: one or two pairs then have 64 splits at least beyond 32768 keys (few query
// heads, whose partial results stay small).  By spans of 1280 / with 64, one pair of four heads, d = 64 | 128 | 256: 33001 keys 16.2 / 14.2 |
// 21.7 / 18.0 | 42.8 / 34.8; 50001 16.9 / 16.3 | 22.4 / 20.9 | 44.6 / 41.5; 65536 17.9 / 17.0 | 23.5 / 21.7 | 47.3 / 44.0; two pairs of
// four heads 33001 16.3 / 14.6 | 21.7 / 18.4 | 44.7 / 36.2, 65536 18.4 / 17.6 | 24.2 / 22.9 | 48.6 / 45.3; four pairs of two heads, 65536
// 19.1 / 20.3 | 29.1 / 30.0 | 55.2 / 55.7.
// A split has at least 256 keys; up to 384 keys there is one split, without partial results and merge: 300 keys x 8 / 2,
// d = 64, 150 kept 8.2 -> 7.1; 384, all kept, d = 128 10.5 -> 9.7 (512 keys, all kept: 10.7 in two, 11.1 in one).
// With keys_per_split rounded up to 256 every split is non-empty.
int decode_num_splits(int B, int H, int Hk, int Lk, int d, bool masked) {
    const int pairs = B * Hk > 0 ? B * Hk : 1, cus = device_cus();
    int splits = 0;
    for (int per_cu = d <= 64 ? 3 : (d <= 128 ? 2 : 1); per_cu > 1 && splits == 0; per_cu--)
        if ((int64_t)(cus * per_cu / pairs) * 8192 <= Lk) splits = cus * per_cu / pairs;
    if (splits == 0) {
        splits = cus / pairs;
        const bool idle = 16 * splits * pairs < 13 * cus || (d <= 64 && splits == 2 && 2 * pairs < cus);
        if (d <= 128 && idle && Lk >= (d <= 64 ? 8192 : 16384)) splits = 2 * cus / pairs;
        const int least = !masked && pairs <= 2 && B * H <= 64 ? 64 : 32, spans = (Lk + 1279) / 1280;
        const int most = Lk > 32768 ? (spans > least ? spans : least) : 32;
        if (splits > most) splits = most;
    }
    const int max_by_len = Lk <= 384 ? 1 : (Lk + 255) / 256;
    if (splits > max_by_len) splits = max_by_len;
    if (splits > CMB_MAX_SPLITS) splits = CMB_MAX_SPLITS;
    return decode_splits_at_most(splits, Lk);
}

// shrinks so that no split is empty after rounding keys_per_split up to a multiple of 256
int decode_splits_at_most(int splits, int Lk) {
    if (splits < 1) splits = 1;
    while (splits > 1) {
        const int kps = ((Lk + splits - 1) / splits + 255) / 256 * 256;
        if ((int64_t)(splits - 1) * kps < Lk) break;
        splits--;
    }
    return splits;
}

int64_t decode_num_counters(int B, int H, int Hk, int Lk, int d) {
    if (B <= 0 || Hk <= 0 || decode_num_splits(B, H, Hk, Lk, d, true) <= 1) return 0;  // (with a mask or without: one split of the same calls)
    const int G = H / Hk;
    return (int64_t)B * Hk * ((G + DEC_COLS - 1) / DEC_COLS);
}

hipError_t launch_fwd_decode(const FwdParams &p, int dtype, hipStream_t stream) {
    if (p.B <= 0) return hipSuccess;
    return dtype == 0 ? launch_decode_t<bf16_tag>(p, stream) : launch_decode_t<fp16_tag>(p, stream);
}

}  // namespace fdma
