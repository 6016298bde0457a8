// Keep-mask builders on the device: the reference's topk_mask / relu_mask / block_smooth
// (flash_sparse_attn/utils/mask.py:47-160) as ONE kernel per call instead of masked_fill + topk + zeros + scatter
// (+ view / sum / copy for the smoothing) through a tensor library.
//
// One workgroup owns one row of `seqlen_k` bias values (16-bit floats).  The `window` largest are found by a two-level
// radix select on an order-preserving 16-bit key: a 256-bin histogram of the high byte in LDS (several copies in different
// banks: the high byte is sign and exponent, so most of a row falls into a handful of bins), a wave-parallel suffix scan
// that finds the bin holding the window-th largest value, the same again for the low byte inside that bin.  That yields the
// exact threshold value T, the number of entries above it and how many entries EQUAL to T are still needed; those are taken
// in ascending column order (the reference's torch.topk leaves the choice among equal values unspecified).
//
// A row is a chain of dependent steps with hardly any bytes, so make_mask_kernel keeps it in registers from the one load
// to the last output: a thread holds KPT chunks of 8 columns; every wave finds the bins for itself (no broadcast, five
// barriers in all), and mask, bit row and the list of kept columns come out of one prefix sum over the workgroup.  (Passes
// over memory for each step, the list from the stored mask: 64 rows of 4093 keys 16.7 us, in registers 8.1, two columns an instruction 6.1.)  Rows of fewer than 8
// or more than 65536 keys and block smoothing take make_mask_memory_kernel, which walks the row in memory.
//
// As in the reference, entries excluded by an incoming mask are pushed to `min_value` before the selection, and a
// selected entry whose value equals `min_value` is not kept; the optional block smoothing then replaces every
// aligned block of `block_size` keys by the majority vote of its entries (a shorter tail block votes over its own
// length; exactly half is dropped).
#include <type_traits>

#include "fdma_common.h"
#include "fdma_params.h"
#include "fdma_scan.h"

namespace fdma {
namespace {


// 16-bit float bits (bf16 or fp16: sign, exponent, mantissa) -> key whose unsigned order is the numeric order
__device__ __forceinline__ uint32_t order_key(uint32_t bits) { return (bits & 0x8000u) ? (~bits & 0xffffu) : (bits | 0x8000u); }

// hist[256] (LDS), k >= 1, sum(hist) >= k.  Wave 0 finds the bin b with count(bins > b) < k <= count(bins >= b) and
// writes {b, count(bins > b)} to res[0..1].  Lane l owns bins 255-4l .. 252-4l.
__device__ __forceinline__ void find_bin(const uint32_t *hist, uint32_t k, uint32_t *res) {
    const int lane = threadIdx.x & 63;
    uint32_t c[4], s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        c[j] = hist[255 - 4 * lane - j];
        s += c[j];
    }
    int total;
    const uint32_t incl = (uint32_t)wave_scan((int)s, lane, total);
    uint32_t a = incl - s;
    if (a < k && k <= incl) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (a < k && k <= a + c[j]) {
                res[0] = 255 - 4 * lane - j;
                res[1] = a;
            }
            a += c[j];
        }
    }
}

// The same by every wave for itself, the answer in scalar registers.  h: 256 bins.
__device__ __forceinline__ void find_bin_wave(const uint32_t *h, uint32_t k, uint32_t &bin, uint32_t &above) {
    const int lane = threadIdx.x & 63;
    uint32_t c[4], s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        c[j] = h[255 - 4 * lane - j];
        s += c[j];
    }
    int total;
    const uint32_t incl = (uint32_t)wave_scan((int)s, lane, total);
    uint32_t a = incl - s, mine_bin = 0, mine_above = 0;
    const uint64_t who = __ballot(a < k && k <= incl);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (a < k && k <= a + c[j]) {
            mine_bin = 255 - 4 * lane - j;
            mine_above = a;
        }
        a += c[j];
    }
    const int l = who ? __builtin_ctzll(who) : 0;
    bin = __builtin_amdgcn_readlane(mine_bin, l);
    above = __builtin_amdgcn_readlane(mine_above, l);
}

// ---- pairs of 16-bit values in one register
typedef __attribute__((ext_vector_type(2))) uint16_t u16x2_t;
typedef __attribute__((ext_vector_type(2))) int16_t s16x2_t;
__device__ __forceinline__ uint32_t order_keys(uint32_t x) {  // order_key of both
    const uint32_t sign = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2_t, x) >> (s16x2_t){15, 15});
    return x ^ (sign | 0x80008000u);
}
// one where a half of x is not zero
__device__ __forceinline__ uint32_t not_zero2(uint32_t x) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, x), (u16x2_t){1, 1}));
}
// one where a half of x is above that of t
__device__ __forceinline__ uint32_t above2(uint32_t x, uint32_t t) {
    return not_zero2(__builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2_t, x), __builtin_bit_cast(u16x2_t, t))));
}
// the ones of four pairs (columns 2 e, 2 e + 1 of a chunk), gathered as acc |= ones << 2 e, as a bit per column
__device__ __forceinline__ uint32_t column_bits(uint32_t acc) { return (acc & 0x55u) | ((acc >> 15) & 0xaau); }

// One row in registers: NT threads, chunk c of thread t = columns (c * NT + t) * 8 .. + 7.  Lk >= 8, Lk <= NT * 8 * KPT.
//
// Bound by the vector instructions of the one CU that has the row (its load and its barriers are 3 us).  The columns are kept as ordered
// keys, two to a register, and what is compared, filled and counted is two columns an instruction: some 25 instructions a column,
// where one at a time, the key made again in each pass, was 60.  Kept and tied columns share a prefix sum, and the list leaves through LDS.
// Before / now, us (2.5 of them the launch): 64 rows of 4093, 1024 kept 7.2 / 6.1; 4 of 8000, 1024 8.3 / 6.9; 8 of 15738, 1524 12.0 / 9.6; 2 of 26876,
// 3072 17.6 / 13.2, all of them 27.2 / 12.8; 2 of 60000, 4096 37.4 / 21.4; 8192 rows of 4096 (bit rows) 56.1 / 35.9.
template <int NT, int KPT>
__global__ void __launch_bounds__(NT) make_mask_kernel(const MaskParams p) {
    constexpr int NW = NT / 64, LOG1 = NT >= 512 ? 4 : 3, REP1 = 1 << LOG1, LOG2 = 2, REP2 = 1 << LOG2;
    __shared__ __attribute__((aligned(16))) uint32_t hist1[256 * REP1], hist2[256 * REP2], hsum[2][256];
    __shared__ uint32_t s_tot[KPT * NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = blockIdx.x;
    const int r = row % p.rows, h = (row / p.rows) % p.heads, b = row / (p.rows * p.heads);
    const uint16_t *brow = (const uint16_t *)p.bias + b * p.bi_b + h * p.bi_h + (int64_t)r * p.bi_r;
    const uint8_t *mrow = p.mask_in ? p.mask_in + b * p.mi_b + h * p.mi_h + (int64_t)r * p.mi_r : nullptr;
    uint8_t *orow = p.mask_out + b * p.mo_b + h * p.mo_h + (int64_t)r * p.mo_r;
    const int Lk = p.Lk;
    const uint32_t min_key = order_key(p.min_bits);
    const bool min_zero = (p.min_bits & 0x7fffu) == 0;  // ("is the fill value" compares numerically: +0 == -0)
    auto first_col = [&](int c) -> int { return (c * NT + tid) * 8; };
    auto valid = [&](int c) -> int {  // columns of the chunk inside the row
        const int n = Lk - first_col(c);
        return n >= 8 ? 8 : (n < 0 ? 0 : n);
    };
    // ---- the row, after the masked fill, as ordered keys.  Columns beyond its end: the lowest key, which moves no threshold (there are
    // at least k columns inside); their bits are dropped at the end
    uint32_t v[KPT][4];
    {
        u32x4_t raw[KPT];
        u32x2_t mm[KPT];
#pragma unroll
        for (int c = 0; c < KPT; c++) {
            raw[c] = *(const u32x4_el_t *)(brow + chunk8_at<true>(first_col(c), Lk));
            if (mrow) mm[c] = *(const u32x2_any_t *)(mrow + chunk8_at<true>(first_col(c), Lk));
        }
        for (int i = tid; i < 64 * REP1; i += NT) ((u32x4_t *)hist1)[i] = u32x4_t{0, 0, 0, 0};
        for (int i = tid; i < 64 * REP2; i += NT) ((u32x4_t *)hist2)[i] = u32x4_t{0, 0, 0, 0};
        const uint32_t fill = min_key | (min_key << 16);
#pragma unroll
        for (int c = 0; c < KPT; c++) {
            const u32x4_t x = chunk8_fix<true>(raw[c], first_col(c), Lk);
#pragma unroll
            for (int e = 0; e < 4; e++) v[c][e] = order_keys(x[e]);
            if (mrow) {
                const u32x2_t m = chunk8_fix_mask<true>(mm[c], first_col(c), Lk);
#pragma unroll
                for (int hlf = 0; hlf < 2; hlf++) {
                    uint32_t o = m[hlf];
                    o = ((((o & 0x7f7f7f7fu) + 0x7f7f7f7fu) | o) >> 7) & 0x01010101u;  // nonzero byte -> 0x01
                    const uint32_t z = (o << 8) - o;                                     // 0x01 -> 0xFF per byte
                    const uint32_t k0 = __builtin_amdgcn_perm(0, z, 0x01010000u), k1 = __builtin_amdgcn_perm(0, z, 0x03030202u);
                    v[c][2 * hlf] = (v[c][2 * hlf] & k0) | (fill & ~k0);
                    v[c][2 * hlf + 1] = (v[c][2 * hlf + 1] & k1) | (fill & ~k1);
                }
            }
            const int n = valid(c);
            if (n < 8) {
#pragma unroll
                for (int e = 0; e < 4; e++) v[c][e] &= (n > 2 * e ? 0xffffu : 0u) | (n > 2 * e + 1 ? 0xffff0000u : 0u);
            }
        }
    }
    // exclusive prefix, in column order, of a count per chunk -- or of two, in the halves of a register --: inside the wave (which leaves its
    // totals), and -- behind a barrier -- of the totals, which every wave sums for itself, two per lane; returns the row's
    auto prefix = [&](const uint32_t (&n)[KPT], uint32_t (&before)[KPT]) -> uint32_t {
        constexpr int N = KPT * NW;
        static_assert(N <= 128, "two totals per lane");
#pragma unroll
        for (int c = 0; c < KPT; c++) {
            int total;
            before[c] = (uint32_t)wave_scan((int)n[c], lane, total) - n[c];
            if (lane == 0) s_tot[c * NW + wave] = (uint32_t)total;
        }
        __syncthreads();
        const int t0 = 2 * lane < N ? (int)s_tot[2 * lane] : 0, t1 = 2 * lane + 1 < N ? (int)s_tot[2 * lane + 1] : 0;
        int total;
        const int e1 = wave_scan(t0 + t1, lane, total) - t1, e0 = e1 - t0;
#pragma unroll
        for (int c = 0; c < KPT; c++) {
            const int i = c * NW + __builtin_amdgcn_readfirstlane(wave);
            before[c] += (uint32_t)__builtin_amdgcn_readlane((i & 1) ? e1 : e0, i >> 1);
        }
        return (uint32_t)total;
    };
    // bits of the columns of a chunk whose key is above t (both halves the same)
    auto above = [&](int c, uint32_t t) -> uint32_t {
        uint32_t acc = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) acc |= above2(v[c][e], t) << (2 * e);
        return column_bits(acc);
    };
    auto twice = [](uint32_t x) -> uint32_t { return x | (x << 16); };
    // ... whose key is x
    auto equal = [&](int c, uint32_t x) -> uint32_t {
        uint32_t acc = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) acc |= not_zero2(v[c][e] ^ twice(x)) << (2 * e);
        return column_bits(acc) ^ 0xffu;
    };

    // one bit per column of the chunk: kept whatever else there is; equal to the threshold, of which `need` are kept
    uint32_t keep[KPT], ties[KPT];
    uint32_t need = 0;
    bool some_ties = false;
#pragma unroll
    for (int c = 0; c < KPT; c++) keep[c] = ties[c] = 0;
    if (p.type == 1) {  // relu: keep strictly positive values (NaN is not > 0)
        const uint32_t inf = p.dtype == 0 ? 0x7f80u : 0x7c00u;
#pragma unroll
        for (int c = 0; c < KPT; c++) keep[c] = above(c, twice(0x8000u)) & ~above(c, twice(0x8000u | inf));
    } else if (p.window > 0) {
        const uint32_t k = (uint32_t)(p.window < Lk ? p.window : Lk);
        // sums of the copies of every bin: four copies a thread, a bin's threads side by side
        auto fold = [&](const uint32_t *hist, auto log_c, uint32_t *sum) {
            constexpr int PER = 1 << (decltype(log_c)::value - 2);  // threads of a bin: 1, 2 or 4
#pragma unroll
            for (int t = tid; t < 256 * PER; t += NT) {
                const u32x4_t q = ((const u32x4_t *)hist)[t];
                int s = (int)(q[0] + q[1] + q[2] + q[3]);
                if (PER >= 2) s += __builtin_amdgcn_update_dpp(0, s, 0xb1, 0xf, 0xf, false);  // quad_perm:[1,0,3,2]
                if (PER >= 4) s += __builtin_amdgcn_update_dpp(0, s, 0x4e, 0xf, 0xf, false);  // quad_perm:[2,3,0,1]
                if (t % PER == 0) sum[t / PER] = (uint32_t)s;
            }
            __syncthreads();
        };
        __syncthreads();
        const uint32_t copy1 = (uint32_t)(lane & (REP1 - 1)) * 4, copy2 = (uint32_t)(lane & (REP2 - 1)) * 4;
        auto count = [](uint32_t *hist, uint32_t at) { atomicAdd((uint32_t *)((char *)hist + at), 1u); };
#pragma unroll
        for (int c = 0; c < KPT; c++)
            if (first_col(c) < Lk) {
#pragma unroll
                for (int e = 0; e < 4; e++) {  // (byte offset of a copy of a bin: high byte of the key x 4 REP1)
                    count(hist1, ((v[c][e] >> (6 - LOG1)) & (0xffu << (LOG1 + 2))) | copy1);
                    count(hist1, ((v[c][e] >> (22 - LOG1)) & (0xffu << (LOG1 + 2))) | copy1);
                }
            }
        __syncthreads();
        fold(hist1, std::integral_constant<int, LOG1>(), hsum[0]);
        uint32_t bin1, above1, bin2, above_2;
        find_bin_wave(hsum[0], k, bin1, above1);
        const uint32_t high = twice(bin1 << 8);
#pragma unroll
        for (int c = 0; c < KPT; c++)
            if (first_col(c) < Lk) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t x = v[c][e] ^ high, lo = x & 0xffffu, hi = x >> 16;  // (below 256: in this bin, and where in it)
                    if (lo < 256) count(hist2, (lo << (LOG2 + 2)) | copy2);
                    if (hi < 256) count(hist2, (hi << (LOG2 + 2)) | copy2);
                }
            }
        __syncthreads();
        fold(hist2, std::integral_constant<int, LOG2>(), hsum[1]);
        find_bin_wave(hsum[1], k - above1, bin2, above_2);
        const uint32_t T = (bin1 << 8) | bin2;
        auto is_min_key = [&](uint32_t x) -> bool { return x == min_key || (min_zero && (x == 0x8000u || x == 0x7fffu)); };
        // entries equal to T still to take, >= 1 of hsum[1][bin2]: in column order (none where T is the fill value)
        need = is_min_key(T) ? 0u : k - above1 - above_2;
        some_ties = need != 0 && need < hsum[1][bin2];
#pragma unroll
        for (int c = 0; c < KPT; c++) keep[c] = above(c, twice(T));
        if (need != 0) {
#pragma unroll
            for (int c = 0; c < KPT; c++) ties[c] = equal(c, T);
        }
        if (T < (min_zero ? 0x8000u : min_key)) {  // (the fill value may lie above the threshold)
#pragma unroll
            for (int c = 0; c < KPT; c++) keep[c] &= ~(equal(c, min_key) | (min_zero ? equal(c, 0x8000u) | equal(c, 0x7fffu) : 0u));
        }
    }
#pragma unroll
    for (int c = 0; c < KPT; c++) {
        const uint32_t inside = (1u << valid(c)) - 1u;
        keep[c] &= inside;
        ties[c] &= inside;
    }
    // ---- columns kept in front of each chunk, and the first `need` of the ties.  Where only some ties are kept, both are counted in the halves of a
    // register: the others are below 65536, and so is what lies in front of any chunk; the row's ties may be 65536, whose half of the total wraps to
    // zero and is not looked at
    uint32_t run[KPT], total = 0;
    if (!some_ties) {
#pragma unroll
        for (int c = 0; c < KPT; c++) { keep[c] |= ties[c]; ties[c] = 0; }
    }
    if (some_ties || p.kept_idx) {
        uint32_t n[KPT];
#pragma unroll
        for (int c = 0; c < KPT; c++) n[c] = (uint32_t)__builtin_popcount(keep[c]) | ((uint32_t)__builtin_popcount(ties[c]) << 16);
        total = prefix(n, run);
        if (some_ties) {
            total = (total & 0xffffu) + need;  // (there are more ties than that)
#pragma unroll
            for (int c = 0; c < KPT; c++) {
                const int tied = (int)(run[c] >> 16);
                int left = (int)need - tied;
                run[c] = (run[c] & 0xffffu) + (uint32_t)(left > 0 ? tied : (int)need);
                if (left >= __builtin_popcount(ties[c])) {
                    keep[c] |= ties[c];
                } else {  // (the last ones kept lie in one chunk)
                    for (uint32_t u = ties[c]; left > 0; left--, u &= u - 1) keep[c] |= u & (0u - u);
                }
            }
        }
    }

    // ---- the mask row, and its bits (key j of a row in bit j % 8 of byte j / 8)
#pragma unroll
    for (int c = 0; c < KPT; c++) {
        const int col = first_col(c), n = valid(c);
        const u32x2_t bytes = mask_bits_to_bytes(keep[c]);
        if (n == 8) {
            *(u32x2_any_t *)(orow + col) = bytes;
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < n) orow[col + j] = (uint8_t)((keep[c] >> j) & 1u);
        }
        if (p.bits && n > 0) p.bits[(size_t)row * p.bits_row_bytes + (col >> 3)] = (uint8_t)keep[c];
    }
    // ---- the row as an ordered list of kept columns with inclusive prefix counts (fdma_scan.h), written up to
    // round_up(Lk, 16): the row has room
    if (p.kept_idx) {
        // (a wave's columns of a chunk go through LDS, 512 at most, and leave 64 at a time: a store for each of a lane's eight touched
        // every line of the list eight times)
        int32_t *irow = p.kept_idx + (size_t)row * p.kept_ld, *crow = p.kept_cnt + (size_t)row * p.kept_ld;
        static_assert(256 * REP1 * 4 >= NW * 1024, "the lists of a chunk take the place of the first histogram");
        uint16_t *list = (uint16_t *)hist1 + wave * 512;
#pragma unroll
        for (int c = 0; c < KPT; c++) {
            const int col = first_col(c);
            const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)run[c], 0);
            const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)run[c] + __builtin_popcount(keep[c]), 63) - first;
            uint32_t at = run[c], cv[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t one = (keep[c] >> j) & 1u;
                if (one) list[at - first] = (uint16_t)(col + j);
                cv[j] = at += one;
            }
            __builtin_amdgcn_wave_barrier();
            for (uint32_t i = lane; i < n; i += 64) irow[first + i] = list[i];
            __builtin_amdgcn_wave_barrier();
            if (col < (Lk + 15) / 16 * 16) {
                *(u32x4_t *)(crow + col) = u32x4_t{cv[0], cv[1], cv[2], cv[3]};
                *(u32x4_t *)(crow + col + 4) = u32x4_t{cv[4], cv[5], cv[6], cv[7]};
            }
        }
        if (tid == 0) p.kept_count[row] = (int32_t)total;
    }
}

// The row in memory.  NT threads own one row.  A thread handles 8 consecutive columns at a time (one 16-byte load of bias, one 8-byte
// load of the incoming mask, one 8-byte store of the result when the row addresses allow it).
// REP copies of the histogram, copy = lane % REP, laid out [bin][copy] so that the copies of a bin sit in different
// LDS banks: lanes that hit the same bin do not serialise (32 copies for long rows; 8 for short ones, where clearing
// and folding the copies would cost more than the conflicts).
template <int NT, int REP>
__global__ void __launch_bounds__(NT) make_mask_memory_kernel(const MaskParams p) {
    __shared__ uint32_t hist[256 * REP];  // [bin][copy]
    __shared__ uint32_t hsum[256];
    __shared__ uint32_t res[4];
    __shared__ uint32_t wave_cnt[NT / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = blockIdx.x;
    const int r = row % p.rows, h = (row / p.rows) % p.heads, b = row / (p.rows * p.heads);
    const uint16_t *brow = (const uint16_t *)p.bias + b * p.bi_b + h * p.bi_h + (int64_t)r * p.bi_r;
    const uint8_t *mrow = p.mask_in ? p.mask_in + b * p.mi_b + h * p.mi_h + (int64_t)r * p.mi_r : nullptr;
    uint8_t *orow = p.mask_out + b * p.mo_b + h * p.mo_h + (int64_t)r * p.mo_r;
    const int Lk = p.Lk;
    const uint32_t min_bits = p.min_bits;
    const bool vec_b = ((uintptr_t)brow & 15) == 0, vec_m = ((uintptr_t)mrow & 7) == 0, vec_o = ((uintptr_t)orow & 7) == 0;

    // values of columns idx .. idx+7 after the masked fill, as bits of the bias type; returns how many are in range
    auto load8 = [&](int idx, uint32_t (&v)[8]) -> int {
        const int n = Lk - idx < 8 ? Lk - idx : 8;
        if (vec_b && n == 8) {
            const u32x4_t t = *(const u32x4_t *)(brow + idx);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[2 * j] = t[j] & 0xffffu;
                v[2 * j + 1] = t[j] >> 16;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = j < n ? brow[idx + j] : 0;
        }
        if (mrow) {
            if (vec_m && n == 8) {
                const uint64_t mm = *(const uint64_t *)(mrow + idx);
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (!((mm >> (8 * j)) & 0xffu)) v[j] = min_bits;
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (j < n && !mrow[idx + j]) v[j] = min_bits;
            }
        }
        return n;
    };
    auto store8 = [&](int idx, int n, uint64_t bytes) {
        if (vec_o && n == 8) {
            *(uint64_t *)(orow + idx) = bytes;
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < n) orow[idx + j] = (uint8_t)((bytes >> (8 * j)) & 0xffu);
        }
    };
    // "is the fill value" compares numerically (+0 == -0)
    auto is_min = [&](uint32_t v) -> bool { return v == min_bits || (((v | min_bits) & 0x7fffu) == 0); };
    auto clear_hist = [&]() {
        for (int i = tid; i < 256 * REP; i += NT) hist[i] = 0;
    };
    // sum of the copies of every bin -> hsum; copy (t + i) % REP in step i keeps the lanes on different banks
    auto fold_hist = [&]() {
        for (int t = tid; t < 256; t += NT) {
            uint32_t s = 0;
#pragma unroll
            for (int i = 0; i < REP; i++) s += hist[t * REP + ((t + i) & (REP - 1))];
            hsum[t] = s;
        }
    };

    if (p.type == 1) {  // relu: keep strictly positive values (NaN is not > 0)
        const uint32_t inf = p.dtype == 0 ? 0x7f80u : 0x7c00u;
        for (int idx = tid * 8; idx < Lk; idx += NT * 8) {
            uint32_t v[8];
            const int n = load8(idx, v);
            uint64_t bytes = 0;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t mag = v[j] & 0x7fffu;
                if (!(v[j] & 0x8000u) && mag != 0 && mag <= inf) bytes |= 1ull << (8 * j);
            }
            store8(idx, n, bytes);
        }
    } else {
        const uint32_t k = (uint32_t)(p.window < Lk ? p.window : Lk);
        if (k == 0) {
            for (int idx = tid * 8; idx < Lk; idx += NT * 8) store8(idx, Lk - idx < 8 ? Lk - idx : 8, 0);
        } else {
            const int rep = lane & (REP - 1);
            // ---- level 1: high byte
            clear_hist();
            __syncthreads();
            for (int idx = tid * 8; idx < Lk; idx += NT * 8) {
                uint32_t v[8];
                const int n = load8(idx, v);
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (j < n) atomicAdd(&hist[(order_key(v[j]) >> 8) * REP + rep], 1u);
            }
            __syncthreads();
            fold_hist();
            __syncthreads();
            if (wave == 0) find_bin(hsum, k, res);
            clear_hist();
            __syncthreads();
            const uint32_t bin1 = res[0], above1 = res[1];
            // ---- level 2: low byte inside bin1
            for (int idx = tid * 8; idx < Lk; idx += NT * 8) {
                uint32_t v[8];
                const int n = load8(idx, v);
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const uint32_t key = order_key(v[j]);
                    if (j < n && (key >> 8) == bin1) atomicAdd(&hist[(key & 0xffu) * REP + rep], 1u);
                }
            }
            __syncthreads();
            fold_hist();
            __syncthreads();
            if (wave == 0) find_bin(hsum, k - above1, res + 2);
            __syncthreads();
            const uint32_t T = (bin1 << 8) | res[2];
            const uint32_t need_eq = k - above1 - res[3];  // >= 1 entries equal to T still to take
            const uint32_t total_eq = hsum[res[2]];
            if (need_eq >= total_eq) {  // every entry equal to the threshold is taken: no ordering needed
                for (int idx = tid * 8; idx < Lk; idx += NT * 8) {
                    uint32_t v[8];
                    const int n = load8(idx, v);
                    uint64_t bytes = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        if (order_key(v[j]) >= T && !is_min(v[j])) bytes |= 1ull << (8 * j);
                    store8(idx, n, bytes);
                }
            } else {
                // Ties across the threshold: the first need_eq of them in column order.  Columns are walked in
                // chunks of NT * 8 in order: a prefix over the lanes' counts inside the wave, per-wave counts through LDS.
                uint32_t taken = 0;  // entries equal to T seen in earlier chunks (uniform)
                for (int base = 0; base < Lk; base += NT * 8) {
                    const int idx = base + tid * 8;
                    uint32_t v[8];
                    const int n = idx < Lk ? load8(idx, v) : 0;
                    uint32_t mine = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        if (j < n && order_key(v[j]) == T) mine++;
                    int wave_total;
                    const uint32_t incl = (uint32_t)wave_scan((int)mine, lane, wave_total);
                    if (lane == 0) wave_cnt[wave] = (uint32_t)wave_total;
                    __syncthreads();
                    uint32_t rank = taken + incl - mine, chunk_total = 0;
                    for (int w = 0; w < NT / 64; w++) {
                        if (w < wave) rank += wave_cnt[w];
                        chunk_total += wave_cnt[w];
                    }
                    uint64_t bytes = 0;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const uint32_t key = order_key(v[j]);
                        const bool eq = j < n && key == T;
                        if (j < n && (key > T || (eq && rank < need_eq)) && !is_min(v[j])) bytes |= 1ull << (8 * j);
                        if (eq) rank++;
                    }
                    if (n > 0) store8(idx, n, bytes);
                    taken += chunk_total;
                    __syncthreads();
                }
            }
        }
    }

    // ---- block smoothing (majority vote), on the row this workgroup has just written
    const int bs = p.block_size;
    if (bs > 1) {
        __syncthreads();  // the row's stores are visible to the whole workgroup
        const int n_full = Lk / bs, tail = Lk - n_full * bs;
        const int n_blocks = n_full + (tail ? 1 : 0);
        for (int blk = tid; blk < n_blocks; blk += NT) {
            const int c0 = blk * bs, len = blk < n_full ? bs : tail;
            int votes = 0;
            for (int c = 0; c < len; c++) votes += orow[c0 + c];
            const uint8_t keep = (2 * votes > len) ? 1 : 0;
            for (int c = 0; c < len; c++) orow[c0 + c] = keep;
        }
    }

    // ---- optional second output: the row as an ordered list of kept columns with prefix counts, the form the
    // compaction path of the attention kernels works on (they then need no pass of their own over the mask)
    if (p.kept_idx) {
        __syncthreads();  // the row's stores are visible to the whole workgroup
        scan_mask_row<NT>(orow, Lk, p.kept_idx + (size_t)row * p.kept_ld, p.kept_cnt + (size_t)row * p.kept_ld,
                          p.kept_count + row, (int *)wave_cnt);
    }

    // ---- optional third output: the row packed to one bit per key (key j in bit j % 8 of byte j / 8), the form in
    // which the per-query attention kernels take a mask at an eighth of its traffic.  A thread packs 32 keys into
    // one word; the row it reads was written by this workgroup a moment ago.
    if (p.bits) {
        __syncthreads();  // the row's stores are visible to the whole workgroup
        uint8_t *bits_row = p.bits + (size_t)row * p.bits_row_bytes;
        const int n_bytes = (Lk + 7) / 8;
        for (int w = tid; w * 4 < n_bytes; w += NT) {
            uint32_t word = 0;
            const int c0 = w * 32;
            if (vec_o && c0 + 32 <= Lk) {
#pragma unroll
                for (int q8 = 0; q8 < 4; q8++) {
                    const uint64_t m8 = *(const uint64_t *)(orow + c0 + 8 * q8);  // eight 0 / 1 bytes
                    // (bit 8 i of m8 to bit i: the product gathers them in its top byte)
                    word |= (uint32_t)(((m8 & 0x0101010101010101ull) * 0x0102040810204080ull) >> 56) << (8 * q8);
                }
            } else {
                for (int c = 0; c < 32 && c0 + c < Lk; c++) word |= (orow[c0 + c] ? 1u : 0u) << c;
            }
            if (w * 4 + 4 <= n_bytes) {
                *(uint32_t *)(bits_row + w * 4) = word;  // (rows are 4-byte aligned: bits_row_bytes is a multiple of 4)
            } else {
                for (int k = 0; w * 4 + k < n_bytes; k++) bits_row[w * 4 + k] = (uint8_t)(word >> (8 * k));
            }
        }
    }
}

}  // namespace

hipError_t launch_make_mask(const MaskParams &p, hipStream_t stream) {
    const int64_t n_rows = (int64_t)p.batch * p.heads * p.rows;
    if (n_rows <= 0 || p.Lk <= 0) return hipSuccess;
    if (p.Lk >= 8 && p.Lk <= 65536 && p.block_size <= 1) {
        // few rows: enough threads for one chunk of 8 columns each, up to 16 waves per row (the row is a latency chain);
        // many rows: 4 waves per row and several rows per CU, each thread with more of the row
        auto go = [&](auto kern, int nt) {
            hipLaunchKernelGGL(kern, dim3((unsigned)n_rows), dim3(nt), 0, stream, p);
            return hipGetLastError();
        };
        const bool many = n_rows >= 1024;
        if (p.Lk <= 2048) return go(make_mask_kernel<256, 1>, 256);
        if (many && p.Lk <= 4096) return go(make_mask_kernel<256, 2>, 256);
        if (many && p.Lk <= 8192) return go(make_mask_kernel<256, 4>, 256);
        if (p.Lk <= 4096) return go(make_mask_kernel<512, 1>, 512);
        if (p.Lk <= 8192) return go(make_mask_kernel<1024, 1>, 1024);
        if (p.Lk <= 16384) return go(make_mask_kernel<1024, 2>, 1024);
        if (p.Lk <= 32768) return go(make_mask_kernel<1024, 4>, 1024);
        return go(make_mask_kernel<1024, 8>, 1024);
    }
    // few long rows: 16 waves per row; many rows: 4 waves per row and several rows per CU
    if (p.Lk >= 8192 && n_rows < 2048) hipLaunchKernelGGL((make_mask_memory_kernel<1024, 32>), dim3((unsigned)n_rows), dim3(1024), 0, stream, p);
    else if (p.Lk >= 16384) hipLaunchKernelGGL((make_mask_memory_kernel<256, 32>), dim3((unsigned)n_rows), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((make_mask_memory_kernel<256, 8>), dim3((unsigned)n_rows), dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace fdma
