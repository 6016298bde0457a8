// Shared device-side helpers for the gfx950 dynamic-mask attention kernels.
//
// Register-tile conventions used by every kernel in this directory
// (v_mfma_f32_32x32x16_{bf16,f16}, wave64, lane l, r = l % 32, g = l / 32):
//   A operand  : lane supplies A[m = r][k = 8g .. 8g+7]            (8 x 16-bit = 16 bytes)
//   B operand  : lane supplies B[k = 8g .. 8g+7][n = r]
//   C/D        : lane holds D[m = 8*(i/4) + 4g + i%4][n = r], i = 0..15
// Rows of the A tile are fetched through the permutation pi() below, so that register i of the
// accumulator corresponds to the tile row 16*(i/8) + 8g + i%8: eight consecutive rows per lane.
// That makes an accumulator directly usable as the B operand of a following MFMA whose
// contraction index is that row index (registers 8*blk..8*blk+7 <-> k = 8g..8g+7 of the
// 16-wide contraction block blk), with no cross-lane traffic.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <stdint.h>

#include "fdma_params.h"

namespace fdma {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

struct bf16_tag {};
struct fp16_tag {};

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// tile row held by MFMA row m  (see header comment)
__device__ __forceinline__ int pi_row(int m) {
    int a = m >> 3, gp = (m >> 2) & 1, c = m & 3;
    return 16 * (a >> 1) + 8 * gp + 4 * (a & 1) + c;
}

template <typename T> struct Elem;

template <> struct Elem<bf16_tag> {
    static __device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        f32x2_t f = {lo, hi};
        bf16x2_t h = __builtin_convertvector(f, bf16x2_t);
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ float lo(uint32_t u) { return __uint_as_float(u << 16); }
    static __device__ __forceinline__ float hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
    // acc + lo(pk) + hi(pk) in one instruction (v_dot2c_f32_bf16 with the constant (1, 1))
    static __device__ __forceinline__ float add_pair(uint32_t pk, float acc) {
        const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pk), ones, acc, false);
    }
    // Side-row arithmetic (see fdma_fwd_colmask.hip): an fp32 number x is handed to the MFMA as 16-bit pieces.
    // kPieceScale: the pieces of a bias value hold x * kPieceScale and meet the constant 1 / kPieceScale (keeps the
    // pieces inside the type's range).  kRefWeight: weight of the coarse piece of a reference point.  bf16 has the
    // range of fp32, so both are 1.
    static constexpr float kPieceScale = 1.f, kRefWeight = 1.f, kMaxFinite = 3.3895314e38f;
};

template <> struct Elem<fp16_tag> {
    static __device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        f32x2_t f = {lo, hi};
        f16x2_t h = __builtin_convertvector(f, f16x2_t);
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ float lo(uint32_t u) {
        f16x2_t h = __builtin_bit_cast(f16x2_t, u);
        return (float)h[0];
    }
    static __device__ __forceinline__ float hi(uint32_t u) {
        f16x2_t h = __builtin_bit_cast(f16x2_t, u);
        return (float)h[1];
    }
    static __device__ __forceinline__ float add_pair(uint32_t pk, float acc) {
        const f16x2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, pk), ones, acc, false);
    }
    // fp16 ends at 65504: bias pieces hold x / 2 (|bias * log2e| < 94507), the coarse reference piece x / 64
    static constexpr float kPieceScale = 0.5f, kRefWeight = 64.f, kMaxFinite = 65504.f;
};

// Three 16-bit pieces whose sum (in fp32) is x * kPieceScale to the last bit of x (8 or 11 significant bits each);
// a non-finite x goes into the first piece alone.  Returned as {piece0 | piece1 << 16, piece2}.
template <typename T> __device__ __forceinline__ u32x2_t split3(float x) {
    using E = Elem<T>;
    const float u = x * E::kPieceScale;
    const uint32_t w0 = E::pack2(u, 0.f);
    const float r1 = (__builtin_fabsf(u) <= 3.0e38f) ? u - E::lo(w0) : 0.f;
    const uint32_t w1 = E::pack2(r1, 0.f);
    const float r2 = r1 - E::lo(w1);
    u32x2_t out;
    out[0] = (w0 & 0xffffu) | (w1 << 16);
    out[1] = E::pack2(r2, 0.f) & 0xffffu;
    return out;
}

// Reference point of a softmax row as the MFMA sees it: minus the reference in two 16-bit pieces (a, b), worth
// kRefWeight * a + b.  Returns the packed pair (a low, b high) and, in `enc`, the number the pair really stands for.
template <typename T> __device__ __forceinline__ uint32_t encode_ref(float ref, float &enc) {
    using E = Elem<T>;
    const float lim = E::kMaxFinite;
    float a = -ref * (1.f / E::kRefWeight);
    a = fminf(fmaxf(a, -lim), lim);
    const float ra = E::lo(E::pack2(a, 0.f)) * E::kRefWeight;
    float b = -ref - ra;
    b = fminf(fmaxf(b, -lim), lim);
    const uint32_t w = E::pack2(a, b);
    enc = -(E::lo(w) * E::kRefWeight + E::hi(w));
    return w;
}

typedef __attribute__((address_space(3))) char lds_char_t;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

// Transposing LDS read (ds_read_b64_tr_b16).  Within each group of 16 lanes, lane j = 4e + c
// supplies the address of four consecutive 16-bit elements: row e, columns 4c..4c+3 of a
// 4 x 16 block; lane i of the group receives column i of that block (rows 0..3).
__device__ __forceinline__ u32x2_t lds_read_tr16(const char *smem_base, uint32_t byte_off) {
    const lds_char_t *p = (const lds_char_t *)smem_base + byte_off;
    s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)p);
    return __builtin_bit_cast(u32x2_t, v);
}

// LDS accesses by absolute byte address.  A lane keeps its part of an address (row, chunk, swizzle) in one register
// that already includes the start of the workgroup's dynamic LDS; what is added to it at compile time then lands
// in the offset field of the instruction.  (XOR-ing compile-time bits below 256 into such an address equals XOR-ing
// them into the offset alone as long as the dynamic LDS starts at a multiple of 256 bytes: declare it aligned(256).)
__device__ __forceinline__ uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)(const lds_char_t *)p; }
__device__ __forceinline__ u32x4_t lds_ld128(uint32_t addr) {
    return *(const __attribute__((address_space(3))) u32x4_t *)(uintptr_t)addr;
}
__device__ __forceinline__ u32x2_t lds_ld_tr16(uint32_t addr) {
    s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t *)(uintptr_t)addr);
    return __builtin_bit_cast(u32x2_t, v);
}
__device__ __forceinline__ uint32_t lds_ld32(uint32_t addr) { return *(const __attribute__((address_space(3))) uint32_t *)(uintptr_t)addr; }
__device__ __forceinline__ void lds_st32(uint32_t addr, uint32_t v) { *(__attribute__((address_space(3))) uint32_t *)(uintptr_t)addr = v; }

// Eight mask bits (key j in bit j, lowest first) to the eight 0 / 1 bytes of the bool mask's form.  (Bits i of a
// nibble times 0x00204081 land on positions 8 i, among others that the mask removes; no two products share a bit.)
__device__ __forceinline__ u32x2_t mask_bits_to_bytes(uint32_t b) {
    u32x2_t r;
    r[0] = ((b & 0xfu) * 0x00204081u) & 0x01010101u;
    r[1] = (((b >> 4) & 0xfu) * 0x00204081u) & 0x01010101u;
    return r;
}

// The byte with the bits of keys kk .. kk+7 (kk a multiple of 8) out of the aligned 8-byte piece of a bit row that
// holds it -- the kernels fetch bits in the same 8-byte loads as mask bytes, so that one instruction serves both forms.
__device__ __forceinline__ uint32_t mask_bits_byte(u32x2_t piece, int kk) {
    const int sh = ((kk >> 3) & 7) * 8;
    return ((sh & 32) ? piece[1] >> (sh & 31) : piece[0] >> sh) & 0xffu;
}

// A pointer that all lanes share, in scalar registers (the global address space survives the integer round trip).
typedef const __attribute__((address_space(1))) char *gptr_t;
__device__ __forceinline__ gptr_t uniform_ptr(const void *ptr) {
    const uint64_t v = (uint64_t)ptr;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (gptr_t)(((uint64_t)hi << 32) | lo);
}

// The running kernel's first argument, a struct, read where the launch left it through a pointer that the compiler cannot follow: what
// a branch of its own (another job of the same launch) loads of it is not held in scalar registers by the rest of the kernel, nor the
// other way round.
template <typename P> __device__ __forceinline__ const P &kernel_args_apart() {
    typedef const __attribute__((address_space(4))) P *args_t;
    args_t args = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return *(const P *)args;
}

// Direct loads: every lane's 16 or 4 bytes at `base` + off go to LDS, lane after lane from address `dst` on (both the same for all lanes).
// In assembly, because behind the compiler's builtin every LDS read waits for all LDS operations in flight.  So the compiler
// neither waits for them nor knows that they write LDS: a kernel waits by hand (s_waitcnt vmcnt) in front of the barrier that publishes
// them, AND, for those that are still in flight behind its last tile, in front of whatever it puts into that LDS next; no barrier does
// it.  MEMORY: other accesses stay on their side of the load.  m0 carries the address; nothing else in these kernels uses it.
template <bool MEMORY = false> __device__ __forceinline__ void load_lds16(uint32_t off, gptr_t base, uint32_t dst) {
    if constexpr (MEMORY) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(dst) : "memory");
    else asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(dst));
}
__device__ __forceinline__ void load_lds4(uint32_t off, gptr_t base, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(base), "s"(dst));
}
// ... from an address of each lane's own (16: as with MEMORY)
__device__ __forceinline__ void load_lds16_at(const void *src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(dst) : "memory");
}
__device__ __forceinline__ void load_lds4_at(gptr_t src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(src), "s"(dst));
}

// What a lane supplies to a transposing read (lds_ld_tr16): row te of four, its 8-byte piece tc of a 32-byte half row tdh.  tcp: the
// piece in the order in which the results are rows of an accumulator (see pi_row).
struct TrLane {
    int te, tc, tcp, tdh;
};
__device__ __forceinline__ TrLane tr_lane(int lane) {
    const int tj = lane & 15, tc = tj & 3;
    return {tj >> 2, tc, (tc == 1) ? 2 : (tc == 2 ? 1 : tc), (lane >> 4) & 1};
}

// Swizzle of tiles with unpadded rows: chunk c of 16 bytes lives at chunk c ^ chunk_swz(row) (see LdsTile).  Rows of 512 bytes meet the
// banks as rows of 256 do: the 16 chunks of a half row are permuted.  Two rows of 128 bytes share a line of banks: four
// consecutive ones lie in different 64-byte quarters (transposing reads), sixteen in different chunks (fragment reads).
template <int D> __device__ __forceinline__ uint32_t chunk_swz(int row) {
    return D == 64 ? (uint32_t)((((row >> 1) & 1) << 2) | ((row >> 2) & 3)) : (uint32_t)(((row & 3) << 2) | ((row >> 2) & 3));
}

// Where a lane's piece of a transposing read lies in such a tile: row 8 g + te, elements 16 tdh + 4 tcp .. + 3 of its first 32.
template <int D> __device__ __forceinline__ uint32_t tr_chunk(int g, const TrLane &t) {
    const int row = 8 * g + t.te, c = 2 * t.tdh + (t.tcp >> 1);
    // (above 64 the same as c ^ chunk_swz(row), in the form that costs the kernels fewest registers)
    const uint32_t at = D == 64 ? ((uint32_t)c ^ chunk_swz<D>(row)) << 4 : ((uint32_t)t.te << 6) | (((uint32_t)c ^ (uint32_t)(2 * g)) << 4);
    return (uint32_t)row * (2 * D) + (at | ((uint32_t)(t.tcp & 1) << 3));
}

// Row-major LDS tile of 16-bit elements ([row][head dim]) that is read two ways: as MFMA fragments (ds_read_b128:
// lane (r, g) takes the 16 bytes of chunk 2*ks + g of row pi_row(r)) and through transposing reads (lds_read_tr16:
// 16 lanes take four 8-byte pieces of each of four consecutive rows), and written row by row (16 lanes per row).
// At head dim 128 a row is exactly 256 bytes, the width of the LDS banks, and the 16-byte chunks of a row are
// permuted by a XOR with a function of the row: chunk c of row `row` lives at chunk c ^ swz(row) with
// swz(row) = 4*(row & 3) + ((row >> 2) & 3).  Four consecutive rows then sit in four different 64-byte quarters of
// the banks (what the transposing reads need: measured 145 bytes/clk per CU against 60 with rows padded to 272
// bytes) and sixteen consecutive rows in sixteen different chunks (what the fragment reads need: 230 bytes/clk, the
// same as with padding).  Other head dims keep rows padded by 8 elements.
// Offsets are bytes; a "base" is a lane constant, the *_at functions add the compile-time part.
template <int D> struct LdsTile {
    static constexpr bool SWZ = D == 128;
    static constexpr int S = SWZ ? D : D + 8;  // row stride, elements
    static constexpr int ROW_BYTES = S * 2;
    static __device__ __forceinline__ uint32_t swz(int row) { return chunk_swz<128>(row); }
    // 16-byte chunk c of a row (tile writes)
    static __device__ __forceinline__ uint32_t chunk(int row, int c) {
        return SWZ ? (uint32_t)row * 256u + ((((uint32_t)c) ^ swz(row)) << 4) : (uint32_t)((row * S + c * 8) * 2);
    }
    // fragment reads: chunk 2*ks + g of `row`; rows 32 apart share the base (add 32 * ROW_BYTES)
    static __device__ __forceinline__ uint32_t frag_base(int row, int g) {
        return SWZ ? (uint32_t)row * 256u + ((((uint32_t)g) ^ swz(row)) << 4) : (uint32_t)((row * S + g * 8) * 2);
    }
    static __device__ __forceinline__ uint32_t frag_at(uint32_t base, int ks) {
        return SWZ ? (base ^ ((uint32_t)ks << 5)) : base + (uint32_t)ks * 32u;
    }
    // transposing reads: lane (g, t) supplies row 8*g + te, elements 16*tdh + 4*tcp .. +3 of a 32-element block db, in 16-row
    // block rb; hi = 1: the same four rows further down
    static __device__ __forceinline__ uint32_t tr_base(int g, const TrLane &t) {
        return SWZ ? tr_chunk<128>(g, t) : (uint32_t)(((8 * g + t.te) * S + 16 * t.tdh + 4 * t.tcp) * 2);
    }
    static __device__ __forceinline__ uint32_t tr_at(uint32_t base, int rb, int db, int hi) {
        return SWZ ? (base ^ (((uint32_t)db << 6) | ((uint32_t)hi << 4))) + (uint32_t)(hi * 4 * 256 + rb * 16 * 256)
                   : base + (uint32_t)(((16 * rb + 4 * hi) * S + 32 * db) * 2);
    }
};

// Bytes c[u] .. c[u]+15 of a row of n bytes, zero at and beyond n; nothing outside the row is read and the row may start
// at any address (global loads of 16 bytes need no alignment on gfx950).  A piece that would cross the end of the row is
// fetched further in front and shifted, without a branch, so that all N loads are in flight together (a branch per piece
// made a trip to memory of each: decode over 65536 keys 23.1 instead of 22.5 us).
typedef u32x4_t __attribute__((aligned(1))) u32x4_any_t;
__device__ __forceinline__ u32x4_t shift_row16(const u32x4_t &v, int past) {  // `past`: bytes of the piece at or beyond the end
    uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    if (past >= 8) { lo = hi; hi = 0; }
    const int s = past > 0 ? 8 * (past & 7) : 0;
    lo = (lo >> s) | ((hi << 1) << (63 - s));
    hi >>= s;
    if (past >= 16) lo = 0;
    return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}
template <int N> __device__ __forceinline__ void ld_row16(const uint8_t *row, const int (&c)[N], int n, u32x4_t (&v)[N]) {
    if (n >= 16) {
#pragma unroll
        for (int u = 0; u < N; u++) v[u] = *(const u32x4_any_t *)(row + (c[u] + 16 <= n ? c[u] : n - 16));
        // (nothing to put back in a wave without a piece that crosses the end: thirty instructions a piece)
        bool cross = false;
#pragma unroll
        for (int u = 0; u < N; u++) cross = cross || c[u] + 16 > n;
        if (__any(cross)) {
#pragma unroll
            for (int u = 0; u < N; u++) v[u] = shift_row16(v[u], c[u] + 16 - n);
        }
    } else {
#pragma unroll
        for (int u = 0; u < N; u++) {
            v[u] = u32x4_t{0, 0, 0, 0};
            for (int e = 0; c[u] + e < n; e++) {
                const uint32_t x = (uint32_t)row[c[u] + e] << (8 * (e & 3));
                v[u][0] |= e < 4 ? x : 0u;
                v[u][1] |= e >= 4 && e < 8 ? x : 0u;
                v[u][2] |= e >= 8 && e < 12 ? x : 0u;
                v[u][3] |= e >= 12 ? x : 0u;
            }
        }
    }
}
__device__ __forceinline__ u32x4_t ld_row16(const uint8_t *row, int c, int n) {
    const int cc[1] = {c};
    u32x4_t v[1];
    ld_row16(row, cc, n, v);
    return v[0];
}

// The 8-key chunk of a mask or bias row that starts at key kk (a multiple of 8), for rows that may start at any address
// (mask: any byte, bias: any element).  chunk8_at (fdma_params.h): the key the chunk is fetched from, and chunk8_fix / chunk8_fix_mask put
// a chunk that was fetched further in front back in place (only the chunk that straddles the end of the row is; the caller
// drops keys at or beyond the end, and chunks that start there hold anything).  ODD = false: rows of whole, aligned chunks,
// nothing to put back -- a kernel of its own, because the test for it costs the memory-bound kernels 7 % at head dim 64.
typedef u32x2_t __attribute__((aligned(1))) u32x2_any_t;
typedef u32x4_t __attribute__((aligned(2))) u32x4_el_t;
template <bool ODD> __device__ __forceinline__ u32x2_t chunk8_fix_mask(u32x2_t m, int kk, int Lk) {
    if (!ODD) return m;
    const int by = kk - chunk8_at<true>(kk, Lk);
    const uint64_t v = ((uint64_t)m[0] | ((uint64_t)m[1] << 32)) >> (8 * (by < 8 ? by : 0));
    return u32x2_t{(uint32_t)v, (uint32_t)(v >> 32)};
}
template <bool ODD> __device__ __forceinline__ u32x4_t chunk8_fix(u32x4_t b, int kk, int Lk) {
    if (!ODD) return b;
    const int by = kk - chunk8_at<true>(kk, Lk);
    if (by > 0 && by < 8) {
        uint64_t lo = (uint64_t)b[0] | ((uint64_t)b[1] << 32), hi = (uint64_t)b[2] | ((uint64_t)b[3] << 32);
        if (by >= 4) { lo = hi; hi = 0; }
        const int s = 16 * (by & 3);
        lo = (lo >> s) | ((hi << 1) << (63 - s));
        hi >>= s;
        b = u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
    }
    return b;
}

// Key columns that query row `row` of Lq may see among Lk (CMP: of the kept ones, by the counts `cnt` of their row), below zero
// or zero: none.  Without a branch around the load: the two or three of a prologue and the number of kept keys are then one trip to memory.
template <bool CMP> __device__ __forceinline__ int visible_columns(int row, int Lq, int Lk, const int32_t *cnt) {
    const int c = (row < Lq ? row : Lq - 1) + Lk - Lq;
    if (!CMP) return c + 1;
    const int n = cnt[c < 0 ? 0 : (c < Lk ? c : Lk - 1)];
    return c < 0 ? 0 : n;
}

// Eight elements times `by`, rounded back to their type; all zero unless `keep` (by a mask of bits: a branch around each of a fragment's
// registers was ten instructions of them, and what is dropped may be infinite)
__device__ __forceinline__ u32x4_t kept8(u32x4_t v, bool keep) {
    uint32_t bits = keep ? ~0u : 0u;
    asm volatile("" : "+v"(bits));
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] &= bits;
    return v;
}
template <typename T> __device__ __forceinline__ u32x4_t scaled8(u32x4_t v, float by, bool keep) {
    using E = Elem<T>;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = E::pack2(E::lo(v[e]) * by, E::hi(v[e]) * by);
    return kept8(v, keep);
}

// max / sum across the two 32-lane halves of a wave (lanes l and l ^ 32)
__device__ __forceinline__ float xhalf_max(float x) {
    uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
    uint32_t u = __float_as_uint(x);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Inclusive prefix sum of x over the lanes of a wave, and the wave's total (uniform).  Four shifted adds inside
// each row of 16 lanes (data-parallel primitives: no LDS traffic), then the row totals through scalar registers.
__device__ __forceinline__ int wave_scan(int x, int lane, int &total) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1 (lanes without a source add 0)
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    const int t0 = __builtin_amdgcn_readlane(x, 15), t1 = __builtin_amdgcn_readlane(x, 31);
    const int t2 = __builtin_amdgcn_readlane(x, 47), t3 = __builtin_amdgcn_readlane(x, 63);
    const int row = lane >> 4;
    x += (row >= 1 ? t0 : 0) + (row >= 2 ? t1 : 0) + (row >= 3 ? t2 : 0);
    total = t0 + t1 + t2 + t3;
    return x;
}

// Reductions over the lanes of a wave, the result in every lane: lane i with i ^ 32, ^ 16, ^ 8, ^ 4, ^ 2, ^ 1, in this order, by lane
// swaps and data-parallel primitives.  (A shuffle is a trip through the LDS pipe, ten times the latency of one of these: 36
// of them one behind the other were 1.5 of the 8 us of a mask row.)
template <typename X, typename Op> __device__ __forceinline__ X wave_reduce(X x, Op op) {
    static_assert(sizeof(X) == 4, "32-bit values");
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    x = op(__builtin_bit_cast(X, (uint32_t)r32[0]), __builtin_bit_cast(X, (uint32_t)r32[1]));
    const uint32_t w = __builtin_bit_cast(uint32_t, x);
    const auto r16 = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    x = op(__builtin_bit_cast(X, (uint32_t)r16[0]), __builtin_bit_cast(X, (uint32_t)r16[1]));
    // (inside a row of 16 the values repeat with the distance last added: rotating is exchanging)
    auto step = [&](auto ctrl) {
        x = op(x, __builtin_bit_cast(X, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, false)));
    };
    step(std::integral_constant<int, 0x128>());  // row_ror:8
    step(std::integral_constant<int, 0x124>());  // row_ror:4
    step(std::integral_constant<int, 0x4e>());   // quad_perm:[2,3,0,1]
    step(std::integral_constant<int, 0xb1>());   // quad_perm:[1,0,3,2]
    return x;
}
template <typename X> __device__ __forceinline__ X wave_sum(X x) { return wave_reduce(x, [](X a, X b) { return a + b; }); }
__device__ __forceinline__ float wave_max(float x) { return wave_reduce(x, [](float a, float b) { return fmaxf(a, b); }); }
__device__ __forceinline__ int wave_max(int x) { return wave_reduce(x, [](int a, int b) { return a > b ? a : b; }); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

}  // namespace fdma
