// Host-side check of the mapping from workgroups to blocks of query rows (row_grid / row_unit in flash-dmattn_amd/csrc/fdma_params.h, built and
// run by tests/test_row_units.py with g++), over random batches of one length and ragged ones: every block of rows that a
// call computes has exactly one workgroup per query head, no other workgroup names one, a launch is made of whole turns over the 8 XCDs,
// and rounding the blocks of the longest entry up to its lists no more than doubles it.  And of the places of rows in pieces of 16 (row_piece),
// where a matrix has more bytes than 32 bits count, of the steps of an entry (kv_head_steps) for lengths below zero, and
// of what is fetched for 8-key chunks of mask rows (mask_piece_at).
#include <cstdio>
#include <cstring>
#include <vector>

#include "fdma_params.h"

using namespace fdma;

int main() {
    unsigned rng = 1u;
    auto next = [&]() { rng = rng * 1664525u + 1013904223u; return (int)(rng >> 8); };
    long long checked = 0, whole = 0;
    for (int rep = 0; rep < 12000; rep++) {
        FwdParams p;
        std::memset(&p, 0, sizeof(p));
        const int G = 1 + next() % 4, bm = (next() & 1) ? 64 : ((next() & 1) ? 128 : 256), longest = 1 + next() % ((next() & 1) ? 3000 : 300);
        p.Hk = 1 + next() % 34;
        p.H = p.Hk * G;
        p.B = 1 + next() % ((next() & 1) ? 12 : 70);
        std::vector<int> cu(p.B + 1, 0);
        int most = 1;
        for (int b = 0; b < p.B; b++) {
            const int n = next() % 4 == 0 ? 0 : next() % (longest + 1);
            cu[b + 1] = cu[b] + n;
            most = n > most ? n : most;
        }
        const bool ragged = next() % 3 != 0;
        p.Lq = ragged ? (next() % 8 ? most : 1 + next() % most) : longest;  // (a caller may name less than the longest: the rest is not computed)
        if (ragged) p.cu_q = cu.data();
        p.total_q = cu[p.B];
        const int n_mb = (p.Lq + bm - 1) / bm, grid = row_grid(p, bm), all = p.B * p.Hk * n_mb * G;
        whole += p.row_lists < 0;
        if (grid % 8 || grid > 2 * all + 8 * n_mb * G + (ragged ? 0 : 8 * p.B * p.Hk * G)) {
            std::printf("FAILED: %d workgroups for B %d Hk %d G %d blocks %d ragged %d\n", grid, p.B, p.Hk, G, n_mb, ragged);
            return 1;
        }
        std::vector<int> seen((size_t)p.B * p.H * n_mb, 0);
        for (int id = 0; id < grid; id++) {
            const RowUnit u = row_unit(p, id, bm);
            if (u.block < 0) continue;
            if (u.pair < 0 || u.pair >= p.B * p.Hk || u.block >= n_mb) {
                std::printf("FAILED: workgroup %d has block %d of pair %d\n", id, u.block, u.pair);
                return 1;
            }
            seen[((size_t)(u.pair / p.Hk) * p.H + u.pair % p.Hk * G + (id / 8) % G) * n_mb + u.block]++;
        }
        for (int b = 0; b < p.B; b++)
            for (int i = 0; i < p.H * n_mb; i++) {
                const int want = i % n_mb * bm < (ragged ? cu[b + 1] - cu[b] : p.Lq) ? 1 : 0;
                if (seen[(size_t)b * p.H * n_mb + i] != want) {
                    std::printf("FAILED: B %d Hk %d G %d ragged %d: entry %d, head %d, block %d has %d workgroups\n", p.B, p.Hk, G, ragged, b, i / n_mb, i % n_mb,
                                seen[(size_t)b * p.H * n_mb + i]);
                    return 1;
                }
            }
        checked += grid;
    }
    // steps of an entry, and per part of a batch, whatever lengths come out of a caller's longest length and totals
    for (int lq : {-5000, -64, -1, 0, 1, 64, 700})
        for (int lk : {-90000, -128, -1, 0, 1, 129, 3000})
            for (int causal = 0; causal < 2; causal++)
                for (int bm : {32, 64}) {
                    const int64_t steps = kv_head_steps(lq, lk, causal, bm);
                    if (steps < 0 || ((lq <= 0 || lk <= 0) && steps != 0) || kv_part_quota(steps * 64) < KV_PART_MIN) {
                        std::printf("FAILED: %lld steps for %d rows, %d keys\n", (long long)steps, lq, lk);
                        return 1;
                    }
                }
    // rows of a matrix in pieces of 16, at any size: where 32 bits hold neither the matrix nor the way to a row
    for (int rows : {1, 15, 16, 17, 300, 46352, 65536, 131071})
        for (uint32_t row_bytes : {16u, 2u * 46352u, 2u * 65536u, (1u << 25) - 16u})
            for (int first = 0; first < rows; first += 16)
                for (int i = 0; i < 16; i++) {
                    const RowPiece at = row_piece(first, rows, i, row_bytes);
                    const int row = first + i < rows ? first + i : rows - 1;
                    if (at.base + (int64_t)at.off != (int64_t)row * row_bytes || at.off > (15u << 25)) {
                        std::printf("FAILED: row %d of %d, %u bytes each, lies at %lld + %u\n", row, rows, row_bytes, (long long)at.base, at.off);
                        return 1;
                    }
                }
    // what is fetched for a chunk of a mask row: inside the row, and the chunk's keys are among it
    for (int lk = 8; lk < 700; lk++)
        for (int kk = 0; kk < lk + 512; kk += 8) {
            const int at = mask_piece_at(false, kk, lk), bits = mask_piece_at(true, kk, lk), row_bytes = ((lk + 7) / 8 + 7) / 8 * 8;
            const bool in = at >= 0 && at + 8 <= lk && (kk >= lk || (at <= kk && kk < at + 8 && at == (lk % 8 ? chunk8_at<true>(kk, lk) : chunk8_at<false>(kk, lk))));
            const bool in_bits = bits >= 0 && bits % 8 == 0 && bits + 8 <= row_bytes && (kk >= lk || (8 * bits <= kk && kk < 8 * bits + 64));
            if (!in || !in_bits) {
                std::printf("FAILED: chunk %d of %d keys is fetched from %d (bits: byte %d)\n", kk, lk, at, bits);
                return 1;
            }
        }
    std::printf("%s (%lld workgroups, %lld batches of whole entries)\n", whole > 100 ? "OK" : "FAILED", checked, whole);
    return whole > 100 ? 0 : 1;
}
