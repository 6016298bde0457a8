// Host-side check of the division by a launch-time number (Divisor / quotient in flash-dmattn_amd/csrc/fdma_params.h, built and run by
// tests/test_quotient.py with g++): against the division of the language, around every multiple where a quotient steps and at the ends of
// the range, for the small divisors all of them and for large ones the powers of two, their neighbours and others.
#include <cstdio>

#include "fdma_params.h"

using namespace fdma;

int main() {
    unsigned rng = 1u;
    auto next = [&]() { rng = rng * 1664525u + 1013904223u; return rng >> 1; };
    long long checked = 0;
    auto check = [&](uint32_t by) {
        const Divisor d = divisor(by);
        auto one = [&](int64_t n) {
            if (n < 0 || n > 0x7fffffff) return true;
            checked++;
            if (quotient((int)n, d) == (int)(n / by)) return true;
            std::printf("FAILED: %lld / %u\n", (long long)n, by);
            return false;
        };
        for (int i = 0; i < 64; i++) {
            const int64_t at = (int64_t)(next() / by) * by, low = (int64_t)i * by, high = (0x7fffffff / by - i) * (int64_t)by;
            for (int64_t n : {at, low, high})
                for (int e = -1; e <= 1; e++)
                    if (!one(n + e)) return false;
        }
        return one(0x7fffffff) && one(0x7ffffffe);
    };
    for (uint32_t by = 1; by <= 20000; by++)
        if (!check(by)) return 1;
    for (int s = 1; s < 31; s++)
        for (int e = -1; e <= 1; e++)
            if ((1u << s) + e > 0 && !check((1u << s) + e)) return 1;
    for (int i = 0; i < 20000; i++)
        if (!check(next() | 1u) || !check(1u + next() % (1u << (1 + i % 30)))) return 1;
    std::printf("OK (%lld quotients)\n", checked);
    return 0;
}
