/* The sub-bins of a range of keys (geistlib_amd/csrc/sampler_window_range.h): every key of the range
 * has one of WIN_SUB places, in descending order of the keys; every key outside has none. Prints the
 * number of violations and of keys looked at. */
#include <cstdio>
#include <random>

#include "../../geistlib_amd/csrc/sampler_window_range.h"

int main() {
    std::mt19937 g(1);
    long         bad = 0, total = 0;
    for (int t = 0; t < 4000; ++t) {
        /* up to the whole of 2^-32 .. 1; a single key among them */
        const uint32_t span = t % 7 == 0 ? 0u : g() >> (5 + g() % 27);
        const uint32_t lo = 0x20000000u + (g() & 0x0fffffffu), hi = lo + span;
        const gs::WinRange r = gs::win_range(lo, hi);
        auto inside = [&](uint32_t k) {
            const int s = gs::win_sub(r, k);
            bad += s < 0 || s >= gs::WIN_SUB;
            if (k > lo) /* the next lower key: the same sub-bin or the next */
                bad += gs::win_sub(r, k - 1) - s != 0 && gs::win_sub(r, k - 1) - s != 1;
            /* the sub-bin's own range: this key, and the next ones of the same sub-bin alone */
            const gs::WinRange in = gs::win_range_of_sub(r, s);
            bad += gs::win_sub(in, k) < 0;
            bad += k > lo && (gs::win_sub(in, k - 1) >= 0) != (gs::win_sub(r, k - 1) == s);
            bad += k < hi && (gs::win_sub(in, k + 1) >= 0) != (gs::win_sub(r, k + 1) == s);
            bad += in.span >= r.span && r.span != 0;
            ++total;
        };
        auto outside = [&](uint32_t k) {
            bad += gs::win_sub(r, k) != -1;
            ++total;
        };
        for (uint32_t k : {lo, hi, lo + span / 2})
            inside(k);
        for (int i = 0; i < 50; ++i)
            inside(lo + (span ? g() % (span + 1) : 0));
        for (uint32_t d : {1u, 2u, 511u, 512u, 1u << 19, 1u << 24}) {
            outside(lo - d);
            outside(hi + d);
        }
        bad += gs::win_sub(r, hi) != 0;
    }
    std::printf("%ld %ld\n", bad, total);
    return 0;
}
