/*
 * sampler_window_range.h -- the keys of a range of the mass histogram's bins, cut into sub-bins
 * (sampler_window.h). Compiles as host C++ and as HIP device code.
 */
#ifndef GEIST_SAMPLER_WINDOW_RANGE_H
#define GEIST_SAMPLER_WINDOW_RANGE_H

#include "glibc_expf.h" /* GEIST_HD */

namespace gs {

constexpr int WIN_SUB = 512; /* sub-bins of a range's keys: a few entries each */

/* The keys klo .. khi, cut into at most WIN_SUB sub-bins of 2^shift from the greatest down. */
struct WinRange {
    uint32_t khi, span;
    int      shift;
};
GEIST_HD WinRange win_range(uint32_t klo, uint32_t khi) {
    WinRange r;
    r.khi  = khi;
    r.span = khi - klo;
    const int bits = r.span ? 32 - __builtin_clz(r.span) : 0;
    static_assert(WIN_SUB == 1 << 9, "nine bits of the range");
    r.shift = bits > 9 ? bits - 9 : 0;
    return r;
}
/* The sub-bin of a key, -1 for one outside klo .. khi: an index into WIN_SUB words. */
GEIST_HD int win_sub(const WinRange &r, uint32_t key) {
    const uint32_t at = r.khi - key; /* (wraps beyond span for a key above khi) */
    return at <= r.span ? (int) (at >> r.shift) : -1;
}
/* The range of the keys of sub-bin b. */
GEIST_HD WinRange win_range_of_sub(const WinRange &r, int b) {
    const uint32_t off  = (uint32_t) b << r.shift; /* of its greatest key */
    const uint32_t own  = (1u << r.shift) - 1u, left = r.span - off;
    const uint32_t span = own < left ? own : left;
    return win_range(r.khi - off - span, r.khi - off);
}

} // namespace gs
#endif
