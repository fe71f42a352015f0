/*
 * sampler_window.h -- top-p / min-p over the whole vocabulary (src/engine/sampler.c:232-305) for
 * rows whose kept prefix is too wide for the thread-maxima shortcut: nothing is sorted and nothing
 * is listed but the entries around the two places that decide the token.
 *
 * The exp-sum pass leaves, per chunk, a histogram of the masses p = expf((l - max) inv_t) over
 * WIN_BINS bins (16 to a factor of two of p, from p = 1 down). From their sum over the row's chunks
 * (window_locate) the bins are known in which the kept prefix ends and in which the draw falls; the
 * histogram's masses are sums of weights cut to 19 bits, so each place is a range of bins wide enough
 * for what was cut. One pass over the row then (k_window, a workgroup per chunk or few) adds up the exact masses
 * of the normalised probabilities above each range and lists the entries inside them, a few
 * hundred; the workgroup that arrives last orders what little of the list it needs and walks it.
 * Masses are integers (2^-62), so they do not depend on the order of the additions.
 *
 * The histogram decides where to look, never the token: the last workgroup checks that the exact
 * masses put the edge and the draw inside their ranges, and that neither is tied with an entry
 * outside. A row that fails (a range with more entries than the list, a crowd of more than WIN_MANY,
 * sums that are not finite, prefixes that end below p = 2^-32) takes the whole-row walk. Runs of equal values are cut by their ids (window_long).
 */
#ifndef GEIST_SAMPLER_WINDOW_H
#define GEIST_SAMPLER_WINDOW_H

#include "sampler_window_range.h"

namespace gs {

constexpr int WIN_STAGE = 2048; /* entries a workgroup stages in LDS */
constexpr int WIN_MANY  = 8192; /* a crowd of more entries is sooner walked than listed: 24 rows of 50257 in
                                 * halves 99 us so, 229 with lists of up to 16384 */

/* Where to look in a row: the bins [e0, e1] hold the entry at which the nucleus reaches top_p
 * (need_p), [d0, d1] the entry drawn; `last` is the last bin that can hold a kept entry. thr: every
 * element of the bins that matter has a softmax argument above it. ok = 0: not to be found in
 * the histogram. */
struct WinPlan {
    int   e0, e1, d0, d1, last;
    int   need_p, need_m, ok;
    float thr;
};
struct WinLocateShared {
    double cum[4 * TPB];
    double scan[NWAVES];
    int    hit[4];
};

/* The histogram's four bins 4 tid .. 4 tid + 3 (the first `quads` threads', quads = nb / 4), summed
 * over the row's chunks; nb: how many bins are written, a multiple of four. Every thread of the
 * workgroup calls. The loads are asked for before anything is waited for. */
__device__ __forceinline__ void window_sum_hist(const float *__restrict__ hist, int n_chunks, int nb,
                                                WinLocateShared &sh, double (&h)[4]) {
    static_assert(WIN_BINS <= 4 * TPB, "a thread sums four bins");
    const int tid = threadIdx.x;
    h[0] = h[1] = h[2] = h[3] = 0.0;
    /* where that leaves threads over, `groups` of threads with every groups-th chunk each: the
     * step is a few round trips to the second-level cache */
    const int quads  = nb >> 2;
    const int groups = TPB / quads; /* 1 or more: nb <= WIN_BINS */
    const int g      = tid / quads, q = tid - g * quads;
    if (g < groups) {
        const float4 *p = reinterpret_cast<const float4 *>(hist) + q;
        for (int c0 = g; c0 < n_chunks; c0 += 16 * groups) {
            /* sixteen loads in flight: the chunk's number is clamped, not tested (a branch around
             * a load would wait for it before the next) */
            float4 v[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int c = c0 + k * groups < n_chunks ? c0 + k * groups : n_chunks - 1;
                v[k]        = p[(long) c * (WIN_BINS / 4)];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float in = c0 + k * groups < n_chunks ? 1.0f : 0.0f; /* (the bins are finite) */
                h[0] += (double) (v[k].x * in);
                h[1] += (double) (v[k].y * in);
                h[2] += (double) (v[k].z * in);
                h[3] += (double) (v[k].w * in);
            }
        }
    }
    if (groups > 1) {
        /* (a group's sums: 4 quads doubles, groups * quads <= TPB) */
        if (g < groups)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sh.cum[i * TPB + tid] = h[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h[i] = 0.0;
            if (tid < quads)
                for (int x = 0; x < groups; ++x)
                    h[i] += sh.cum[i * TPB + x * quads + tid];
        }
        __syncthreads();
    }
}

/* The plan of a row from window_sum_hist's bins; every thread of the workgroup calls and receives
 * the same, and so does every other workgroup that reads the same bins. */
__device__ __forceinline__ WinPlan window_locate(const double (&h)[4], int nb, double sum, float top_p,
                                                 float min_p, float u, int cap, WinLocateShared &sh) {
    const int  tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    const bool use_p = top_p > 0.0f && top_p < 1.0f, use_m = min_p > 0.0f;
    const double own = (h[0] + h[1]) + (h[2] + h[3]);
    double       run = wave_scan_f64_dpp(own);
    if (lane == WAVE - 1)
        sh.scan[w] = run;
    if (tid < 4)
        sh.hit[tid] = nb;
    __syncthreads();
    run -= own;
    for (int x = 0; x < w; ++x)
        run += sh.scan[x];
    double cum[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        run += h[i];
        cum[i]               = run;
        sh.cum[4 * tid + i] = run;
    }
    __syncthreads();
    /* hit[slot], hit[slot + 1]: the first bins at which the running mass reaches a and b. The first: a
     * thread's masses and its neighbour's are rounded on their own ways, so the running mass can
     * step back by a last bit between them, and a target within that bit is reached twice. */
    auto find = [&](int slot, double a, double b) {
        double before = tid ? sh.cum[4 * tid - 1] : -1.0; /* (a target of 0 is reached in bin 0) */
        if (tid == 0) {
            a = a > 0.0 ? a : 0.0;
            b = b > 0.0 ? b : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (before < a && cum[i] >= a)
                atomicMin(&sh.hit[slot], 4 * tid + i);
            if (before < b && cum[i] >= b)
                atomicMin(&sh.hit[slot + 1], 4 * tid + i);
            before = cum[i];
        }
    };
    /* A bin is an integer sum of weights of 19 bits (win_weight), each cut by less than 2^-17 of itself,
     * scaled with one rounding: too small by at most 7.7e-6 of its mass, never too large by more than
     * 6e-8. With the roundings of pn and of the tolerance mode's exponentials (some 1e-7) twice
     * and a half fits the margin. k_window checks where edge and draw lie; which of top-p and min-p
     * ends the prefix first rests on this bound alone. */
    const double m = 2e-5 * sum, t = (double) top_p * sum;
    if (use_p)
        find(0, t - m, t + m);
    __syncthreads();
    WinPlan r;
    r.e0 = use_p ? sh.hit[0] : nb;
    r.e1 = use_p ? (sh.hit[1] < nb ? sh.hit[1] : nb - 1) : nb;
    bool have_p = use_p && r.e0 < nb;
    /* the bins around min_p (of the row's largest p, which is 1) */
    int  f0 = nb, f1 = nb;
    bool have_m = false;
    if (use_m && min_p <= 1.0f) {
        const float up = (float) ((double) min_p * (1.0 + 1e-6)), dn = (float) ((double) min_p * (1.0 - 1e-6));
        f0     = up < 1.0f ? win_bin(__float_as_uint(up)) : 0;
        f1     = win_bin(__float_as_uint(dn));
        have_m = f1 < nb;
    }
    /* the kept prefix is the shorter of the two */
    r.ok     = (have_p || have_m) && !(use_m && min_p > 1.0f);
    r.need_p = have_p && !(have_m && f1 < r.e0);
    r.need_m = have_m && !(have_p && r.e1 < f0);
    r.last   = 0;
    r.d0 = r.d1 = 0;
    r.thr       = 0.0f;
    double lo = 0.0, hi = 0.0;
    if (r.ok) {
        lo     = __builtin_inf();
        hi     = __builtin_inf();
        r.last = nb - 1;
        if (r.need_p) {
            lo     = t;
            hi     = t + (double) __uint_as_float(win_key_hi(r.e0)) + m;
            r.last = r.e1;
        }
        if (r.need_m) {
            const double a = (f0 > 0 ? sh.cum[f0 - 1] : 0.0) - m, b = sh.cum[f1] + m;
            lo     = a < lo ? a : lo;
            hi     = b < hi ? b : hi;
            r.last = f1 < r.last ? f1 : r.last;
        }
    }
    find(2, (double) u * lo - m, (double) u * hi + m);
    __syncthreads();
    r.d0 = sh.hit[2] < r.last ? sh.hit[2] : r.last;
    r.d1 = sh.hit[3] < r.last ? sh.hit[3] : r.last;
    /* a range of which the masses alone tell that its entries are too many -- more than the list's (weights
     * are rounded down, so the number is), or a crowd, far above the ranges beside it --: the row is
     * walked in full, and its workgroups need not find that out */
    auto below    = [&](int d) { return d >= 0 ? sh.cum[d < nb ? d : nb - 1] : 0.0; };
    auto too_many = [&](int a, int b) {
        const double mass = below(b) - below(a - 1), p = (double) __uint_as_float(win_key_hi(a));
        if (mass <= (double) WIN_MANY * p)
            return false;
        const int    w      = b - a + 1;
        const double beside = (below(a - 1) - below(a - 1 - w)) + (below(b + w) - below(b));
        return mass > (double) (cap + 1) * p || mass > 2.0 * beside;
    };
    if (r.ok && (too_many(r.d0, r.d1) || (r.need_p && too_many(r.e0, r.e1))))
        r.ok = 0;
    int deep = r.d1;
    if (r.need_p && r.e1 > deep)
        deep = r.e1;
    if (r.need_m && f1 > deep)
        deep = f1;
    /* (a deep p of 2^-32 at least: the logarithm's error is far below the slack) */
    r.thr = __logf(__uint_as_float(win_key_lo(deep))) - 1e-3f;
    __syncthreads(); /* the shared words may be used again */
    return r;
}

/* A row of the pass's workspace; `arrive` and `count` are zero between launches. */
struct WinRow {
    uint32_t arrive, count;
    WinPlan  plan;
    float    mx;
    double   sum;
    uint32_t pad[18];
};
static_assert(sizeof(WinRow) == 128, "a cache line per row");
struct alignas(32) WinChunk { /* what a workgroup reports, within a cache line: */
    uint64_t above_e, above_d, above_m; /* mass before the edge's bins, the draw's, of the min-p prefix */
};

struct WinFindShared {
    uint64_t mass[2][WIN_SUB]; /* of the edge's range, of the draw's */
    uint64_t small[TPB];
    uint64_t scan[2][NWAVES];
    uint64_t res_before, out_pack, out_mass;
    int      res_bin, n_small, found, stray;
    uint32_t kmin, kmax;
};

/* a list entry: pack_best(pn, id) with its two leading id bits replaced by the roles */
constexpr uint64_t WIN_ROLE_E = 0x80000000ull, WIN_ROLE_D = 0x40000000ull;
__device__ __forceinline__ uint64_t win_entry(uint32_t key, uint32_t id, bool edge, bool draw) {
    return (pack_best(key, id) & ~(WIN_ROLE_E | WIN_ROLE_D)) | (edge ? WIN_ROLE_E : 0ull) |
           (draw ? WIN_ROLE_D : 0ull);
}
__device__ __forceinline__ uint64_t win_pack(uint64_t entry) { return entry | WIN_ROLE_E | WIN_ROLE_D; }

/* Of the c entries in sh.small, at most one per thread, the one at which the running mass, sh.res_before
 * before them, reaches `target`. */
__device__ __forceinline__ void window_pick(int c, uint64_t target, WinFindShared &sh) {
    const int tid = threadIdx.x;
    if (tid < c) {
        /* the running mass up to this entry: no order needed, the entries are few */
        const uint64_t me = sh.small[tid], fx = pn_fx_bits(best_key(me));
        uint64_t       r = sh.res_before;
        for (int j = 0; j < c; ++j) {
            const uint64_t o = sh.small[j];
            r += o >= me ? pn_fx_bits(best_key(o)) : 0ull;
        }
        if (r >= target && r - fx < target) {
            sh.out_pack = me;
            sh.out_mass = r;
            sh.found    = 1;
        }
    }
}

/* The first entry of the list with role `role` and pack >= lim, in the order of the packs from the
 * greatest down, at which the running mass reaches `target`: sh.out_pack, and sh.out_mass, the
 * mass with it. each(f): f(entry) for every entry of the list, the workgroup's threads sharing them.
 * run: the running mass before this thread's two sub-bins, m0 and m1 their masses. False when it is
 * not reached, or a sub-bin holds more entries than the workgroup has threads (window_long's).
 * Entries below lim leave the sub-bins' masses too great from the sub-bin of lim on, where no target
 * lies beyond lim. sh.res_bin is -1 and sh.n_small, sh.found are 0 on entry (behind a barrier). */
template <typename Each>
__device__ __forceinline__ bool window_find(Each each, uint64_t role, uint64_t lim,
                                            const WinRange &range, uint64_t run, uint64_t m0,
                                            uint64_t m1, uint64_t target, WinFindShared &sh) {
    const int tid  = threadIdx.x;
    auto      here = [&](int b, uint64_t m) { /* (a mass can tell that the entries are too many) */
        if (m && run < target && run + m >= target &&
            m / TPB <= pn_fx_bits(range.khi - ((uint32_t) b << range.shift))) {
            sh.res_bin    = b;
            sh.res_before = run;
        }
        run += m;
    };
    here(2 * tid, m0);
    here(2 * tid + 1, m1);
    __syncthreads();
    const int b = sh.res_bin;
    if (b < 0)
        return false;
    each([&](uint64_t e) {
        if ((e & role) && win_sub(range, best_key(e)) == b && win_pack(e) >= lim) {
            const int at = atomicAdd(&sh.n_small, 1);
            if (at < TPB)
                sh.small[at] = win_pack(e);
        }
    });
    __syncthreads();
    const int c = sh.n_small;
    if (c > TPB)
        return false;
    window_pick(c, target, sh);
    __syncthreads();
    return sh.found != 0;
}

/* The running masses before thread tid's two words 2 tid, 2 tid + 1 of mass[], itself without them;
 * m0, m1: the two. The words are complete (a barrier behind their additions). */
__device__ __forceinline__ uint64_t window_scan_subs(const uint64_t *mass, uint64_t *scan, uint64_t &m0,
                                                     uint64_t &m1) {
    static_assert(WIN_SUB == 2 * TPB, "two sub-bins to a thread");
    const int tid = threadIdx.x;
    m0            = mass[2 * tid];
    m1            = mass[2 * tid + 1];
    uint64_t run  = wave_scan_u64(m0 + m1);
    if ((tid & (WAVE - 1)) == WAVE - 1)
        scan[tid / WAVE] = run;
    __syncthreads();
    run -= m0 + m1;
    for (int w = 0; w < tid / WAVE; ++w)
        run += scan[w];
    return run;
}

/* An entry's mass to word `at` of mass[], -1: none; every lane of the wavefront calls. The lanes with
 * the first one's word and key are one addition: a run of equal values would queue up at its word. */
__device__ __forceinline__ void window_add(uint64_t *mass, int at, uint32_t key) {
    const uint64_t any = __ballot(at >= 0);
    if (!any)
        return;
    const int      lead = __ffsll((long long) any) - 1;
    const uint32_t k0   = readlane_u32(key, lead);
    const int      at0  = (int) readlane_u32((uint32_t) at, lead);
    const uint64_t same = __ballot(at == at0 && key == k0);
    const bool     one  = (int) (threadIdx.x & (WAVE - 1)) == lead;
    const uint64_t fx   = pn_fx_bits(key) * (one ? (uint64_t) __popcll(same) : 1ull);
    if (one || (at >= 0 && !(at == at0 && key == k0)))
        atomicAdd((unsigned long long *) &mass[at], (unsigned long long) fx);
}

/* The same for lists that window_find does not serve, with a crowd in one sub-bin: edge and draw, the checks of k_window included; the token, or -1. A sub-bin with more
 * entries than threads is cut into sub-bins in turn, from its least key to its greatest, and where
 * these are one, by the ids (below n_ids), so runs of equal values end as any others do. Called by the
 * whole workgroup; sh.mass[0] is used again. */
template <typename Over, typename Under>
__device__ __forceinline__ int window_long(const uint64_t *list, uint32_t total, const WinPlan &plan,
                                           const WinRange &re, const WinRange &rd, uint64_t above_e,
                                           uint64_t above_d, uint64_t above_m, int n_ids, float top_p,
                                           uint32_t floor_key, float u, Over key_over, Under key_under,
                                           WinFindShared &sh) {
    const int     tid = threadIdx.x;
    constexpr int PER = 8; /* entries of a thread that stay in registers, and loads in flight for the rest */
    uint64_t      first[PER];
    auto load = [&](uint32_t i0, uint64_t (&e)[PER]) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const uint32_t i = i0 + q * TPB + tid;
            e[q]             = coop_ld64(list + (i < total ? i : total - 1u));
            e[q]             = i < total ? e[q] : 0ull;
        }
    };
    load(0, first);
    auto each = [&](auto &&f) {
        uint64_t e[PER], next[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q)
            e[q] = first[q];
#pragma unroll 1
        for (uint32_t i0 = 0; i0 < total; i0 += PER * TPB) {
            if (i0 + PER * TPB < total)
                load(i0 + PER * TPB, next);
#pragma unroll
            for (int q = 0; q < PER; ++q)
                f(e[q]);
#pragma unroll
            for (int q = 0; q < PER; ++q)
                e[q] = next[q];
        }
    };
    uint64_t edge_pack = 0ull, mass_keep = 0ull;
#pragma unroll 1
    for (int draw = plan.need_p ? 0 : 1; draw < 2; ++draw) {
        if (draw && plan.need_m && (!plan.need_p || floor_key > best_key(edge_pack))) {
            edge_pack = (uint64_t) floor_key << 32;
            mass_keep = above_m;
        }
        const uint64_t target = draw ? (uint64_t) __double2ull_rd((double) u * (double) mass_keep) + 1ull
                                     : (uint64_t) __double2ull_ru((double) top_p * 0x1p62);
        const uint64_t role   = draw ? WIN_ROLE_D : WIN_ROLE_E;
        uint64_t       before = draw ? above_d : above_e;
        if (before >= target || (draw && target > mass_keep))
            return -1;
        WinRange range = draw ? rd : re;
        uint32_t key   = 0u; /* with by_id: the key whose (complemented) ids the range holds */
        bool     by_id = false, whole = true;
        auto     sub   = [&](uint64_t e) {
            if (!(e & role))
                return -1;
            if (!by_id)
                return win_sub(range, best_key(e));
            return best_key(e) == key ? win_sub(range, (uint32_t) win_pack(e)) : -1;
        };
        int c;
#pragma unroll 1
        for (;;) {
            __syncthreads(); /* the words are read */
            for (int i = tid; i < WIN_SUB; i += TPB)
                sh.mass[0][i] = 0ull;
            if (tid == 0) {
                sh.res_bin = -1;
                sh.n_small = 0;
                sh.found   = 0;
                sh.kmin    = 0xffffffffu;
                sh.kmax    = 0u;
            }
            __syncthreads();
            uint32_t kmin = 0xffffffffu, kmax = 0u;
            auto     span = [&](uint64_t e) {
                const uint32_t k = best_key(e);
                kmin             = k < kmin ? k : kmin;
                kmax             = k > kmax ? k : kmax;
            };
            auto spans = [&]() { /* (behind a barrier) */
                if (kmin <= kmax) {
                    atomicMin(&sh.kmin, kmin);
                    atomicMax(&sh.kmax, kmax);
                }
            };
            auto ids_of = [&](uint32_t k) { /* the entries of one key, by their ids */
                key   = k;
                by_id = true;
                range = win_range(0xffffffffu - (uint32_t) (n_ids - 1), 0xffffffffu);
            };
            each([&](uint64_t e) {
                const int at = sub(e);
                if ((e & role) && at < 0 && whole)
                    sh.stray = 1; /* (in no list of a workgroup with this plan) */
                if (at >= 0)
                    span(e);
                window_add(sh.mass[0], at, best_key(e));
            });
            if (!by_id)
                spans();
            __syncthreads();
            if (!by_id && sh.kmin == sh.kmax && !sh.stray) {
                whole = false;
                ids_of(sh.kmax);
                continue;
            }
            uint64_t m0, m1, run = before + window_scan_subs(sh.mass[0], sh.scan[0], m0, m1);
            if (m0 && run < target && run + m0 >= target) {
                sh.res_bin    = 2 * tid;
                sh.res_before = run;
            }
            run += m0;
            if (m1 && run < target && run + m1 >= target) {
                sh.res_bin    = 2 * tid + 1;
                sh.res_before = run;
            }
            __syncthreads();
            const int b = sh.res_bin;
            if (b < 0 || sh.stray)
                return -1;
            const uint64_t run_b = sh.res_before;
            __syncthreads(); /* the words are read */
            if (tid == 0) {
                sh.kmin = 0xffffffffu;
                sh.kmax = 0u;
            }
            kmin = 0xffffffffu;
            kmax = 0u;
            __syncthreads();
            each([&](uint64_t e) {
                if (sub(e) == b && win_pack(e) >= edge_pack) {
                    span(e);
                    const int at = atomicAdd(&sh.n_small, 1);
                    if (at < TPB)
                        sh.small[at] = win_pack(e);
                }
            });
            spans();
            __syncthreads();
            c = sh.n_small;
            if (c <= TPB)
                break;
            before = run_b;
            whole  = false;
            if (by_id)
                range = win_range_of_sub(range, b); /* (2^20 ids: four to a sub-bin at the second turn) */
            else if (sh.kmin == sh.kmax)
                ids_of(sh.kmax);
            else
                range = win_range(sh.kmin, sh.kmax);
        }
        window_pick(c, target, sh);
        __syncthreads();
        if (!sh.found)
            return -1;
        const uint64_t got = sh.out_pack;
        if (best_key(got) >= key_over(draw ? plan.d0 : plan.e0) ||
            best_key(got) <= key_under(draw ? plan.d1 : plan.e1))
            return -1;
        if (draw)
            return (int) best_idx(got);
        edge_pack = got;
        mass_keep = sh.out_mass;
    }
    return -1;
}

/* LOCATE: every workgroup finds its row's plan for itself (small batches: one launch less, and no
 * shortcut in front); otherwise the rows flagged 1 by k_final_sorted are served, with its plans.
 *
 * What bounds it: in a small batch a chain of waits -- for 24 rows of 50257 (device timestamps) 3.0
 * us to the histograms' sums, 2.3 to the plan, 2.5 over the elements, 2 to list, report and arrive,
 * 1.0 to read the reports, 3.0 to find edge and draw --, in a large one the exponentials and exact
 * divisions of the kept elements (256 rows of 262144 with half of each kept: 200 us). The exp-sum pass pays
 * for the histogram with 32-bit integer additions in LDS, 8.2 -> 10.4 us for those 24 rows in chunks
 * of 8192; binary32 additions took it to 17.0. A large batch whose rows keep some hundreds pays more than
 * the list of the kept entries took that this replaces (256 rows of 100000, scale 3, T 0.8, top-p 0.9: the
 * pass 34 -> 40 us, list and list walk 41 -> k_window 48, the call 88 -> 99). 24 rows of 50257, top-p 0.95, nuclei from ten entries
 * to ten thousand: 152 -> 26 us a call (four to six launches before, half of the rows walked in
 * full); 64 rows of 128256 normal logits 163 -> 63, one 80 -> 23.
 * The whole-row walk is in the small form and for the first calls with such rows in a large one; that and
 * penalties cost the large form 64 bytes of scratch. */
template <bool PEN, bool LOCATE>
__global__ __launch_bounds__(TPB, 3) void k_window(RowView rv, SortedRowArgs g, WinSpace win, int win_bins, int per_wg,
                                                float top_p, float min_p,
                                                const float *__restrict__ uniforms,
                                                int32_t *__restrict__ row_flag,
                                                int32_t *__restrict__ out,
                                                int32_t *__restrict__ path, int defer_walk,
                                                uint32_t *__restrict__ walk_hint,
                                                uint32_t walk_call) {
    constexpr int NV = LOCATE ? 2 : 8;
    /* LDS in two parts: the plan's words, then the list's staging, or the whole-row walk's words; and
     * the history's count table, then the words of window_find */
    __shared__ union {
        uint64_t        list[WIN_STAGE];
        SortedGenShared gen;
        struct {
            WinLocateShared loc;
            double          csum[MAX_CHUNKS];
        } first;
    } sa;
    __shared__ union {
        WinFindShared find;
        __align__(16) uint32_t cnt16[PEN ? NV * TPB * 2 : 1];
    } sb;
    __shared__ uint64_t s_tab[32];
    __shared__ uint64_t s_part[NWAVES][3];
    __shared__ uint64_t s_sum[3];
    __shared__ uint32_t s_n, s_base;
    __shared__ int      s_last;
    __shared__ double   s_total;
    __shared__ int      s_scan[NWAVES];
    __shared__ int      s_pick;
    int row, wg; /* the row's workgroup number wg has the chunks from wg * per_wg on */
    xcd_row_chunk(row, wg);
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), C = rv.n_chunks, W = (int) gridDim.x;
    WinRow     *wr   = static_cast<WinRow *>(win.row) + row;
    int         flag = 1;
    if (!LOCATE) {
        flag = row_flag[row];
        if (flag != 1 && flag != 2)
            return;
    }
    const float u = uniforms[row];
    WinPlan     plan;
    float       mx;
    double      tot;
    int         base, end;
    chunk_bounds<NV>(rv, wg * per_wg, base, end);
    float4 v[NV];
    load_raw<NV>(rv, rv.logits + (long) row * rv.ld, base, end, v);
    if (LOCATE) {
        static_assert(MAX_CHUNKS <= TPB, "a thread per chunk");
        const double   cs = tid < C ? g.chunk_sum[(long) row * C + tid] : 0.0;
        const uint64_t cb = tid < C ? g.chunk_best[(long) row * C + tid] : 0ull;
        double         h[4];
        window_sum_hist(win.hist + (long) row * C * WIN_BINS, C, win_bins, sa.first.loc, h);
        if (tid < C)
            sa.first.csum[tid] = cs;
        mx  = key2f(best_key(block_max_u64(cb, s_part[0])));
        tot = 0.0;
        for (int c = 0; c < C; ++c)
            tot += sa.first.csum[c];
        if (tot != tot && !(min_p > 0.0f)) { /* (k_final_sorted's answer for such a row) */
            if (wg == 0 && tid == 0) {
                row_flag[row] = 0;
                out[row]      = rv.n_vocab - 1;
                path[row]     = PATH_WINDOW;
            }
            return;
        }
        plan = window_locate(h, win_bins, tot, top_p, min_p, u, win.cap, sa.first.loc);
        const bool finite = tot > 0.0 && tot < __builtin_inf() && mx > -__builtin_inff() && mx < __builtin_inff();
        flag = finite && plan.ok ? 1 : 2;
    } else {
        plan = wr->plan;
        mx   = wr->mx;
        tot  = wr->sum;
    }
    bool served = false;
    if (flag == 1) {
        const uint64_t tabv = g_expf_tab[tid & 31];
        if (tid < 32)
            s_tab[tid] = tabv;
        if (tid == 0)
            s_n = 0;
        const float pn_0    = (float) (1.0 / tot);
        const float floor_w = __fmul_rn(min_p, pn_0);
        const int   e0 = plan.need_p ? plan.e0 : 0, e1 = plan.need_p ? plan.e1 : -1;
        uint64_t    a_e = 0, a_d = 0, a_m = 0;
        const int last_chunk = (wg + 1) * per_wg < C ? (wg + 1) * per_wg : C;
#pragma unroll 1
        for (int chunk = wg * per_wg;;) {
            transform_loaded_chunk<NV, PEN>(rv, row, rv.n_rows, base, end, sb.cnt16, v);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const int id = base + 4 * (j * TPB + tid);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float arg = softmax_arg(f4_get(v[j], c), mx, g.inv_t);
                    if (arg > plan.thr) { /* (what pads a chunk holds -inf) */
                        const float    p  = geist_expf_glibc_le0(arg, s_tab);
                        const int      d  = win_bin(__float_as_uint(p));
                        const float    pn = (float) ((double) p / tot);
                        const uint32_t k  = __float_as_uint(pn);
                        const uint64_t fx = pn_fx_bits(k);
                        a_e += d < e0 ? fx : 0ull;
                        a_d += d < plan.d0 ? fx : 0ull;
                        a_m += pn >= floor_w ? fx : 0ull;
                        const bool re = d >= e0 && d <= e1, rd = d >= plan.d0 && d <= plan.d1;
                        if (re || rd) {
                            const uint32_t at = __hip_atomic_fetch_add(&s_n, 1u, __ATOMIC_RELAXED,
                                                                       __HIP_MEMORY_SCOPE_WORKGROUP);
                            if (at < (uint32_t) WIN_STAGE)
                                sa.list[at] = win_entry(k, (uint32_t) (id + c), re, rd);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (LOCATE || ++chunk >= last_chunk)
                break;
            chunk_bounds<NV>(rv, chunk, base, end);
            load_raw<NV>(rv, rv.logits + (long) row * rv.ld, base, end, v);
            __syncthreads(); /* the history table is rebuilt for the next chunk */
        }
        a_e = wave_scan_u64(a_e);
        a_d = wave_scan_u64(a_d);
        a_m = wave_scan_u64(a_m);
        if (lane == WAVE - 1) {
            s_part[tid / WAVE][0] = a_e;
            s_part[tid / WAVE][1] = a_d;
            s_part[tid / WAVE][2] = a_m;
        }
        __syncthreads();
        const uint32_t n = s_n;
        if (tid == 0 && n)
            s_base = __hip_atomic_fetch_add(&wr->count, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        WinChunk *slots = static_cast<WinChunk *>(win.chunk) + (long) row * W;
        if (tid < 3) {
            uint64_t t = 0;
#pragma unroll
            for (int w = 0; w < NWAVES; ++w)
                t += s_part[w][tid];
            coop_st64(&slots[wg].above_e + tid, t);
        }
        uint64_t      *rl  = win.list + (long) row * win.cap;
        const uint32_t cap = (uint32_t) win.cap;
        if (n) {
            __syncthreads();
            const uint32_t b = s_base;
            if (n <= (uint32_t) WIN_STAGE) {
                for (uint32_t i = tid; i < n && b + i < cap; i += TPB)
                    coop_st64(rl + b + i, sa.list[i]);
            } else if (b + n <= cap) {
                /* more entries than the stage holds -- they crowd in one place of the row, or share a
                 * value -- but counted: a second time over the chunks, 1024 elements at a time, and
                 * straight to their places in the row's list */
                if (tid == 0)
                    s_n = 0;
                const int from = wg * per_wg * rv.per_chunk;
                const int to   = last_chunk * rv.per_chunk < rv.n_vocab ? last_chunk * rv.per_chunk : rv.n_vocab;
#pragma unroll 1
                for (int b0 = from; b0 < to; b0 += 4 * TPB) {
                    float4 w[1];
                    __syncthreads(); /* the history table is rebuilt; s_n */
                    fetch_chunk<1, PEN>(rv, row, rv.n_rows, b0, b0 + 4 * TPB < to ? b0 + 4 * TPB : to,
                                        sb.cnt16, w);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float arg = softmax_arg(f4_get(w[0], c), mx, g.inv_t);
                        if (arg > plan.thr) {
                            const float p  = geist_expf_glibc_le0(arg, s_tab);
                            const int   d  = win_bin(__float_as_uint(p));
                            const bool  re = d >= e0 && d <= e1, rd = d >= plan.d0 && d <= plan.d1;
                            if (re || rd) {
                                const uint32_t at = __hip_atomic_fetch_add(&s_n, 1u, __ATOMIC_RELAXED,
                                                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                                coop_st64(rl + b + at,
                                          win_entry(__float_as_uint((float) ((double) p / tot)),
                                                    (uint32_t) (b0 + 4 * tid + c), re, rd));
                            }
                        }
                    }
                }
            }
        }
        /* everything reported is performed before the arrival is */
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            const uint32_t before = __hip_atomic_fetch_add(&wr->arrive, 1u, __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT);
            s_last = before == (uint32_t) W - 1u;
        }
        __syncthreads();
        if (!s_last)
            return;
        /* ---- the row's last workgroup ---- */
        constexpr int EARLY = 4;
        /* (a thread per workgroup; the list's first entries are asked for before its length is known) */
        const uint32_t total = coop_ld32(&wr->count);
        uint64_t       part[3], first[EARLY];
        static_assert(WIN_CAP_MIN >= EARLY * TPB, "the list has places for the early loads");
        const int slot = tid < W ? tid : W - 1;
#pragma unroll
        for (int q = 0; q < 3; ++q)
            part[q] = coop_ld64(&slots[slot].above_e + q);
#pragma unroll
        for (int q = 0; q < EARLY; ++q)
            first[q] = coop_ld64(rl + q * TPB + tid);
#pragma unroll
        for (int q = 0; q < 3; ++q)
            part[q] = tid < W ? part[q] : 0ull;
        /* most lists are in registers with that; the rest of a long one is read each time */
        auto each = [&](auto &&f) {
#pragma unroll
            for (int q = 0; q < EARLY; ++q)
                if ((uint32_t) (q * TPB + tid) < total)
                    f(first[q]);
#pragma unroll 1
            for (uint32_t i0 = EARLY * TPB + tid; i0 < total; i0 += 8 * TPB) {
                uint64_t e[8]; /* eight loads in flight */
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    e[q] = coop_ld64(rl + (i0 + q * TPB < total ? i0 + q * TPB : total - 1u));
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (i0 + q * TPB < total)
                        f(e[q]);
            }
        };
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const uint64_t t = wave_scan_u64(part[q]);
            if (lane == WAVE - 1)
                s_part[tid / WAVE][q] = t;
        }
        __syncthreads();
        for (int i = tid; i < 2 * WIN_SUB; i += TPB)
            (&sb.find.mass[0][0])[i] = 0ull;
        if (tid == 0) {
            coop_st32(&wr->count, 0u);
            coop_st32(&wr->arrive, 0u);
            sb.find.res_bin = -1;
            sb.find.n_small = 0;
            sb.find.found   = 0;
            sb.find.stray   = 0;
        }
        if (tid < 3) {
            uint64_t t = 0;
#pragma unroll
            for (int w = 0; w < NWAVES; ++w)
                t += s_part[w][tid];
            s_sum[tid] = t;
        }
        __syncthreads();
        const uint64_t above_e = s_sum[0], above_d = s_sum[1], above_m = s_sum[2];
        auto pn_bits = [&](uint32_t key) {
            return __float_as_uint((float) ((double) __uint_as_float(key) / tot));
        };
        /* the keys next to a range of bins: an entry outside the range has a key of at least the
         * first or of at most the second */
        auto key_over  = [&](int d) { return d > 0 ? pn_bits(win_key_hi(d) + 1u) : 0xffffffffu; };
        auto key_under = [&](int d) { return pn_bits(win_key_lo(d) - 1u); };
        bool     ok = total <= cap;
        bool     have_p = false;
        uint64_t edge_pack = 0ull, mass_keep = 0ull;
        const WinRange re = win_range(pn_bits(win_key_lo(plan.need_p ? plan.e1 : 0)),
                                      pn_bits(win_key_hi(plan.need_p ? plan.e0 : 0)));
        const WinRange rd = win_range(pn_bits(win_key_lo(plan.d1)), pn_bits(win_key_hi(plan.d0)));
        if (ok) {
            /* both ranges' masses by sub-bin (the words were cleared before the last barrier) */
            each([&](uint64_t e) {
                const uint64_t fx = pn_fx_bits(best_key(e));
                const int      be = e & WIN_ROLE_E ? win_sub(re, best_key(e)) : 0;
                const int      bd = e & WIN_ROLE_D ? win_sub(rd, best_key(e)) : 0;
                if ((be | bd) < 0) /* (in no list of a workgroup with this plan) */
                    sb.find.stray = 1;
                if ((e & WIN_ROLE_E) && be >= 0)
                    atomicAdd((unsigned long long *) &sb.find.mass[0][be], (unsigned long long) fx);
                if ((e & WIN_ROLE_D) && bd >= 0)
                    atomicAdd((unsigned long long *) &sb.find.mass[1][bd], (unsigned long long) fx);
            });
            __syncthreads();
            static_assert(WIN_SUB == 2 * TPB, "two sub-bins to a thread");
            uint64_t m[2][2], run[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                m[k][0] = sb.find.mass[k][2 * tid];
                m[k][1] = sb.find.mass[k][2 * tid + 1];
                run[k]  = wave_scan_u64(m[k][0] + m[k][1]);
                if (lane == WAVE - 1)
                    sb.find.scan[k][tid / WAVE] = run[k];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                run[k] -= m[k][0] + m[k][1];
                for (int w = 0; w < tid / WAVE; ++w)
                    run[k] += sb.find.scan[k][w];
                run[k] += k == 0 ? above_e : above_d;
            }
            ok = sb.find.stray == 0;
            if (ok && plan.need_p) {
                const uint64_t target = (uint64_t) __double2ull_ru((double) top_p * 0x1p62);
                ok = above_e < target && window_find(each, WIN_ROLE_E, 0ull, re, run[0],
                                                     m[0][0], m[0][1], target, sb.find);
                if (ok) {
                    edge_pack = sb.find.out_pack;
                    mass_keep = sb.find.out_mass;
                    have_p    = true;
                    ok = best_key(edge_pack) < key_over(plan.e0) &&
                         best_key(edge_pack) > key_under(plan.e1);
                }
                __syncthreads(); /* (the words are written again) */
                if (tid == 0) {
                    sb.find.res_bin = -1;
                    sb.find.n_small = 0;
                    sb.find.found   = 0;
                }
                __syncthreads();
            }
            if (ok && plan.need_m) {
                const uint32_t kf = __float_as_uint(floor_w);
                if (!have_p || kf > best_key(edge_pack)) {
                    edge_pack = (uint64_t) kf << 32; /* every id with a key at or above the floor */
                    mass_keep = above_m;
                }
            }
            if (ok) {
                /* running mass > u * kept mass  <=>  running mass >= floor(u * kept mass) + 1 */
                const uint64_t target2 = (uint64_t) __double2ull_rd((double) u * (double) mass_keep) + 1ull;
                ok = above_d < target2 && target2 <= mass_keep &&
                     window_find(each, WIN_ROLE_D, edge_pack, rd, run[1], m[1][0],
                                 m[1][1], target2, sb.find);
                if (ok) {
                    const uint64_t got = sb.find.out_pack;
                    ok = best_key(got) < key_over(plan.d0) && best_key(got) > key_under(plan.d1);
                    if (ok && tid == 0) {
                        out[row]  = (int32_t) best_idx(got);
                        path[row] = PATH_WINDOW;
                        row_flag[row] = 0;
                    }
                }
            }
        }
        served = ok;
        if (!ok && total <= cap) {
            const int tok = window_long(rl, total, plan, re, rd, above_e, above_d, above_m, rv.n_vocab, top_p,
                                        __float_as_uint(floor_w), u, key_over, key_under, sb.find);
            served = tok >= 0;
            if (served && tid == 0) {
                out[row]      = tok;
                path[row]     = PATH_WINDOW;
                row_flag[row] = 0;
            }
        }
    } else {
        /* a row without a plan, walked by one workgroup: another from row to row. These alone stay, and as
         * every W-th of an XCD's launch order they would share a quarter of its compute units (64 rows
         * of 128256 in halves 1487 us with the first of each row, 638 so) */
        const int r = row >> 3;
        if (wg != (r + r / W) % W)
            return;
    }
    if (served)
        return;
    /* the whole-row walk: by this workgroup, or by the launch behind that spreads such rows */
    if (tid == 0) {
        row_flag[row] = 2;
        if (walk_hint)
            *walk_hint = walk_call;
    }
    if (defer_walk)
        return;
    const int tok = sorted_general_row<NV, PEN>(rv, row, rv.n_rows, g, top_p, min_p, u, sa.gen, sb.cnt16,
                                                s_tab, s_scan, &s_pick, &s_total);
    if (tid == 0) {
        out[row]  = tok;
        path[row] = PATH_ONE_WORKGROUP;
    }
}

} // namespace gs
#endif
