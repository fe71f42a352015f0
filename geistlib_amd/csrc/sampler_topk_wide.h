/*
 * sampler_topk_wide.h -- top-k for a k of hundreds (sampler.c:178-228 and the chain behind it).
 *
 *   k_tmax_scan   (chunks, rows): the largest of every 32 logits, raw where the penalties can only
 *                 lower one (they, and the soft-cap, are then this file's).
 *   k_topk_wide   (rows), 1024 threads. The k_sel-th largest of the row's thread maxima (k_sel >= k,
 *                 with penalties by a margin) bounds the row's k-th largest element from below: by a
 *                 two-digit histogram of the maxima. The threads at or above it are read again, 32
 *                 logits each, what reaches the bound is listed, penalised, capped and put in order
 *                 (bins of the keys' range, a bin's few entries by counting), and the tail shared by
 *                 every sorted mode draws. A row that this cannot certify -- fewer than k reach the
 *                 bound after the penalties, long runs of equal values, rows of -inf -- selects over
 *                 the whole row (topk_row_general).
 *
 * Before, k above 128 (and the rows of smaller k whose thread lists overflowed) went to the whole-row
 * selection, five passes by one workgroup: us a call before / now, k = 150 1 x 104576 178 / 11.4, 8 x
 * 128230 306 / 13.8, 256 x 151936 295 / 38.9; k = 200 with 500 ids of history 8 x 128230 469 / 15.9, 111 x
 * 162496 482 / 27; k = 173 with a soft-cap 7 x 90368 1177 / 13.1; k = 1000 64 x 128256 395 / 28.7; the
 * kernel alone 5 to 9 us of that.
 *
 * Bound by its chain of steps (about thirty, a barrier each), not by bytes: a row's maxima are 16
 * KB for 128256 logits and what is read again 25 to 40. Hence one workgroup of 1024 threads to a row,
 * and no ordering by comparing all with all: n entries take n / 1024 turns whatever n is.
 */
#ifndef GEIST_SAMPLER_TOPK_WIDE_H
#define GEIST_SAMPLER_TOPK_WIDE_H

namespace gs {

constexpr int WK_THREADS = 1024;
constexpr int WK_WAVES   = WK_THREADS / WAVE;
constexpr int WK_BINS    = 2 * WK_THREADS; /* a digit of eleven bits; bins of the final order */
constexpr int WK_LIST    = 2048;           /* elements at or above the bound */
constexpr int WK_SEL     = 2048;           /* threads that are read again */
constexpr int WK_NV      = 8;              /* float4 groups of a scanning thread */
constexpr int WK_TURN    = 4;              /* groups a thread reads before it uses them */
static_assert(WIDE_K_SEL_MAX < WK_SEL && WIDE_K_SEL_MAX < WK_LIST, "room beyond what is wanted");
static_assert(WK_LIST == 2 * WK_THREADS && WK_LIST <= HT_SLOTS / 2, "two entries per thread");

/* LDS of the workgroup; the history's table and the bins end before the entries are ordered, the
 * whole-row selection uses none of them. */
struct WideShared {
    uint64_t pack[WK_LIST];     /* entries in order */
    uint32_t val[WK_LIST];      /* listed entries: the logit's bits, then its key */
    uint32_t idx[WK_LIST];
    uint32_t bins[WK_BINS];
    uint16_t sel[WK_SEL];
    int      scan[WK_WAVES];
    uint32_t mx;
    int      n_sel, n_list, n_real, digit, left;
};

/* Inclusive sums over the workgroup's 1024 threads in thread order; ends behind a barrier. */
__device__ __forceinline__ int wide_scan(int v, int *s_scan) {
    const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    v = wave_scan_i32_dpp(v);
    if (lane == WAVE - 1)
        s_scan[w] = v;
    __syncthreads();
    const int t    = s_scan[lane & (WK_WAVES - 1)]; /* sixteen totals, the same in every row of lanes */
    const int incl = wave_scan_i32_dpp(lane < WK_WAVES ? t : 0);
    const int off  = w ? (int) readlane_u32((uint32_t) incl, w - 1) : 0;
    return v + off;
}

/* The digit (eleven bits from `shift`) in which the `need`-th largest of the counted keys lies, and
 * its rank among that digit's; false when fewer were counted. `bins` are counted and published. */
__device__ __forceinline__ bool wide_pick(WideShared &w, int &need, uint32_t &digit) {
    const int tid = threadIdx.x;
    const int b1 = (int) w.bins[WK_BINS - 1 - 2 * tid], b0 = (int) w.bins[WK_BINS - 2 - 2 * tid];
    if (tid == 0)
        w.digit = -1;
    const int incl = wide_scan(b0 + b1, w.scan), before = incl - b0 - b1;
    if (before < need && incl >= need) {
        const bool low = before + b1 < need;
        w.digit        = WK_BINS - 1 - 2 * tid - (low ? 1 : 0);
        w.left         = need - before - (low ? b1 : 0);
    }
    __syncthreads();
    const int d = w.digit;
    digit       = (uint32_t) d;
    need        = w.left;
    return d >= 0;
}

/* The row's candidates, ordered, in w.pack[0..k): true. False: the row selects over all of it. */
template <bool PEN, bool MASK, int KPT>
__device__ __forceinline__ bool topk_wide_row(const RowView &rv, const FinalArgs &a, int row,
                                              WideShared &w, int *hkey, uint32_t *hcnt) {
    const int tid = threadIdx.x, n_max = rv.n_chunks * TPB;
    /* the thread maxima, entry q * 1024 + tid */
    const float *tm = a.tmax + (long) row * n_max;
    float        raw[KPT];
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        raw[q] = q * WK_THREADS + tid < n_max ? tm[q * WK_THREADS + tid] : __builtin_nanf("");
    int            hid0 = -1, hid1 = -1, hlen = 0;
    const int32_t *hrow = nullptr;
    if (PEN) { /* the history's first 2048 ids are asked for here */
        hlen = rv.hist_len[row];
        hlen = hlen > rv.hist_ld ? (int) rv.hist_ld : hlen;
        hrow = rv.hist + (long) row * rv.hist_ld;
        if (tid < hlen)
            hid0 = hrow[tid];
        if (tid + WK_THREADS < hlen)
            hid1 = hrow[tid + WK_THREADS];
        static_assert(HT_SLOTS == 4 * WK_THREADS, "one 16-byte piece of each array per thread");
        reinterpret_cast<uint4 *>(hkey)[tid] = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (tid < HT_SLOTS / 8)
            reinterpret_cast<uint4 *>(hcnt)[tid] = make_uint4(0u, 0u, 0u, 0u);
    }
    auto clear_bins = [&] { reinterpret_cast<uint2 *>(w.bins)[tid] = make_uint2(0u, 0u); };
    clear_bins();
    if (tid == 0) {
        w.mx     = 0u;
        w.n_sel  = 0;
        w.n_list = 0;
        w.n_real = 0;
    }
    __syncthreads();
    /* The bound: two digits of eleven bits; a NaN's key is 0 and is not counted. Up to a rank of a
     * quarter of the threads each enters only the largest of its maxima: at least as many reach a
     * bound as of those do, for an eighth of the additions, which queue in the few bins that a row's
     * maxima fall into (256 x 262144, k = 64: 1.9 us). In rows without order a few more than the rank
     * reach it (a thirtieth at 64, an eighth at 256); where the leaders share threads, ids equal modulo
     * 1024 in chunks four apart, up to KPT times the rank do, and a row whose list that overflows selects
     * over the whole row. */
    uint32_t key[KPT];
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        key[q] = f2key(raw[q]);
    if (a.k_sel <= WK_THREADS / 4) {
#pragma unroll
        for (int q = 1; q < KPT; ++q) {
            key[0] = key[q] > key[0] ? key[q] : key[0];
            key[q] = 0u;
        }
    }
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        if (key[q])
            atomicAdd(&w.bins[key[q] >> 21], 1u);
    __syncthreads();
    int      need = a.k_sel;
    uint32_t d1, d2;
    if (!wide_pick(w, need, d1))
        return false; /* fewer maxima than that */
    clear_bins();
    __syncthreads();
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        if (key[q] && (key[q] >> 21) == d1)
            atomicAdd(&w.bins[(key[q] >> 10) & (WK_BINS - 1)], 1u);
    __syncthreads();
    (void) wide_pick(w, need, d2);
    const uint32_t tau = (d1 << 21) | (d2 << 10);
    if (tau < KEY_LOWEST_FINITE)
        return false; /* -inf: the bound says nothing */
    const float B = key2f(tau);
    /* the threads at or above it */
    uint32_t mask = 0u;
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        mask |= (uint32_t) (raw[q] >= B) << q;
    int pos = wave_reserve(__popc(mask), &w.n_sel);
#pragma unroll
    for (int q = 0; q < KPT; ++q)
        if ((mask >> q) & 1u) {
            if (pos < WK_SEL)
                w.sel[pos] = (uint16_t) (q * WK_THREADS + tid);
            ++pos;
        }
    __syncthreads();
    const int n_sel = w.n_sel;
    if (n_sel > WK_SEL)
        return false; /* long runs of equal maxima */
    /* their elements again; what reaches the bound is listed */
    const float *rowp = rv.logits + (long) row * rv.ld;
    const int    n    = rv.n_vocab;
    for (int t0 = 0; t0 < n_sel * WK_NV; t0 += WK_TURN * WK_THREADS) {
        float4 g[WK_TURN];
        int    e[WK_TURN];
#pragma unroll
        for (int r = 0; r < WK_TURN; ++r) {
            const int t = t0 + r * WK_THREADS + tid;
            const float none = __builtin_nanf(""); /* reaches no bound */
            g[r] = make_float4(none, none, none, none);
            e[r] = 0;
            if (t < n_sel * WK_NV) {
                const int s = w.sel[t / WK_NV];
                e[r] = (s / TPB) * rv.per_chunk + 4 * ((t % WK_NV) * TPB + s % TPB);
                if (rv.vec_ok && e[r] + 3 < n) {
                    g[r] = *reinterpret_cast<const float4 *>(rowp + e[r]);
                } else {
                    g[r].x = e[r] + 0 < n ? rowp[e[r] + 0] : none;
                    g[r].y = e[r] + 1 < n ? rowp[e[r] + 1] : none;
                    g[r].z = e[r] + 2 < n ? rowp[e[r] + 2] : none;
                    g[r].w = e[r] + 3 < n ? rowp[e[r] + 3] : none;
                }
            }
        }
        uint32_t keep = 0u;
#pragma unroll
        for (int r = 0; r < WK_TURN; ++r) {
            uint32_t m4 = (uint32_t) (g[r].x >= B) | (uint32_t) (g[r].y >= B) << 1 |
                          (uint32_t) (g[r].z >= B) << 2 | (uint32_t) (g[r].w >= B) << 3;
            if (MASK && m4)
                m4 &= allowed_nibble(rv, row, e[r]);
            keep |= m4 << (4 * r);
        }
        int at = wave_reserve(__popc(keep), &w.n_list);
#pragma unroll
        for (int r = 0; r < WK_TURN; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if ((keep >> (4 * r + c)) & 1u) {
                    if (at < WK_LIST) {
                        w.val[at] = __float_as_uint(f4_get(g[r], c));
                        w.idx[at] = (uint32_t) (e[r] + c);
                    }
                    ++at;
                }
    }
    clear_bins();
    __syncthreads();
    const int n_list = w.n_list;
    if (n_list > WK_LIST)
        return false; /* long runs of equal values */
    /* every thread has the entries tid and tid + 1024 from here on */
    const bool has[2] = {tid < n_list, tid + WK_THREADS < n_list};
    uint32_t   slot[2] = {0u, 0u};
    if (PEN) { /* the candidates claim slots of a table, the history is looked up in it */
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (has[i]) {
                const int id = (int) w.idx[tid + i * WK_THREADS];
                slot[i]      = hist_hash(id);
#pragma unroll 1
                for (int pr = 0; pr < HT_SLOTS && atomicCAS(&hkey[slot[i]], -1, id) != -1; ++pr)
                    slot[i] = (slot[i] + 1u) & (HT_SLOTS - 1);
            }
        __syncthreads();
        auto look_up = [&](int id) {
            if ((unsigned) id >= (unsigned) n)
                return;
            uint32_t h = hist_hash(id);
            int      k = hkey[h];
#pragma unroll 1
            for (int pr = 0; pr < HT_SLOTS && k != id && k != -1; ++pr) {
                h = (h + 1u) & (HT_SLOTS - 1);
                k = hkey[h];
            }
            if (k == id) /* 16-bit counters, two a word: a history holds fewer than 65536 ids */
                atomicAdd(&hcnt[h >> 1], 1u << (16 * (h & 1u)));
        };
        look_up(hid0);
        look_up(hid1);
#pragma unroll 1
        for (int i = tid + 2 * WK_THREADS; i < hlen; i += WK_THREADS)
            look_up(hrow[i]);
        __syncthreads();
    }
    const float    Bc   = a.cap_after ? softcap1(B, rv.softcap) : B;
    const uint32_t lo_k = a.cap_after ? f2key(Bc) : tau;
    uint32_t       ky[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ky[i] = 0u;
        if (!has[i])
            continue;
        float x = __uint_as_float(w.val[tid + i * WK_THREADS]);
        if (PEN) {
            const uint32_t times = (hcnt[slot[i] >> 1] >> (16 * (slot[i] & 1u))) & 0xffffu;
            if (times)
                x = penalise(x, times, rv.rep, rv.inv_rep, rv.freq, rv.pres);
        }
        if (x >= B) { /* (a NaN fails; a capped value has to lie above the capped bound:
                       * FinalArgs::cap_after) */
            if (a.cap_after) {
                const float xc = softcap1(x, rv.softcap);
                ky[i]          = xc > Bc ? f2key(xc) : 0u;
            } else {
                ky[i] = f2key(x);
            }
        }
    }
    {
        const int      real = __popcll(ballot64(ky[0] != 0u)) + __popcll(ballot64(ky[1] != 0u));
        const uint32_t mxk  = wave_max_u32(ky[0] > ky[1] ? ky[0] : ky[1]);
        if ((tid & (WAVE - 1)) == 0 && real) {
            atomicMax(&w.mx, mxk);
            atomicAdd(&w.n_real, real);
        }
    }
    __syncthreads();
    if (w.n_real < a.k)
        return false;
    /* order: bin 0 holds the largest; what a bin holds lies together, then by counting */
    const uint32_t range = w.mx - lo_k;
    const int      sh    = range < (uint32_t) WK_BINS ? 0 : 21 - __clz((int) range);
    uint32_t       bin[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        bin[i] = ky[i] ? (w.mx - ky[i]) >> sh : 0u;
        if (ky[i])
            atomicAdd(&w.bins[bin[i]], 1u);
    }
    __syncthreads();
    {
        const uint2 b    = reinterpret_cast<const uint2 *>(w.bins)[tid];
        const int   incl = wide_scan((int) (b.x + b.y), w.scan);
        reinterpret_cast<uint2 *>(w.bins)[tid] =
            make_uint2((uint32_t) incl - b.x - b.y, (uint32_t) incl - b.y); /* where a bin starts */
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (ky[i])
            w.pack[atomicAdd(&w.bins[bin[i]], 1u)] = pack_best(ky[i], w.idx[tid + i * WK_THREADS]);
    __syncthreads(); /* bins[b] is now where bin b ends */
    int      to[2];
    uint64_t me[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        to[i] = a.k;
        if (!ky[i])
            continue;
        const int from = bin[i] ? (int) w.bins[bin[i] - 1] : 0, end = (int) w.bins[bin[i]];
        me[i] = pack_best(ky[i], w.idx[tid + i * WK_THREADS]);
        if (from >= a.k)
            continue; /* beyond the k largest whatever its place */
        to[i] = from;
        for (int j = from; j < end; ++j)
            to[i] += w.pack[j] > me[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (to[i] < a.k)
            w.pack[to[i]] = me[i];
    __syncthreads();
    return true;
}

template <bool PEN, bool MASK, int KPT>
__global__ __launch_bounds__(WK_THREADS) void k_topk_wide(RowView rv, FinalArgs a) {
    __shared__ __align__(16) WideShared s_w;
    __shared__ __align__(16) uint32_t   s_hist[PEN ? HT_SLOTS + HT_SLOTS / 2 : 4];
    __shared__ uint64_t                 s_tab[32];
    __shared__ FinishShared             s_fs;
    __shared__ GeneralShared            s_gs;
    const int row = blockIdx.x, tid = threadIdx.x;
    if (tid < 32)
        s_tab[tid] = g_expf_tab[tid];
    const float u = a.uniforms[row];
    const bool  ok =
        topk_wide_row<PEN, MASK, KPT>(rv, a, row, s_w, reinterpret_cast<int *>(s_hist), s_hist + HT_SLOTS);
    if (a.row_flag && tid == 0)
        a.row_flag[row] = ok ? 1 : 2; /* diagnostics: which path served the row */
    /* what follows is written for one wavefront, or for four */
    if (tid >= (ok && a.k <= 4 * WAVE ? WAVE : TPB))
        return;
    int k = a.k;
    if (!ok) {
        static_assert(!PEN || (HT_SLOTS + HT_SLOTS / 2) >= WK_NV * TPB * 2, "room for a tile's counts");
        __syncthreads();
        k = topk_row_general<WK_NV, PEN, MASK>(rv, row, a.k, s_w.pack, WK_LIST, s_hist, s_gs);
    }
    int tok;
    if (k > 4 * WAVE) {
        tok = finish_sorted(k, s_w.pack, a.inv_t, a.top_p, a.min_p, u, s_fs);
    } else {
        if (tid >= WAVE)
            return;
        tok = k <= WAVE ? finish_sorted_wave<1>(k, s_w.pack, a.inv_t, a.top_p, a.min_p, u, s_tab)
                        : finish_sorted_wave<4>(k, s_w.pack, a.inv_t, a.top_p, a.min_p, u, s_tab);
    }
    if (tid == 0)
        a.out[row] = tok;
}

} // namespace gs
#endif
