/*
 * sampler_kernels.h -- host-visible launch interface of the sampling kernels.
 */
#ifndef GEIST_SAMPLER_KERNELS_H
#define GEIST_SAMPLER_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gs {

constexpr int MAX_CHUNKS     = 128;  /* chunks per row */
constexpr int TMAX_LDS       = 8192; /* thread maxima of one row the final kernel holds in LDS */
constexpr int SEL_MAX        = 192;  /* threads whose elements the final kernel re-reads */
constexpr int TOPK_FAST_MAX  = 128;  /* largest k served by the candidate path */
constexpr int WIDE_K_SEL_MAX = 1024; /* largest rank of the bound of k_topk_wide's path ... */
constexpr int WIDE_CHUNKS_MAX = 32;  /* ... whose rows have at most so many chunks of 8192 logits */
/* Above this rank (k, and half of it again with penalties) rows that no scan hands candidates on for
 * take k_topk_wide, below it k_final_topk, whose 256 threads have the shorter chain while few elements
 * are read again: rank 40 2 x 50001 11.9 against 10.9 us, 200 x 60001 23.9 / 23.1; rank 48 11.2 / 11.3
 * and 23.5 / 24.2; 56 11.1 / 12.1 and 23.6 / 24.8; 72 12.5 / 14.7 and 25.3 / 26.8. From rank 90 on
 * k_final_topk's list of 192 threads starts to overflow: 16 x 128255, k = 128, 14.0 / 163. With a
 * soft-cap, which that kernel applies to every element it reads again, from rank 17 on (rank 20 12.0 /
 * 12.9, rank 40 12.4 / 16.6), in rows of up to 16 chunks from the first (rank 5 2 x 50001 11.7 / 12.4, 51 x
 * 223709 23.3 / 22.3). */
constexpr int WIDE_RANK_MIN        = 48;
constexpr int WIDE_RANK_MIN_CAPPED = 16;
/* Rows whose scan could hand candidates on (k_cand_scan, k_final_cand) take that path too, whatever the
 * rank, in batches of 2^25 logits, rows of more than 16 chunks from 2^24 on: their scan leaves the maxima
 * alone, 45.6 against 53.9 us for 256 x 262144. Maxima / candidates: 256 x 262144, k = 64, 56.3 / 63.9; 192 x
 * 262144, k = 40, 43.7 / 48.5 and with penalties 45.3 / 49.2; 256 x 131072 (2^25) 30.0 / 30.6; 64 x 262144 (2^24)
 * 19.3 / 19.3, k = 64 19.6 / 20.1, with penalties 21.0 / 19.8; 110 x 152960 k = 64 19.9 / 26.0, k = 40 with
 * penalties 21.4 / 27.7; of fewer chunks below 2^25 128 x 131072 19.0 / 18.3 and with penalties 20.8 / 19.4, 256 x
 * 65536 19.4 / 18.3 and 21.2 / 19.4, 256 x 100000 24.6 / 24.2 and 26.6 / 25.1. Other rows (masks, unaligned)
 * go by the rank alone: k = 20 with a mask 64 x 262144 21.5 / 20.3, 192 x 262144 46.5 / 44.9. */
inline bool wide_by_size(size_t logits, int n_chunks) {
    return logits >= (size_t) 1 << (n_chunks > 16 ? 24 : 25);
}
constexpr int TOPK_MAX       = 8192; /* the reference caps top_k here (sampler.c:213-215) */
constexpr int HISTORY_MAX    = 65535;

enum { FINAL_TEMPERATURE = 1, FINAL_TOPK = 2, FINAL_SORTED = 3 };

/* One batch of logit rows as the kernels see it, with the transform applied while reading. */
struct RowView {
    const float   *logits; /* row 0 */
    long           ld;
    int            n_vocab;
    int            per_chunk;
    int            n_chunks;
    int            vec_ok; /* rows are 16-byte aligned: float4 loads allowed */
    int            stream_loads; /* this pass is the last to read the rows and they come from HBM:
                                    non-temporal loads */
    const int32_t *hist;   /* NULL = no penalties */
    long           hist_ld;
    const int32_t *hist_len;
    float          rep, freq, pres;
    double         inv_rep; /* 1.0 / (double) rep, see penalise() */
    float          softcap; /* 0 = off */
    int            n_rows; /* rows of the batch (hist_len has that many entries) */
    const uint32_t *allowed;   /* NULL = no mask; bit e of a row's mask set = token e allowed */
    long            allowed_ld; /* words between rows, 0 = one mask for all rows */
    uint64_t       *draw_states = nullptr; /* the rows' generators, when this scan (launch_tmax_scan,
                                    launch_cand_scan, launch_scan_expsum) takes a draw of each and
                                    leaves it in draws[row] for the launches behind; or NULL */
    float          *draws       = nullptr;
};

/* Where the workgroups of a row meet in the one-pass exp-sum kernel (k_scan_expsum): one 64-bit
 * slot per (row, chunk), zero until the chunk's workgroup stores its packed maximum there (never
 * zero). Two such arrays take turns from launch to launch: a launch finds its own array all
 * zero and zeroes the slots that the launch before it used in the other. */
constexpr int ARRIVE_STRIDE_INTS = 32; /* a cache line of its own for every row's counter */
struct MeetSpace {
    uint64_t *slots;       /* [rows * n_chunks] of this launch, zero on entry */
    uint64_t *stale;       /* the slots of the launch before, zeroed by this one */
    uint32_t  stale_count;
    uint32_t  wait_limit;  /* polls before a workgroup reads the row for itself; 0 = do not wait */
    uint32_t  local;       /* the workgroups that meet run on one XCD (the grid deals a row's
                            * workgroups to one, and the device was seen to place them so): a slot
                            * is written with a plain store, which that XCD's L2 holds and serves
                            * to the polls -- a device-scope store is written through to memory
                            * first (a meeting of 63 workgroups: 0.6 against 2.5 us). Should the
                            * workgroups not share an XCD after all, the polls never see the slot,
                            * the bounded wait runs out and each workgroup reads the row itself. */
};

/* Where a sampling step reports that the ids of all its rows are written: `epoch` goes into
 * *h_done (page-locked host memory) after them. h_done == NULL: nobody is told. `rows_done` is a
 * zeroed device counter that the one-launch top-k kernel leaves zeroed (its rows finish in any
 * order; the last one reports). */
struct Notify {
    uint64_t *h_done;
    uint64_t  epoch;
    uint32_t *rows_done;
};
/* a small fill kernel: n 64-bit words at p become zero (recorded into HIP graphs in place of a
 * memset node) */
void launch_zero_words(hipStream_t stream, uint64_t *p, uint32_t n);
/* the same report from a launch of its own, for the steps whose last kernel does not make it */
void launch_publish_epoch(hipStream_t stream, const Notify &nt);

struct Launch {
    RowView     rv;
    int         rows;
    int         nv;  /* float4 groups per thread: 2 or 8 */
    bool        pen; /* history lookup on */
    hipStream_t stream;
};

/* Workspace of the candidate lists of the min-p modes. Elements are binned by z = (max - l) * inv_t
 * in steps of 1/ZBIN_PER_NAT; min_p bounds the last bin that can hold an element of the kept
 * prefix, the exp-sum pass lists the elements up to that bin with their softmax arguments, and a
 * row-final kernel works on the list. */
constexpr int ZBINS        = 128;
constexpr int ZBIN_PER_NAT = 4;
constexpr int CAND_CAP     = 16384; /* list entries per row */
constexpr int CAND_ROW     = 2 * CAND_CAP; /* words of a row: its keys, then its ids */
constexpr int CAND_LDS     = 4096;  /* lists up to this length are staged in LDS */
constexpr int CAND_COUNT_STRIDE = 32;
/* What geist_hip_sampler_row_paths reports: the walk that has run and given the token. */
enum RowPath : int32_t {
    PATH_SHORTCUT      = 1, /* the thread maxima (or a row whose sum is NaN: no walk) */
    PATH_LIST          = 2, /* the list under the min-p bound */
    PATH_ONE_WORKGROUP = 3, /* the whole row, by one workgroup */
    PATH_SPREAD        = 4, /* the whole row, by the workgroups of its chunks */
    PATH_WINDOW        = 5, /* narrow ranges of the mass histogram (k_window) */
};
struct CandSpace {
    uint32_t *key;       /* [rows][CAND_CAP], rows CAND_ROW apart: bits of the softmax argument */
    uint32_t *idx;       /* ... vocabulary ids */
    int32_t  *count;     /* [rows * CAND_COUNT_STRIDE]: a row's counter has a cache line to itself
                          * (the appending wavefronts' atomic adds to one line serialise); behind it
                          * the word of its crowded chunks of 2048, a bit for every 8192 ids */
    int32_t  *path;      /* [rows] which walk served the row, a RowPath */
};

/* Workspace of the rows of the top-p / min-p modes that the thread-maxima shortcut does not serve
 * (sampler_window.h): per chunk a histogram of the masses and what the chunk's workgroup reports,
 * per row a record and the list of the entries around its nucleus edge and its draw. */
constexpr int WIN_SHIFT = 19;   /* a bin of the histogram spans 2^19 neighbouring binary32 p: ... */
constexpr int WIN_BINS  = 512;  /* ... 16 bins to a factor of two, down from 1 to 2^-32 */
/* List entries per row, n the sampler's longest vocabulary: an eighth of it, as both ranges may hold a
 * sixteenth of an octave in the middle of a flat row, 9000 elements each of 262144 at scale 0.5 (256 such
 * rows, top-p 0.5: with 16384 a fifth of them were walked, 969 us a call; 392 so). */
constexpr int WIN_CAP_MIN = 16384;
inline int    win_cap_for(size_t n) { return n / 8 > WIN_CAP_MIN ? (int) ((n / 8 + 255) / 256 * 256) : WIN_CAP_MIN; }
/* Launches of up to WIN_SMALL chunks of 2048, and of so many chunks' histograms read (every
 * workgroup reads all of its row's), find their plans in k_window. One row of 128256 (63 x 63) 22.5
 * us against 38 by chunks of 8192 with a row-final kernel, one of 262144 26 / 35, 16 x 128256 (16 x
 * 63 x 63 reads) 39.3 / 43.5; 8 x 262144 (8 x 128 x 128) 58 / 54, 48 x 100000 (2352 chunks) 48 / 21. */
constexpr int WIN_SMALL       = 1024;
constexpr int WIN_SMALL_READS = 65536;
/* Whether a min-p batch is cut into chunks of 2048 (n of them to a row) or of 8192: us a call, those / these.
 *   Without a soft-cap up to 1088 of them, and so many slots polled (every workgroup polls all of its
 * row's): rows that share no XCD up to 32768 -- 2 x 54912 14.1 / 16.0, 46 x 45893 (1058 chunks) 19.8 / 22.6,
 * 29 x 65528 (29696 polls) 18.4 / 18.3, but 21 x 80920 (33600) 17.9 / 17.7, 18 x 95256 (39762) 18.3 / 17.4, 22 x
 * 89112 (42592) 18.3 / 17.6 -- and rows in eights, each on one XCD, or with penalties up to 46080: 8 x 151936
 * (45000) 15.6 / 16.5, 14 x 110000 with penalties (40824) 19.6 / 22.2; beyond, the one gives and the other
 * takes: 12 x 128256 (47628) 18.1 / 17.4 and with penalties 19.1 / 20.7, 11 x 152960 (61875) 18.8 / 17.7 and
 * 19.7 / 20.4.
 *   With one, whose tanhf makes a chunk's arithmetic the longest step, up to 3400 chunks: 2 x 54912 19.2 /
 * 35.1, 52 x 131072 (3328) 44.6 / 51.6, 150 x 45000 (3300) 42.9 / 51, 64 x 128256 (4032) 54.7 / 52.4; with
 * penalties, whose registers hold seven workgroups on a compute unit for eight, up to 3072: 37 x 162840
 * (2960) 48.7 / 50.5, 48 x 130072 (3072) 48.6 / 50.4, 26 x 248856 (3172) 55.1 / 53.3, 67 x 101400 (3350) 54.4 /
 * 53.3. Long rows in eights that are not all resident at once (rows / 8 x chunks on 32 compute units, which
 * wait for the rest of their row meanwhile) keep the chunks of 8192: from 81 chunks a row on 24 x 261144
 * 58.4 / 47.7, 40 x 171032 53.9 / 51.9, 16 x 261144 43.6 / 41.0, but 40 x 158744 (78) 4 % less; with penalties
 * from 65 on 32 x 203800 66.9 / 50.8, 40 x 142360 53.9 / 49.8, 48 x 138264 57.5 / 51.7, but 48 x 121880 (60)
 * 47.9 / 50.3; 1792 chunks are resident, 16 x 195608 32.0 / 41.8, 16 x 228376 42.3 / 42.2. */
inline bool minp_small_chunks(size_t rows, size_t n, bool pen, bool capped) {
    const bool   eights = rows % 8 == 0;
    const size_t wgs    = rows * n;
    if (!capped)
        return wgs <= 1088 && wgs * n <= (eights || pen ? 46080 : 32768);
    return wgs <= (pen ? 3072 : 3400) && (!eights || n <= (pen ? 64 : 80) || wgs <= 1792);
}
struct WinSpace {
    float    *hist;  /* [rows][chunks][WIN_BINS], by the launch's chunks */
    uint64_t *list;  /* [rows][cap] */
    int       cap;
    void     *chunk; /* [rows][chunks] x WIN_CHUNK_BYTES */
    void     *row;   /* [rows] x WIN_ROW_BYTES, zero before the first use */
};
constexpr size_t WIN_CHUNK_BYTES = 32, WIN_ROW_BYTES = 128;
/* how many bins can hold an element of a kept prefix (a multiple of four) */
int win_bins_for(float top_p, float min_p, size_t n_vocab);

/* Workspace of the candidate path of the top-k modes: what each scanning wavefront hands on to
 * the row-final kernel. A row is scanned by n_chunks * 4 wavefronts; wavefront w of row r owns
 * CAND_GROUPS slots. */
constexpr int NWAVES_PER_CHUNK = 4; /* a chunk is scanned by one workgroup of four wavefronts */
constexpr int CAND_SLOTS     = 32;  /* float4 groups a wavefront has room for ... */
constexpr int CAND_GROUPS    = 32;  /* ... and how many it may hand on */
constexpr int CAND_CHUNKS_MAX = 32; /* rows of up to 32 chunks of 8192 logits take this path */
constexpr int CAND_K_MAX     = 64;  /* largest k: the survivors are ordered one per lane */
constexpr int CAND_LANES_MAX = 16;  /* largest `m` (see k_cand_scan) that leaves room in the slots */
struct WaveCands {
    float4   *val;   /* [rows][waves][CAND_SLOTS] the groups */
    int32_t  *idx;   /* [rows][waves][CAND_SLOTS] index of each group's first element, -1 = unused */
    uint32_t *bound; /* [rows][waves] key of the wavefront's bound T; 0xffffffff = it had too many
                      * groups and handed none on */
};
/* bytes of the three arrays for `row_waves` = rows * waves per row */
inline size_t wave_cands_bytes(size_t row_waves) {
    return row_waves * (CAND_SLOTS * (sizeof(float4) + sizeof(int32_t)) + 8); /* 648 */
}
inline WaveCands wave_cands_at(void *base, size_t row_waves) {
    WaveCands w;
    w.val   = static_cast<float4 *>(base);
    w.idx   = reinterpret_cast<int32_t *>(w.val + row_waves * CAND_SLOTS);
    w.bound = reinterpret_cast<uint32_t *>(w.idx + row_waves * CAND_SLOTS);
    return w;
}
/* What the wavefronts of the one-launch form of that path (k_cand_scan_final) hand on to the
 * workgroup that finishes the row: per scanning wavefront (16 per workgroup, G workgroups per row)
 * OL_SLOTS float4 groups -- those that hold an element at or above the workgroup's bound T_w --
 * with the index of each group's first element, and their number (more than OL_SLOTS: it had too
 * many and the row cannot be certified) beside the key of T_w. */
constexpr int OL_TOP      = 8;   /* maxima a wavefront enters for its workgroup's bound */
constexpr int OL_SLOTS    = 16;  /* groups a scanning wavefront may hand on */
constexpr int OL_WG_MAX   = 8;   /* workgroups per row (CAND_CHUNKS_MAX chunks, four each) */
constexpr int OL_RANK_MAX = 64;  /* largest rank `r` of the workgroup's bound the path is used for */
struct WgCands {
    float4   *val;   /* [rows][OL_SLOTS][G * 16] the float4 groups */
    uint32_t *idx;   /* [rows][OL_SLOTS][G * 16] index of each group's first element */
    uint32_t *count; /* [rows][G][16] key of T_w (its sixteen leading bits) | number of groups */
};
inline size_t wg_cands_bytes(size_t rows, size_t wgs_per_row) {
    return rows * wgs_per_row * (16 * OL_SLOTS * 20 + 16 * sizeof(uint32_t));
}
inline WgCands wg_cands_at(void *base, size_t rows, size_t wgs_per_row) {
    WgCands w;
    w.val   = static_cast<float4 *>(base);
    w.idx   = reinterpret_cast<uint32_t *>(w.val + rows * wgs_per_row * 16 * OL_SLOTS);
    w.count = w.idx + rows * wgs_per_row * 16 * OL_SLOTS;
    return w;
}
/* `r` for a workgroup that holds `elems` of a row's n_vocab logits, of which about k_eff lead:
 * the smallest rank such that the workgroup holding that many of the k_eff is a one-in-10^8 event
 * when the logits' order is unrelated to the vocabulary's (all of them when it holds the whole
 * row). 0 = the one-launch form does not pay (r would exceed OL_RANK_MAX). */
int cand_rank_for(int k_eff, size_t n_vocab, size_t elems);

/* The final stage of that path keeps its candidates (at most 16 x 64 ids) in an open-addressing
 * table of HT_SLOTS slots in LDS and looks the row's token history up in it. */
constexpr int HT_SLOTS       = 4096;

/* `m` for a row of n_vocab logits of which about k_eff lead: the smallest number of lanes such
 * that a wavefront (2048 logits) holding that many of the k_eff is a one-in-10^8 event when the
 * logits' order is unrelated to the vocabulary's. 0 = the candidate path does not pay
 * (m would exceed CAND_LANES_MAX). */
int cand_lanes_for(int k_eff, size_t n_vocab);

struct FinalLaunch {
    CandSpace       cand;
    WinSpace        win;
    int             win_bins;
    bool            win_locate;  /* a small batch: k_window finds the rows' plans itself, no row-final
                                    kernel in front */
    bool            minp_listed; /* the exp-sum pass has listed the rows under the min-p bound; the
                                    row-final kernel sends those whose list holds to its walk */
    bool            minp_direct; /* the exp-sum pass has listed the rows under the min-p bound and the
                                    list walk runs straight after it: no row-final kernel; a row
                                    whose list overflowed goes to the whole-row walk */
    int             mode, k, k_sel;
    bool            cap_after; /* top-k: the scan ran before the soft-cap, the row-final kernel
                                  applies it to what it keeps */
    float           inv_t, top_p, min_p;
    const float    *uniforms;
    uint64_t       *rng; /* launch_cand_scan_final: the rows' generators in place of uniforms, or NULL */
    const uint64_t *chunk_best;
    const double   *chunk_sum;
    const double   *slab_sum;
    const float    *tmax;
    int32_t        *out;
    int32_t        *row_flag;
};

/* The one pass over the rows of the modes that weigh every element (k_scan_expsum): tmax and
 * chunk_best as launch_tmax_scan writes them, and chunk_sum[row][chunk], the sum of
 * expf((l - max) * inv_t) over the chunk in double.
 * probe_token != NULL: the rows are n_seq * (probe_L + 1) target rows of a speculative batch and
 * probe_token holds the n_seq * probe_L draft ids; probe_p[row] receives p at the row's draft id.
 * list != NULL (min-p set): the pass also lists, per row, every element up to z bin zb_list with
 * its softmax argument -- the min-p bound needs nothing but the row maximum (the pass clears
 * list->count itself).
 * slab_sum != NULL (and no list): also the sums of the chunk's slabs of 1024 elements,
 * [rows][chunks][8], which the index-order walks locate their starting point with.
 * fast: the weights of the sums from the hardware's 2^z (relative error about 1e-7) instead of
 * the bit-exact expf; p at the probed token stays exact. Without penalties and without a list
 * the workgroups of a row then do not meet: each sums against its chunk's maximum and a second,
 * small launch scales the sums to the row's (k_rescale_sums).
 * hist != NULL (no list, no slab sums): also the chunks' histograms of the masses,
 * [rows][chunks][WIN_BINS], of which the first hist_bins bins are written.
 * Returns 0 or a hipError_t value (the launch itself is checked by the caller as usual). */
int launch_scan_expsum(const Launch &L, float inv_t, float *tmax, uint64_t *chunk_best,
                       double *chunk_sum, const int32_t *probe_token, int probe_L, float *probe_p,
                       const CandSpace *list, int zb_list, double *slab_sum, const MeetSpace &meet,
                       bool fast = false, float *hist = nullptr, int hist_bins = 0);
/* The temperature draw in one kernel (sampler_draw.h): out[row] = the id drawn with
 * uniforms[row]. For L.nv == 2. `meet.slots` holds 2 * rows * n_chunks zeroed words: the
 * workgroups of a row meet twice, the second time all of them or, with `collect`, the last chunk's
 * alone (which then also reads and advances the row's generator alone). */
/* The rows' generators, when a kernel takes its draws from them itself: states[row] is read by the
 * row's workgroups and advanced by the last of them; arrive: a zeroed counter per row, ARRIVE_STRIDE_INTS
 * apart, left zeroed. states == NULL: the draws are in `uniforms`. */
struct RowGenerators {
    uint64_t *states;
    uint32_t *arrive;
};
void launch_temperature_draw(const Launch &L, float inv_t, const float *uniforms,
                             const RowGenerators &rng, int32_t *out, const MeetSpace &meet, bool collect);
/* last z bin that can hold an entry passing min_p (with slack); ZBINS - 1 when min_p is off or
 * that deep */
int zbin_of_min_p(float min_p);

struct SpecLaunch {
    int             n_seq, L, greedy;
    float           inv_t;
    const float    *q;
    long            ld_q;
    const int32_t  *draft;
    const float    *uniforms;
    const uint64_t *chunk_best;
    const double   *chunk_sum;
    const float    *probe_p;
    double         *resid_sum;
    double         *resid_slab; /* [n_seq][chunks][8] */
    const double   *slab_sum;   /* [rows][chunks][8] from the exp-sum pass */
    void           *verdict; /* [n_seq] x SPEC_VERDICT_BYTES, written by the acceptance kernel */
    int32_t        *out_tokens;
    int32_t        *n_accepted;
};
constexpr int SLABS_MAX         = 8; /* slab sums are stored 8 per chunk whatever NV is */
constexpr int SPEC_DRAFT_MAX      = 63;
constexpr int NGRAM_SUFFIX_MAX    = 8;  /* session.c:455-456 */
constexpr int NGRAM_DRAFT_MAX     = 16; /* GEIST_SPEC_KMAX_HARDCAP, session.c:515 */
constexpr int SPEC_VERDICT_BYTES = 24;
/* meet != NULL (stochastic verification only): the residual sums and the draw in one launch (the
 * workgroups of a sequence wait for one another); NULL: two launches */
void launch_spec(const Launch &L, const SpecLaunch &sp, const MeetSpace *meet = nullptr);
/* workgroups of the one-launch kernel per compute unit, by what its registers allow: 146 with
 * chunks of 8192, 78 with chunks of 2048. Chunks of 2048, one launch / two launches:
 * 13 sequences x 1 draft x 98432 (637 workgroups) 19.8 / 21.2 us, 28 x 2 x 36992 (532) 19.6 / 21.4,
 * 20 x 1 x 90000 (900) 19.2 / 20.4, at T 0.8 0.4 to 1.2 us less. Four is also the most that
 * chunks of 2048 make of a verification on 256 compute units */
constexpr int SPEC_ONE_LAUNCH_WGS_PER_CU   = 2;
constexpr int SPEC_ONE_LAUNCH_WGS_PER_CU_2 = 4;
/* argmax of every row in one launch (sampler_greedy.h); meet: a word per (row, chunk) */
void launch_greedy(const Launch &L, int32_t *out, const MeetSpace &meet);
/* chunk_best may be NULL when only the thread maxima are wanted */
void launch_tmax_scan(const Launch &L, float *tmax, uint64_t *chunk_best,
                      int32_t *zero_per_row = nullptr);
void launch_row_final(const Launch &L, const FinalLaunch &f);
/* the candidate path of top-k (sampler_cands.h): L.nv == 8, no soft-cap, no mask, 16-byte aligned
 * rows of at most CAND_CHUNKS_MAX chunks; the scan reads the logits raw (penalties are the final
 * kernel's) and also stores the thread maxima */
void launch_cand_scan(const Launch &L, float *tmax, const WaveCands &wc, int m);
void launch_final_cand(const Launch &L, const FinalLaunch &f, const WaveCands &wc);
/* both in one launch (k_cand_scan_final): `arrive` holds one zeroed counter per row,
 * ARRIVE_STRIDE_INTS apart, and is left zeroed; `tmax` receives the thread maxima of the rows that
 * fall back to the slower paths. r_w / r_last: the rank of the bound of a full workgroup and of
 * the row's last one (cand_rank_for). far_always: read the hand-over with agent-scope loads whatever
 * the placement of the row's workgroups (for tests of that branch). */

/* *same_xcd: workgroups of a grid whose linear ids are equal modulo 8 run on one XCD (and so
 * share an L2): then launch_cand_scan_final hands a row over through that L2. Runs a small
 * kernel and waits for it. Returns a hipError_t value. */
int probe_workgroup_placement(hipStream_t stream, bool *same_xcd);
void launch_cand_scan_final(const Launch &scan, const Launch &L, const FinalLaunch &f, float *tmax,
                            const WgCands &wc, int r_w, int r_last, uint32_t *arrive,
                            bool far_always, const Notify &nt, int wgs_per_row, int groups);
/* k_topk_wide behind launch_tmax_scan(chunks of 8192, raw where the penalties can only lower a
 * logit and before the soft-cap): k and k_sel up to WIDE_K_SEL_MAX */
void launch_topk_wide(const Launch &L, const FinalLaunch &f);
/* returns a hipError_t value */
int  launch_topk_general(const Launch &L, const FinalLaunch &f);
/* Per-device kernel attributes; call once with the device current. Returns a hipError_t value. */
int configure_device_kernels();
/* what follows the exp-sum pass (minp_direct: the walk over the lists it made) or the sorted
 * row-final kernel (otherwise: rows it flagged are served by k_window); rows that neither can serve
 * take the whole-row walk, in the same launch or spread over their chunks behind it */
/* The whole-row walk spread over the workgroups of the row's chunks (sampler_walk_coop.h), for
 * the rows flagged 2 when `spread` is set: `rows` is the workspace of
 * walk_coop_bytes(max rows) bytes, zero before its first use and cleared again by this call when
 * `clear` is set; the steps of this launch are numbered from step_base + 1 on (at most 16); `hint`
 * (two words of page-locked host memory, or null): a launch in which a row was walked in full
 * writes the call's number `call` to word 0, one in which a wait ran out (the workspace then has
 * to be cleared) to word 1. */
struct WalkCoop {
    void     *rows;
    bool      spread;
    bool      behind; /* no spreading, but a launch of its own, one workgroup per row */
    bool      clear;
    uint32_t  step_base;
    uint32_t  wait_limit;
    uint32_t *hint;
    uint32_t  call;
};
size_t walk_coop_bytes(size_t rows);
void launch_candidates(const Launch &L, const FinalLaunch &f, float *probs, long ld_probs,
                       const WalkCoop &wc);
/* row_flag != NULL: only rows flagged 2 are written */
void launch_write_probs(const Launch &L, float inv_t, const uint64_t *chunk_best,
                        const double *chunk_sum, float *probs, long ld_probs,
                        const int32_t *row_flag);
/* after launch_tmax_scan(L, tmax, chunk_best): out[row][j] = log_softmax(row)[tokens[row][j]] */
void launch_logprob(const Launch &L, const uint64_t *chunk_best, double *chunk_sum,
                    const int32_t *tokens, long tokens_ld, int k_per_row, double *out, long out_ld);
void launch_ngram_draft(hipStream_t stream, const int32_t *history, long history_ld,
                        const int32_t *history_len, const int32_t *seeds, int n_seq, int k_max,
                        int max_suffix, int32_t *out, long out_ld, int32_t *out_count,
                        int32_t *out_match);
void launch_penalties(const Launch &L, float *logits_rw);
void launch_rng_units(hipStream_t stream, uint64_t *states, int shared, int rows, float *uniforms);

} // namespace gs
#endif
