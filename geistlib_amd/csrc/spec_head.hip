/*
 * spec_head.hip -- the reference's speculative output head for greedy decoding
 * (src/archs/transformer/forward/spec_head.c) over a tied F16 table in device memory, for gfx950.
 *
 * Built once per model (spec_head.c:402-607): the `sketch_dim` dimensions of the table with the
 * largest variance over a sample of rows, every row's values in those dimensions as int8 with
 * one scale per row, and two norms per row for the certainty bound.
 *
 * Per token (spec_head.c:624-889):
 *   k_spec_act        the hidden row in int8, its kept dimensions, the activation norms
 *   k_q8w_gemv        rough[r] = (float)(a . sketch[r]) * row_scale[r]: the int8 projection kernel
 *                     of the dense head. The dot is formed in binary32 there, which is exact for
 *                     sums below 2^24 (sketch_dim <= 1040), so the scores equal the reference's
 *                     integer dot bit for bit. Its epilogue leaves the maximum of every group
 *                     of 32 consecutive scores (the rows one wavefront computes).
 *   k_spec_score      the topk-th largest of those maxima: at least topk scores reach it, so
 *                     the topk best rows are among the rows >= it (about 1.2 topk rows); those
 *                     groups are read again, and the candidates' exact logits formed, one wavefront
 *                     per row, in the order of summation of f16_gemv_m1 (16 chains, fixed tree), so
 *                     that a finalist's logit is the dense head's in every bit
 *   k_spec_final      the topk best candidates (the reference's heap) and among them the best exact
 *                     logit, lowest index first
 *   k_spec_verify     (optional, GEIST_SPEC_VERIFY) the upper bound of every excluded row
 *                     against the winner; any row that could have won withdraws the answer
 *
 * Differences from the reference that cannot show in a token: sums that only feed the bound
 * (norms of rows and of the activation) are accumulated in double here and in index order in
 * binary32 there. One that can: among rough scores equal to the topk-th best the reference keeps
 * whichever rows its heap's sift order leaves, this code the lowest indices.
 */
#include "spec_head_kernels.h"

#include "lm_head_kernels.h"
#include "rmsnorm_device.h"
#include "sampler_device.h"

#include <hip/hip_fp16.h>

namespace gs {

namespace {

constexpr int SP_TPB  = 256;
constexpr int SP_WAVE = 64;

typedef uint32_t nt_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint16_t h) {
    return __half2float(__ushort_as_half(h));
}

/* Keys that order like the floats; NaN (an empty thread's maximum) sorts below everything. */
__device__ __forceinline__ uint32_t ordered_key(float f) {
    if (f != f)
        return 0u;
    const uint32_t b = __float_as_uint(f + 0.0f); /* -0 orders as +0 */
    return (b >> 31) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_to_float(uint32_t k) {
    return __uint_as_float((k >> 31) ? (k & 0x7fffffffu) : ~k);
}

/* orders the LDS traffic of one wavefront: what its lanes wrote before is what they read after */
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        v += __shfl_xor(v, d, SP_WAVE);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        v = __builtin_fmaxf(v, __shfl_xor(v, d, SP_WAVE));
    return v;
}

/* ---- build ------------------------------------------------------------------------------- */

__global__ __launch_bounds__(SP_TPB) void k_spec_dim_stats(const uint16_t *__restrict__ w,
                                                           long vocab, int d_model, long vstep,
                                                           float *__restrict__ dvar) {
    const int i = blockIdx.x * SP_TPB + threadIdx.x;
    if (i >= d_model)
        return;
    float sum = 0.0f, sq = 0.0f;
    long  vn  = 0;
    for (long r = 0; r < vocab; r += vstep, ++vn) {
        const float v = h2f(w[r * d_model + i]);
        sum           = __fadd_rn(sum, v);
        sq            = __fadd_rn(sq, __fmul_rn(v, v));
    }
    const float mean = __fdiv_rn(sum, (float) vn);
    dvar[i]          = __fsub_rn(__fdiv_rn(sq, (float) vn), __fmul_rn(mean, mean));
}

/* One wavefront per table row. */
__global__ __launch_bounds__(SP_TPB) void k_spec_sketch_rows(SpecHeadDev d) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint16_t *row  = reinterpret_cast<uint16_t *>(smem) + (size_t) wv * d.d_model;
    const long r   = (long) blockIdx.x * (SP_TPB / SP_WAVE) + wv;
    if (r >= d.vocab)
        return; /* (no workgroup barrier below) */
    const uint16_t *src = d.w + r * d.d_model;
    for (int o = lane * 8; o < d.d_model; o += SP_WAVE * 8)
        *reinterpret_cast<uint4 *>(row + o) = *reinterpret_cast<const uint4 *>(src + o);
    /* largest magnitude over the kept dimensions (spec_head.c:571-578) */
    float amax = 0.0f;
    for (int s = lane; s < d.sketch_dim; s += SP_WAVE)
        amax = __builtin_fmaxf(amax, __builtin_fabsf(h2f(row[d.dims[s]])));
    amax = __builtin_fmaxf(wave_max(amax), 1e-8f);
    const float scale = __fdiv_rn(127.0f, amax);
    int8_t     *sk    = d.sketch + r * d.sketch_dim;
    for (int s = lane; s < d.sketch_dim; s += SP_WAVE) {
        float q = __builtin_rintf(__fmul_rn(h2f(row[d.dims[s]]), scale));
        q       = __builtin_fminf(__builtin_fmaxf(q, -127.0f), 127.0f);
        sk[s]   = (int8_t) (int) q;
    }
    /* norms for the bound (spec_head.c:591-602) */
    double l1 = 0.0, sq = 0.0;
    for (int i = lane; i < d.d_model; i += SP_WAVE) {
        const double v = (double) h2f(row[i]);
        if (d.kept[i])
            l1 += fabs(v);
        else
            sq += v * v;
    }
    l1 = wave_sum(l1);
    sq = wave_sum(sq);
    if (lane == 0) {
        d.row_scale[r] = __fdiv_rn(amax, 127.0f);
        d.w_drop[r]    = (float) sqrt(sq);
        d.w_l1[r]      = (float) l1;
    }
}

/* ---- per token --------------------------------------------------------------------------- */

/* spec_head.c:672-694 and 712-724, one workgroup. With NORM the output norm of head.c:99-101
 * runs in front: h = (x * inv_rms) * norm_w, written to h_out for the finalist kernel, in the
 * arithmetic of the norm kernel of the dense head. */
template <bool NORM>
__global__ __launch_bounds__(NORM_TPB) void k_spec_act(SpecHeadDev d, const float *__restrict__ h_in,
                                                       const float *__restrict__ norm_w, float eps,
                                                       float *__restrict__ h_out) {
    __shared__ NormShared s_norm;
    __shared__ float      s_max[NORM_TPB / SP_WAVE];
    __shared__ double     s_sum[3][NORM_TPB / SP_WAVE];
    __shared__ float      s_h[SPEC_D_MODEL_MAX];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    /* the thread's first kept dimension: asked for with the row */
    const int dim0 = tid < d.sketch_dim ? d.dims[tid] : 0;
    float     v[NORM_PER], inv = 0.0f;
    if (NORM) {
        inv = block_rmsnorm(h_in, norm_w, d.d_model, eps, v, s_norm);
    } else {
#pragma unroll
        for (int k = 0; k < NORM_PER; ++k)
            v[k] = k * NORM_TPB + tid < d.d_model ? h_in[k * NORM_TPB + tid] : 0.0f;
    }
    float  amax = 0.0f;
    double all2 = 0.0;
    auto   take = [&](int i, float y) {
        s_h[i] = y;
        if (NORM)
            h_out[i] = y;
        amax = __builtin_fmaxf(amax, __builtin_fabsf(y));
        all2 += (double) y * (double) y;
    };
#pragma unroll
    for (int k = 0; k < NORM_PER; ++k)
        if (k * NORM_TPB + tid < d.d_model)
            take(k * NORM_TPB + tid, v[k]);
    for (int i = NORM_PER * NORM_TPB + tid; i < d.d_model; i += NORM_TPB)
        take(i, NORM ? __fmul_rn(__fmul_rn(h_in[i], inv), norm_w[i]) : h_in[i]);
    amax = __builtin_fmaxf(block_norm_max(amax, s_max), 1e-8f); /* (its barrier is s_h's too) */
    const float x_q = __fdiv_rn(127.0f, amax);
    double      l1 = 0.0, kept2 = 0.0;
    for (int s = tid; s < d.sketch_dim; s += NORM_TPB) {
        const float e = s_h[s == tid ? dim0 : d.dims[s]];
        float       q = __builtin_rintf(__fmul_rn(e, x_q));
        q             = __builtin_fminf(__builtin_fmaxf(q, -127.0f), 127.0f);
        d.act[s]      = q;
        l1 += fabs((double) e);
        kept2 += (double) e * (double) e;
    }
    all2  = wave_sum(all2);
    l1    = wave_sum(l1);
    kept2 = wave_sum(kept2);
    if (lane == 0)
        s_sum[0][wv] = all2, s_sum[1][wv] = l1, s_sum[2][wv] = kept2;
    __syncthreads();
    if (tid == 0) {
        double a = 0.0, b = 0.0, c = 0.0;
        for (int i = 0; i < NORM_TPB / SP_WAVE; ++i)
            a += s_sum[0][i], b += s_sum[1][i], c += s_sum[2][i];
        const double drop = a - c > 0.0 ? a - c : 0.0;
        d.sc->inv_xq      = __fdiv_rn(1.0f, x_q);
        d.sc->h_l1_kept   = (float) b;
        d.sc->h_l2_drop   = (float) sqrt(drop);
    }
}

constexpr int SP_SEL_TPB = 1024; /* the two selection kernels */
constexpr int SP_WAVES   = SP_SEL_TPB / SP_WAVE;
constexpr int SP_BINS    = 2 * SP_SEL_TPB; /* a digit of up to eleven bits */
constexpr int SP_LDS     = 150 * 1024;     /* most dynamic LDS of a launch */

struct SelectShared {
    uint32_t bins[SP_BINS];
    int      scan[SP_WAVES];
    int      digit, left;
    int      n_cand;
};

/* Inclusive sums over the workgroup in thread order, and the total: ends behind a barrier. */
__device__ __forceinline__ int select_scan(SelectShared &s, int v, int &total) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    v = wave_scan_i32_dpp(v);
    if (lane == SP_WAVE - 1)
        s.scan[wv] = v;
    __syncthreads();
    const int totals = wave_scan_i32_dpp(lane < SP_WAVES ? s.scan[lane] : 0);
    total            = (int) readlane_u32((uint32_t) totals, SP_WAVES - 1);
    return v + (wv ? (int) readlane_u32((uint32_t) totals, wv - 1) : 0);
}
/* The digit in which the `need`-th largest of the counted keys lies, and its rank among that digit's;
 * false when fewer were counted. The bins are counted and published; ends behind a barrier. */
__device__ __forceinline__ bool select_digit(SelectShared &s, int &need, uint32_t &digit) {
    const int tid = threadIdx.x;
    const int b1 = (int) s.bins[SP_BINS - 1 - 2 * tid], b0 = (int) s.bins[SP_BINS - 2 - 2 * tid];
    if (tid == 0)
        s.digit = -1;
    int       total;
    const int incl = select_scan(s, b0 + b1, total), before = incl - b0 - b1;
    if (before < need && incl >= need) {
        const bool low = before + b1 < need;
        s.digit        = SP_BINS - 1 - 2 * tid - (low ? 1 : 0);
        s.left         = need - before - (low ? b1 : 0);
    }
    __syncthreads();
    digit = (uint32_t) s.digit;
    need  = s.left;
    return s.digit >= 0;
}
__device__ __forceinline__ void clear_digits(SelectShared &s) {
    reinterpret_cast<uint2 *>(s.bins)[threadIdx.x] = make_uint2(0u, 0u);
    __syncthreads();
}

/* Phases 2 and 3 of the head (spec_head.c:728-770 and 802-826) up to the exact logits, SPEC_PARTS
 * workgroups of 1024 threads:
 *   1. the topk-th largest group maximum (group g = rows 32 g .. 32 g + 31, written by the
 *      projection's epilogue), to 16 bits: at least topk rough scores reach it, so the topk
 *      best rows are among the rows >= it. Every workgroup finds it for itself, from the same maxima.
 *   2. the groups whose maximum reaches that threshold (topk of them or a few more), dealt out to the
 *      workgroups in index order, are read again; their rows >= it are the candidates (about
 *      1.2 topk, at most 2 topk);
 *   3. the candidates' exact logits, one wavefront per row, in f16_gemv_m1's order of summation
 *      (src/backends/cpu_x86/kernel_f16_gemv.c:25-32, 40-59): sixteen chains of fused multiply-adds,
 *      element k in chain k % 16, folded as (j + j+8), (i + i+4), ((0+1) + (2+3)). Lane c < 16 runs
 *      chain c. Row and activations are laid out in LDS by chain (element k at (k % 16) * pitch +
 *      k / 16), so that a lane reads its chain's next eight weights with one 16-byte load. d_model
 *      is a multiple of 16. `rows_wg` wavefronts of the workgroup have a row's place in LDS.
 * Which of the candidates are the finalists is left to k_spec_final: the cutoff needs all of them.
 *
 * A chain of waits: maxima 1.3 us, their count 1.4, the digits 1.3, then two trips to memory and the
 * sums. One workgroup that did the first two steps took 16.3 us, 7.8 of them to fetch the 1036 groups'
 * 128 bytes each, which one compute unit's share of the memory system cannot do faster; the finalists'
 * logits took a launch of 8 us behind it. 128256 x 2560, topk 1024: the three launches behind the
 * projection 28.1 us, the two now 18.3 (this one 12.3); the step 48.1 -> 39.9, 199992 x 1536 63.8 -> 52.7,
 * 66544 x 2048 47.4 -> 40.8. */
template <int EPT>
__global__ __launch_bounds__(SP_SEL_TPB) void k_spec_score(SpecHeadDev d, const float *__restrict__ h,
                                                           int rows_wg) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ __align__(16) SelectShared s;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = d.n_groups, part = blockIdx.x;
    const int per   = d.d_model >> 4; /* elements per chain */
    const int pitch = (per + 7) & ~7;
    int      *s_ent = reinterpret_cast<int *>(smem);                   /* [slots / 32] groups */
    int32_t  *s_ci  = s_ent + ((d.slots / 32 + 3) & ~3);               /* [slots] candidate rows */
    uint32_t *s_ck  = reinterpret_cast<uint32_t *>(s_ci + d.slots);    /* ... and their keys */
    float    *s_x   = reinterpret_cast<float *>(s_ck + d.slots);       /* [16][pitch] */
    uint16_t *s_row = reinterpret_cast<uint16_t *>(s_x + 16 * pitch) + (size_t) wv * 16 * pitch;
    uint32_t  keys[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
        const int i = e * SP_SEL_TPB + tid;
        keys[e]     = i < n ? ordered_key(d.gmax[i]) : 0u;
    }
    /* the activations are asked for with the maxima and put into LDS below */
    constexpr int X_PER_THREAD = SPEC_D_MODEL_MAX / SP_SEL_TPB;
    float         xv[X_PER_THREAD];
#pragma unroll
    for (int i = 0; i < X_PER_THREAD; ++i)
        xv[i] = i * SP_SEL_TPB + tid < d.d_model ? h[i * SP_SEL_TPB + tid] : 0.0f;
    if (tid == 0)
        s.n_cand = 0;
    clear_digits(s);
    /* 1. (16 bits of the threshold are enough: it only has to be reached by at least topk maxima
     * and by few more rows than topk; the exact cutoff comes from the candidates) */
#pragma unroll
    for (int e = 0; e < EPT; ++e)
        if (keys[e]) /* (a NaN, or beyond the groups: never counted) */
            atomicAdd(&s.bins[keys[e] >> 21], 1u);
    __syncthreads();
    int      need = d.topk;
    uint32_t d1, d2, tkey = 0u;
    if (select_digit(s, need, d1)) {
        clear_digits(s);
#pragma unroll
        for (int e = 0; e < EPT; ++e)
            if (keys[e] && keys[e] >> 21 == d1)
                atomicAdd(&s.bins[keys[e] >> 16 & 31u], 1u);
        __syncthreads();
        (void) select_digit(s, need, d2);
        tkey = d1 << 21 | d2 << 16;
    }
    const float thr = key_to_float(tkey); /* (too few maxima that are numbers: NaN, nothing reaches it) */
#pragma unroll
    for (int i = 0; i < X_PER_THREAD; ++i) {
        const int k = i * SP_SEL_TPB + tid;
        if (k < d.d_model)
            s_x[(k & 15) * pitch + (k >> 4)] = xv[i];
    }
    /* 2. this workgroup's share of the groups that reach the threshold */
    int cnt = 0, n_ent;
#pragma unroll
    for (int e = 0; e < EPT; ++e)
        cnt += keys[e] >= tkey && keys[e] != 0u;
    int at = select_scan(s, cnt, n_ent) - cnt;
    if (part == 0 && tid == 0)
        d.sc->threshold = thr;
    if (n_ent > d.list_cap) { /* (uniform) more around the cutoff than the list holds */
        if (tid == 0)
            d.part_n[part] = part == 0 ? n_ent : 0;
        return;
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e)
        if (keys[e] >= tkey && keys[e] != 0u) {
            if (at % SPEC_PARTS == part)
                s_ent[at / SPEC_PARTS] = e * SP_SEL_TPB + tid;
            ++at;
        }
    __syncthreads();
    const int mine = (n_ent - part + SPEC_PARTS - 1) / SPEC_PARTS; /* groups, at most slots / 32 */
    for (int t0 = wv * SP_WAVE; t0 < mine * 8; t0 += SP_SEL_TPB) { /* (whole wavefronts) */
        const int    t    = t0 + lane;
        const int    r0   = t < mine * 8 ? s_ent[t >> 3] * 32 + 4 * (t & 7) : 0;
        const long   left = t < mine * 8 ? d.vocab - r0 : 0; /* rows of the vocabulary */
        const float4 f    = *reinterpret_cast<const float4 *>(d.rough + r0); /* (allocated in whole groups) */
        const uint32_t m  = (uint32_t) (left > 0 && f.x >= thr) | (uint32_t) (left > 1 && f.y >= thr) << 1 |
                           (uint32_t) (left > 2 && f.z >= thr) << 2 | (uint32_t) (left > 3 && f.w >= thr) << 3;
        int slot = wave_reserve(__popc(m), &s.n_cand);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (m >> c & 1u) {
                s_ci[slot] = r0 + c;
                s_ck[slot] = ordered_key(f4_get(f, c));
                ++slot;
            }
    }
    __syncthreads();
    const int n_cand = s.n_cand;
    if (tid == 0)
        d.part_n[part] = n_cand;
    /* 3. (no workgroup barrier below) */
    if (wv >= rows_wg)
        return;
    for (int c = wv; c < n_cand; c += rows_wg) {
        const uint16_t *src = d.w + (long) s_ci[c] * d.d_model;
        for (int o = lane * 8; o < d.d_model; o += SP_WAVE * 8) {
            const nt_u4 q = __builtin_nontemporal_load(reinterpret_cast<const nt_u4 *>(src + o));
            /* elements o .. o+7: chains (o & 15) .. (o & 15) + 7 at position o / 16 */
            uint16_t *dst = s_row + (o & 15) * pitch + (o >> 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                dst[(2 * i) * pitch]     = (uint16_t) (q[i] & 0xffffu);
                dst[(2 * i + 1) * pitch] = (uint16_t) (q[i] >> 16);
            }
        }
        wave_lds_order();
        float acc = 0.0f;
        if (lane < 16) {
            const uint16_t *wr = s_row + lane * pitch;
            const float    *xr = s_x + lane * pitch;
            int             p  = 0;
            for (; p + 8 <= per; p += 8) {
                const uint4  q  = *reinterpret_cast<const uint4 *>(wr + p);
                const float4 xa = *reinterpret_cast<const float4 *>(xr + p);
                const float4 xb = *reinterpret_cast<const float4 *>(xr + p + 4);
                acc = __builtin_fmaf(h2f((uint16_t) (q.x & 0xffffu)), xa.x, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.x >> 16)), xa.y, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.y & 0xffffu)), xa.z, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.y >> 16)), xa.w, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.z & 0xffffu)), xb.x, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.z >> 16)), xb.y, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.w & 0xffffu)), xb.z, acc);
                acc = __builtin_fmaf(h2f((uint16_t) (q.w >> 16)), xb.w, acc);
            }
            for (; p < per; ++p)
                acc = __builtin_fmaf(h2f(wr[p]), xr[p], acc);
        }
        wave_lds_order(); /* the next row comes to the same place */
        const float v   = __fadd_rn(acc, __shfl_down(acc, 8, SP_WAVE));
        const float q   = __fadd_rn(v, __shfl_down(v, 4, SP_WAVE));
        const float a   = __fadd_rn(q, __shfl_down(q, 1, SP_WAVE));
        const float sum = __fadd_rn(a, __shfl_down(a, 2, SP_WAVE));
        if (lane == 0)
            d.cand[(long) part * d.slots + c] =
                make_uint4(s_ck[c], (uint32_t) s_ci[c], __float_as_uint(sum), 0u);
    }
}

/* The topk-th largest candidate's rough score is the reference's cutoff (its heap's smallest entry); the
 * finalists are the candidates above it and, of those equal to it, as many as complete topk rows -- the
 * lowest indices first. The best exact logit among them, the lowest index among equals
 * (spec_head.c:827). One workgroup: four threads to a part of the candidates, whose entries are asked
 * for before their number is known (a part holds four or five; beyond sixteen a loop of its own). */
__global__ __launch_bounds__(SP_SEL_TPB) void k_spec_final(SpecHeadDev d, SpecResult *__restrict__ res) {
    extern __shared__ __align__(16) uint8_t smem[];
    uint32_t *s_ck = reinterpret_cast<uint32_t *>(smem); /* [list_cap] keys of the rough scores, */
    int32_t  *s_ci = reinterpret_cast<int32_t *>(s_ck + d.list_cap); /* rows, */
    float    *s_ex = reinterpret_cast<float *>(s_ci + d.list_cap);   /* exact logits */
    __shared__ __align__(16) SelectShared s;
    __shared__ uint64_t s_best[SP_WAVES];
    constexpr int       AHEAD = 4;
    static_assert(SP_SEL_TPB == 4 * SPEC_PARTS && 4 * AHEAD <= 32, "a part has places for a group at least");
    const int    tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint4 *mine = d.cand + (long) (tid >> 2) * d.slots;
    const int    own  = d.part_n[tid >> 2];
    uint4        ahead[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
        ahead[i] = mine[(tid & 3) + 4 * i];
    const float thr = d.sc->threshold;
    int         n_cand;
    (void) select_scan(s, (tid & 3) ? 0 : own, n_cand);
    if (tid == 0)
        s.n_cand = 0;
    if (n_cand > d.list_cap || n_cand < d.topk) { /* (uniform) none, or more around the cutoff than the
                                                   * list holds */
        if (tid == 0) {
            res->token = -1, res->answered = 0, res->n_finalists = 0, res->n_listed = n_cand;
            res->cutoff = thr, res->best_exact = 0.0f;
        }
        return;
    }
    clear_digits(s);
    const int some = (tid & 3) < own ? (own - (tid & 3) + 3) / 4 : 0;
    int       at   = wave_reserve(some, &s.n_cand);
    auto put = [&](const uint4 &c) {
        s_ck[at] = c.x;
        s_ci[at] = (int32_t) c.y;
        s_ex[at] = __uint_as_float(c.z);
        ++at;
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
        if (i < some)
            put(ahead[i]);
    for (int i = AHEAD; i < some; ++i)
        put(mine[(tid & 3) + 4 * i]);
    __syncthreads();
    uint32_t prefix = 0, digit = 0;
    int      need = d.topk;
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) { /* digits of 11, 11 and 10 bits */
        const int shift = pass == 0 ? 21 : pass == 1 ? 10 : 0, bits = pass == 2 ? 10 : 11;
        if (pass)
            clear_digits(s);
        for (int i = tid; i < n_cand; i += SP_SEL_TPB) {
            const uint32_t k = s_ck[i];
            if (pass == 0 || k >> (shift + bits) == prefix)
                atomicAdd(&s.bins[k >> shift & ((1u << bits) - 1u)], 1u);
        }
        __syncthreads();
        (void) select_digit(s, need, digit); /* (n_cand >= topk keys were counted) */
        prefix = prefix << bits | digit;
    }
    const uint32_t ckey      = prefix;
    const int      need_ties = need, tie_cnt = (int) s.bins[digit];
    uint64_t       best      = 0;
    for (int i = tid; i < n_cand; i += SP_SEL_TPB) {
        bool in = s_ck[i] >= ckey;
        if (s_ck[i] == ckey && tie_cnt > need_ties) { /* the lowest indices among the rows that tie */
            int before = 0;
            for (int j = 0; j < n_cand; ++j)
                before += (s_ci[j] < s_ci[i] && s_ck[j] == ckey) ? 1 : 0;
            in = before < need_ties;
        }
        const uint64_t p = ((uint64_t) ordered_key(s_ex[i]) << 32) | (uint32_t) (0x7fffffff - s_ci[i]);
        best             = in && p > best ? p : best;
    }
    best = wave_max_u64(best);
    if (lane == 0)
        s_best[wv] = best;
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < SP_WAVES; ++i)
            best = s_best[i] > best ? s_best[i] : best;
        res->token       = 0x7fffffff - (int32_t) (uint32_t) (best & 0xffffffffu);
        res->answered    = 1;
        res->n_finalists = d.topk;
        res->n_listed    = n_cand;
        res->cutoff      = key_to_float(ckey);
        res->best_exact  = key_to_float((uint32_t) (best >> 32));
    }
}

/* spec_head.c:846-872: a row outside the finalists whose upper bound passes the winner's exact
 * logit withdraws the answer. */
__global__ __launch_bounds__(SP_TPB) void k_spec_verify(SpecHeadDev d, SpecResult *__restrict__ res) {
    const long r = (long) blockIdx.x * SP_TPB + threadIdx.x;
    if (r >= d.vocab || res->n_finalists == 0)
        return;
    const float rough = d.rough[r];
    if (rough > res->cutoff)
        return;
    const float inv_xq = d.sc->inv_xq;
    float ub = __fmul_rn(rough, inv_xq);
    ub = __fadd_rn(ub, __fmul_rn(__fmul_rn(0.5f, d.row_scale[r]), d.sc->h_l1_kept));
    ub = __fadd_rn(ub, __fmul_rn(__fmul_rn(0.5f, d.w_l1[r]), inv_xq));
    ub = __fadd_rn(ub, __fmul_rn(d.w_drop[r], d.sc->h_l2_drop));
    if (ub > res->best_exact)
        res->answered = 0;
}

} // namespace

void launch_spec_dim_stats(hipStream_t stream, const uint16_t *w, long vocab, int d_model,
                           long vstep, float *dvar) {
    k_spec_dim_stats<<<dim3((unsigned) ((d_model + SP_TPB - 1) / SP_TPB)), dim3(SP_TPB), 0, stream>>>(
        w, vocab, d_model, vstep, dvar);
}

void launch_spec_sketch_rows(hipStream_t stream, const SpecHeadDev &d) {
    const int    rows_block = SP_TPB / SP_WAVE;
    const size_t lds        = (size_t) rows_block * d.d_model * sizeof(uint16_t);
    k_spec_sketch_rows<<<dim3((unsigned) ((d.vocab + rows_block - 1) / rows_block)), dim3(SP_TPB), lds,
                         stream>>>(d);
}

int configure_spec_kernels() {
    const void *kernels[] = {reinterpret_cast<const void *>(k_spec_score<4>),
                             reinterpret_cast<const void *>(k_spec_score<8>),
                             reinterpret_cast<const void *>(k_spec_score<SPEC_TMAX_EPT_MAX>),
                             reinterpret_cast<const void *>(k_spec_final)};
    for (const void *k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, SP_LDS);
        if (e != hipSuccess)
            return (int) e;
    }
    return 0;
}

void launch_spec_try(hipStream_t stream, const SpecHeadDev &d, const float *h, bool verify,
                     SpecResult *result, const float *norm_w, float eps, float *h_normed) {
    const dim3 one(1), block(SP_TPB), sel(SP_SEL_TPB);
    const dim3 rows((unsigned) ((d.vocab + SP_TPB - 1) / SP_TPB));
    if (norm_w != nullptr) {
        k_spec_act<true><<<one, dim3(NORM_TPB), 0, stream>>>(d, h, norm_w, eps, h_normed);
        h = h_normed;
    } else {
        k_spec_act<false><<<one, dim3(NORM_TPB), 0, stream>>>(d, h, nullptr, 0.0f, nullptr);
    }
    GemvFuse f{};
    f.gmax = d.gmax;
    launch_q8w_gemv(stream, d.sketch, d.row_scale, d.vocab, d.sketch_dim, d.act, d.sketch_dim, 1,
                    d.rough, d.vocab, &f);
    /* as many rows at a time as LDS has room for beside the activations and the candidates (twelve of
     * 5120 columns, sixteen up to 4096) */
    const size_t pitch = (size_t) (((d.d_model >> 4) + 7) & ~7);
    const size_t fixed = (size_t) ((d.slots / 32 + 3) & ~3) * 4 + (size_t) d.slots * 8 + 16 * pitch * sizeof(float);
    const size_t row   = 16 * pitch * sizeof(uint16_t), room = SP_LDS - fixed;
    const int    rows_wg = room / row < (size_t) SP_WAVES ? (int) (room / row) : SP_WAVES;
    const size_t lds_score = fixed + (size_t) rows_wg * row, lds_final = (size_t) d.list_cap * 12;
    auto score = [&](auto kernel) { kernel<<<dim3(SPEC_PARTS), sel, lds_score, stream>>>(d, h, rows_wg); };
    if (d.n_groups <= 4 * SP_SEL_TPB)
        score(k_spec_score<4>);
    else if (d.n_groups <= 8 * SP_SEL_TPB)
        score(k_spec_score<8>);
    else
        score(k_spec_score<SPEC_TMAX_EPT_MAX>);
    k_spec_final<<<one, sel, lds_final, stream>>>(d, result);
    if (verify)
        k_spec_verify<<<rows, block, 0, stream>>>(d, result);
}

} // namespace gs
