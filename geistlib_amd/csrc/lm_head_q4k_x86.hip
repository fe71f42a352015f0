/*
 * lm_head_q4k_x86.hip -- the lm_head projection of one activation row over a Q4_K table with the
 * results of the reference's x86 decode kernel q4kx8_gemv_m1
 * (src/backends/cpu_x86/kernel_q4kx8_gemm_avx512.c:47-77 the activation quantiser, :81-304 the dot
 * products of one row against eight interleaved table rows, :380-399 the sweep; reached from
 * cpu_x86_linear_q4k_m1, src/backends/cpu_x86/linear_q4k.c:163-166, for tables of a multiple of
 * 8 rows). The reference interleaves eight table rows so that eight outputs fill the lanes of a
 * vector; each output's arithmetic involves its own row alone:
 *   activations  ONE scale for the row: amax = max |x|, d_a = amax / 127 (1 when amax is 0),
 *                a = (int) (x / d_a +- 0.5) (round half away from zero), clamped to int8;
 *   per block    integers: I = sum over the eight sub-blocks j of 32 of scale_j * (sum q * a),
 *                M = sum_j min_j * (sum of a over sub-block j); binary32:
 *                acc = fmaf((float) I, d * d_a, acc), acc_min = fmaf((float) M, dmin * d_a,
 *                acc_min), the two products rounded to binary32 first;
 *   result       y = acc - acc_min.
 * The integers cannot overflow (|I| < 2^26), so their order is free; the binary32 steps are the
 * reference's, which makes the result the reference's bit for bit. Finite activations only.
 *
 * The table is read from the packed copy of geist_hip_q4k_pack (lm_head_q6k.hip): a lane owns a
 * table row; a dword holds the 4-bit values of eight consecutive elements, one mask gives the
 * even ones as bytes and a shift and a mask the odd ones, and two v_dot4_i32_i8 multiply them
 * with the activations, which the quantiser lays out to match (per eight elements a dword of the
 * even ones and a dword of the odd ones) and which are scalar operands. Four wavefronts share 64 table
 * rows' blocks for up to three activation rows; batches of four to eight go to the matrix cores
 * (k_q4k_packed_linear_x86_mfma).
 */
#include "lm_head_kernels.h"
#include "rmsnorm_device.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace gs {

constexpr int Q4X_TPB         = 256;
constexpr int Q4X_ROW_DWORDS  = 37;
constexpr int Q4X_PACK_DWORDS = Q4X_ROW_DWORDS * 64; /* the packed copy's dwords per (64 rows, block) */

/* Element t of a super-block, held by thread t modulo 256, given the reciprocal of the row's scale:
 * its int8 value into the block's dwords (ob), the sums per sub-block of 32 behind them. */
__device__ __forceinline__ void q4x_quantize_block(float xv, float inv, bool ties_even,
                                                   uint32_t *__restrict__ ob) {
    const int   t = threadIdx.x & 255;
    const float v = __fmul_rn(xv, inv);
    /* the decode kernel's quantiser rounds half away from zero by truncation and clamps; the
     * batch quantiser is lrintf (|v| <= 127 up to rounding: nothing to clamp) */
    int q = ties_even ? __float2int_rn(v)
                      : __float2int_rz(v < 0.0f ? __fsub_rn(v, 0.5f) : __fadd_rn(v, 0.5f));
    q     = q < -128 ? -128 : q > 127 ? 127 : q;
    int sum       = q;
#pragma unroll
    for (int s = 16; s >= 1; s >>= 1)
        sum += __shfl_xor(sum, s);
    const uint32_t b0 = (uint32_t) q & 0xffu;
    const uint32_t b1 = (uint32_t) __shfl_down(q, 2) & 0xffu;
    const uint32_t b2 = (uint32_t) __shfl_down(q, 4) & 0xffu;
    const uint32_t b3 = (uint32_t) __shfl_down(q, 6) & 0xffu;
    if ((t & 7) < 2) /* elements 8 k + {0, 2, 4, 6} to dword 2 k, 8 k + {1, 3, 5, 7} to 2 k + 1 */
        ob[2 * (t >> 3) + (t & 7)] = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
    if ((t & 31) == 0)
        ob[64 + (t >> 5)] = (uint32_t) sum;
}

/* One workgroup per activation row. act: per row q4k_x86_act_dwords dwords: per super-block
 * Q4X_ACT_DWORDS -- 64 of int8 (per eight elements the even ones, then the odd ones), eight
 * int32 sums per sub-block of 32 --, and behind the row's last block the scale d_a as binary32
 * (and padding that keeps the next row 32-byte aligned). ties_even: the batch quantiser
 * (quantize_q8_Kx4, q8_kx4.c:21-105) instead of the decode kernel's. */
__global__ __launch_bounds__(Q4X_TPB) void k_q8k_row_quantize(const float *__restrict__ x, long ld_x,
                                                             int nb, bool ties_even,
                                                             uint32_t *__restrict__ act) {
    __shared__ float s_max[Q4X_TPB / 64];
    const int        m = blockIdx.x, t = threadIdx.x;
    const float     *xr = x + (long) m * ld_x;
    uint32_t        *o  = act + (long) m * ((long) nb * Q4X_ACT_DWORDS + Q4X_ACT_TAIL);
    float            ax = 0.0f;
    for (int b = 0; b < nb; ++b)
        ax = __builtin_fmaxf(ax, __builtin_fabsf(xr[256 * b + t])); /* (a NaN is passed over) */
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1)
        ax = __builtin_fmaxf(ax, __shfl_xor(ax, s));
    if ((t & 63) == 0)
        s_max[t >> 6] = ax;
    __syncthreads();
    const float amax  = __builtin_fmaxf(__builtin_fmaxf(s_max[0], s_max[1]),
                                        __builtin_fmaxf(s_max[2], s_max[3]));
    const float scale = amax == 0.0f ? 1.0f : __fdiv_rn(amax, 127.0f);
    const float inv   = __fdiv_rn(1.0f, scale);
    if (t == 0)
        o[(long) nb * Q4X_ACT_DWORDS] = __float_as_uint(scale);
    for (int b = 0; b < nb; ++b)
        q4x_quantize_block(xr[256 * b + t], inv, ties_even, o + (long) b * Q4X_ACT_DWORDS);
}

/* The output norm (cpu_scalar_rmsnorm, as k_rmsnorm_rows computes it) and that quantiser in one
 * launch, one workgroup per row, four super-blocks at a time: the normed row goes to y and, as
 * int8, to act. Elements that are not held are read back by the thread that wrote them. n a
 * multiple of 256. */
__global__ __launch_bounds__(NORM_TPB) void k_rmsnorm_q8k_row_rows(const float *__restrict__ x,
                                                                  long ld_x,
                                                                  const float *__restrict__ w,
                                                                  float eps, int n,
                                                                  float *__restrict__ y, long ld_y,
                                                                  bool ties_even,
                                                                  uint32_t *__restrict__ act) {
    __shared__ NormShared s_norm;
    __shared__ float      s_max[NORM_TPB / 64];
    const int    nb = n / 256, m = blockIdx.x, t = threadIdx.x;
    const float *xr = x + (long) m * ld_x;
    float       *yr = y + (long) m * ld_y;
    uint32_t    *o  = act + (long) m * ((long) nb * Q4X_ACT_DWORDS + Q4X_ACT_TAIL);
    float        v[NORM_PER], ax = 0.0f;
    const float  rinv = block_rmsnorm(xr, w, n, eps, v, s_norm);
#pragma unroll
    for (int k = 0; k < NORM_PER; ++k) {
        if (k * NORM_TPB + t < n)
            yr[k * NORM_TPB + t] = v[k];
        ax = __builtin_fmaxf(ax, __builtin_fabsf(v[k]));
    }
    for (int i = NORM_PER * NORM_TPB + t; i < n; i += NORM_TPB) {
        const float e = __fmul_rn(__fmul_rn(xr[i], rinv), w[i]);
        yr[i]         = e;
        ax            = __builtin_fmaxf(ax, __builtin_fabsf(e));
    }
    const float amax  = block_norm_max(ax, s_max);
    const float scale = amax == 0.0f ? 1.0f : __fdiv_rn(amax, 127.0f);
    const float inv   = __fdiv_rn(1.0f, scale);
    if (t == 0)
        o[(long) nb * Q4X_ACT_DWORDS] = __float_as_uint(scale);
#pragma unroll
    for (int k = 0; k < NORM_PER; ++k)
        if (k * NORM_TPB + t < n) /* (whole blocks) */
            q4x_quantize_block(v[k], inv, ties_even,
                               o + (long) ((k * NORM_TPB + t) >> 8) * Q4X_ACT_DWORDS);
    for (int i = NORM_PER * NORM_TPB + t; i < n; i += NORM_TPB)
        q4x_quantize_block(yr[i], inv, ties_even, o + (long) (i >> 8) * Q4X_ACT_DWORDS);
}

typedef uint32_t q4x_u4 __attribute__((ext_vector_type(4)));

struct Q4xBlock {
    uint32_t q[32]; /* the 4-bit values, eight consecutive elements to a dword */
    uint32_t sc[2]; /* the eight scales as bytes */
    uint32_t mn[2]; /* the eight minima as bytes */
    uint32_t dd;    /* d (low half) and dmin, binary16 */
};
__device__ __forceinline__ void q4x_load(const uint32_t *__restrict__ base, int r, Q4xBlock &k) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const q4x_u4 t =
            __builtin_nontemporal_load(reinterpret_cast<const q4x_u4 *>(base + p * 256 + 4 * r));
        k.q[4 * p] = t.x, k.q[4 * p + 1] = t.y, k.q[4 * p + 2] = t.z, k.q[4 * p + 3] = t.w;
    }
    const q4x_u4 t =
        __builtin_nontemporal_load(reinterpret_cast<const q4x_u4 *>(base + 8 * 256 + 4 * r));
    k.sc[0] = t.x, k.sc[1] = t.y, k.mn[0] = t.z, k.mn[1] = t.w;
    k.dd    = __builtin_nontemporal_load(base + 2304 + r);
}

/* 64 table rows to a wavefront, which goes through their blocks in order; M activation rows share a pass
 * over the table (1, and 8 with PAIRS). PAIRS: the binary32 accumulators are joined once per pair of
 * sub-blocks (the reference's 16 x 16 AVX-512 tiles, kernel_q4kx8_gemm_avx512_full.c:94, 729-778) instead
 * of once per super-block. */
template <int M, bool PAIRS>
__global__ __launch_bounds__(Q4X_TPB, PAIRS && M > 2 ? 3 : 4) void k_q4k_packed_gemv_x86_rows(
    const uint32_t *__restrict__ packed, long n_out, int nb, const uint32_t *__restrict__ act,
    float *__restrict__ y, long ld_y) {
    const int  r = threadIdx.x & 63;
    const long g = (long) blockIdx.x * (Q4X_TPB / 64) + threadIdx.x / 64;
    if (g * 64 >= n_out)
        return;
    const long      row    = g * 64 + r;
    const uint32_t *base   = packed + g * nb * Q4X_PACK_DWORDS;
    const long      act_ld = (long) nb * Q4X_ACT_DWORDS + Q4X_ACT_TAIL;
    float           d_a[M], acc[M], acc_min[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        d_a[m] = __uint_as_float(act[m * act_ld + (long) nb * Q4X_ACT_DWORDS]);
        acc[m] = 0.0f, acc_min[m] = 0.0f;
    }
    /* a block ahead: the next block's loads are in flight while this one is worked on */
    Q4xBlock cur, nxt;
    q4x_load(base, r, cur);
    for (int b = 0; b < nb; ++b) {
        if (b + 1 < nb)
            q4x_load(base + (long) (b + 1) * Q4X_PACK_DWORDS, r, nxt);
        const uint32_t *a = act + (long) b * Q4X_ACT_DWORDS; /* uniform: scalar loads */
        typedef uint32_t u8v __attribute__((ext_vector_type(8)));
        const float d    = __half2float(__ushort_as_half((unsigned short) (cur.dd & 0xffffu)));
        const float dmin = __half2float(__ushort_as_half((unsigned short) (cur.dd >> 16)));
        int         iacc[M];
#pragma unroll
        for (int m = 0; m < M; ++m)
            iacc[m] = 0;
        /* With several rows the scalar loads stay near their arithmetic, four rows at a time:
         * a fence that loads may not pass and that needs the sums so far. Hoisted to the top of
         * the block they would not fit the scalar registers. */
        /* the minima against the activations' sums per sub-block: a chain of its own */
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (M > 4 && m % 4 == 0)
                asm volatile("" : "+v"(acc_min[m > 0 ? m - 1 : 0])::"memory");
            const u8v   bs = *reinterpret_cast<const u8v *>(a + m * act_ld + 64);
            const float dm = __fmul_rn(dmin, d_a[m]);
            int         im = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                im += __mul24((int) ((cur.mn[j >> 2] >> (8 * (j & 3))) & 0xffu), (int) bs[j]);
                if (PAIRS ? (j & 1) : j == 7) {
                    acc_min[m] = __builtin_fmaf((float) im, dm, acc_min[m]);
                    im         = 0;
                }
            }
        }
        /* Steps of (sub-block j, group of up to four rows). The activations of a step are
         * scalar loads issued one step ahead, before the fence that opens the step. */
        constexpr int G  = M < 4 ? M : 4;
        constexpr int NG = (M + G - 1) / G;
        u8v           avc[G], avn[G];
        uint32_t      even[4], odd[4];
        int           sc = 0;
        if (M > 1) {
#pragma unroll
            for (int i = 0; i < G; ++i)
                avc[i] = *reinterpret_cast<const u8v *>(a + i * act_ld);
        }
#pragma unroll
        for (int st = 0; st < 8 * NG; ++st) {
            const int j = st / NG, grp = st % NG; /* sub-block j: elements 32 j .. 32 j + 31 */
            if (M > 1) {
                if (st + 1 < 8 * NG) {
                    const int jn = (st + 1) / NG, gn = (st + 1) % NG;
#pragma unroll
                    for (int i = 0; i < G; ++i)
                        if (gn * G + i < M)
                            avn[i] = *reinterpret_cast<const u8v *>(a + (gn * G + i) * act_ld + 8 * jn);
                }
#pragma unroll
                for (int i = 0; i < M; ++i)
                    asm volatile("" : "+v"(iacc[i])::"memory");
            }
            if (grp == 0) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t w = cur.q[4 * j + k];
                    even[k] = w & 0x0f0f0f0fu, odd[k] = (w >> 4) & 0x0f0f0f0fu;
                }
                sc = (int) ((cur.sc[j >> 2] >> (8 * (j & 3))) & 0xffu);
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int m = grp * G + i;
                if (m >= M)
                    continue;
                const u8v av  = M > 1 ? avc[i] : *reinterpret_cast<const u8v *>(a + 8 * j);
                int       dot = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    dot = __builtin_amdgcn_sdot4((int) even[k], (int) av[2 * k], dot, false);
                    dot = __builtin_amdgcn_sdot4((int) odd[k], (int) av[2 * k + 1], dot, false);
                }
                iacc[m] += __mul24(sc, dot);
                if (PAIRS && (j & 1)) {
                    acc[m]  = __builtin_fmaf((float) iacc[m], __fmul_rn(d, d_a[m]), acc[m]);
                    iacc[m] = 0;
                }
            }
            if (M > 1) {
#pragma unroll
                for (int i = 0; i < G; ++i)
                    avc[i] = avn[i];
            }
        }
        if (!PAIRS) {
#pragma unroll
            for (int m = 0; m < M; ++m)
                acc[m] = __builtin_fmaf((float) iacc[m], __fmul_rn(d, d_a[m]), acc[m]);
        }
        if (b + 1 < nb)
            cur = nxt;
    }
    if (row < n_out) {
#pragma unroll
        for (int m = 0; m < M; ++m)
            y[m * ld_y + row] = __fsub_rn(acc[m], acc_min[m]);
    }
}

constexpr int q4x_split_dwords(int m) { return (2 * m + 1) * 64; } /* LDS per block */
constexpr int Q4X_SPLIT_BLOCKS = 32; /* of batches: what 64 KB of LDS hold of three rows */
/* One to three activation rows: the four wavefronts of a workgroup share 64 table rows and take every fourth block
 * each; the blocks' integers, exact whoever forms them, go through LDS, and the binary32 steps over the
 * blocks, which have an order, are then two chains, one to a wavefront. (With 64 table rows to a
 * wavefront, which works through their blocks one after the other, norm, projection and greedy draw of
 * 43680 x 3072 took 31.2 us, 24.2 so, 68320 x 2048 27.4 / 24.0, 150552 x 2304 46.7 / 41.8, 262144 x 1536
 * 47.4 / 45.5, 32000 x 8192 60.4 / 36.6, 256000 x 8192 194 / 191; where it loses: q4x_whole_rows.) */
template <int M>
__global__ __launch_bounds__(Q4X_TPB, 4) void k_q4k_packed_gemv_x86(
    const uint32_t *__restrict__ packed, long n_out, int nb, const uint32_t *__restrict__ act,
    float *__restrict__ y, long ld_y) {
    constexpr int W = Q4X_TPB / 64, PART = q4x_split_dwords(M);
    extern __shared__ __align__(16) uint32_t s_part[]; /* [nb]: I and M per row of the batch, the scales */
    __shared__ float s_min[M][64];
    static_assert(W % 2 == 0, "a wavefront's chains are of one kind");
    const int       r = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const long      row    = (long) blockIdx.x * 64 + r;
    const uint32_t *base   = packed + (long) blockIdx.x * nb * Q4X_PACK_DWORDS;
    const long      act_ld = (long) nb * Q4X_ACT_DWORDS + Q4X_ACT_TAIL;
    Q4xBlock        cur, nxt;
    if (wv < nb)
        q4x_load(base + (long) wv * Q4X_PACK_DWORDS, r, cur);
    for (int b = wv; b < nb; b += W) {
        if (b + W < nb)
            q4x_load(base + (long) (b + W) * Q4X_PACK_DWORDS, r, nxt);
        const uint32_t *a = act + (long) b * Q4X_ACT_DWORDS; /* uniform: scalar loads */
        typedef uint32_t u8v __attribute__((ext_vector_type(8)));
        int       im[M], iacc[M];
        u8v       bs[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            im[m] = 0, iacc[m] = 0;
            bs[m] = *reinterpret_cast<const u8v *>(a + m * act_ld + 64);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int mn = (int) ((cur.mn[j >> 2] >> (8 * (j & 3))) & 0xffu);
            const int sc = (int) ((cur.sc[j >> 2] >> (8 * (j & 3))) & 0xffu);
            uint32_t  even[4], odd[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t w = cur.q[4 * j + k];
                even[k] = w & 0x0f0f0f0fu, odd[k] = (w >> 4) & 0x0f0f0f0fu;
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                im[m] += __mul24(mn, (int) bs[m][j]);
                const u8v av  = *reinterpret_cast<const u8v *>(a + m * act_ld + 8 * j);
                int       dot = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    dot = __builtin_amdgcn_sdot4((int) even[k], (int) av[2 * k], dot, false);
                    dot = __builtin_amdgcn_sdot4((int) odd[k], (int) av[2 * k + 1], dot, false);
                }
                iacc[m] += __mul24(sc, dot);
            }
        }
        uint32_t *out = s_part + b * PART + r;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            out[(2 * m) * 64]     = __float_as_uint((float) iacc[m]);
            out[(2 * m + 1) * 64] = __float_as_uint((float) im[m]);
        }
        out[2 * M * 64] = cur.dd;
        if (b + W < nb)
            cur = nxt;
    }
    __syncthreads();
    /* chain 2 m: I and d of row m, chain 2 m + 1: M and dmin; wavefront w has chains w and w + W */
    const int kind = wv & 1;
    float     acc[(2 * M + W - 1) / W];
#pragma unroll
    for (int i = 0; i < (2 * M + W - 1) / W; ++i) {
        const int c = wv + i * W, m = c >> 1;
        acc[i] = 0.0f;
        if (c >= 2 * M)
            continue;
        const float d_a = __uint_as_float(act[m * act_ld + (long) nb * Q4X_ACT_DWORDS]);
#pragma unroll 4
        for (int b = 0; b < nb; ++b) {
            const uint32_t *in = s_part + b * PART + r;
            const uint32_t  dd = in[2 * M * 64];
            const float d = __half2float(__ushort_as_half((unsigned short) (kind ? dd >> 16 : dd & 0xffffu)));
            acc[i] = __builtin_fmaf(__uint_as_float(in[64 * c]), __fmul_rn(d, d_a), acc[i]);
        }
        if (kind)
            s_min[m][r] = acc[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (2 * M + W - 1) / W; ++i) {
        const int m = (wv + i * W) >> 1;
        if (m < M && !kind && row < n_out)
            y[m * ld_y + row] = __fsub_rn(acc[i], s_min[m][r]);
    }
}

/* The same for 2 to 8 activation rows on the int8 matrix cores. A block's scale has 6 bits and a
 * table value 4: with the scale cut into two digits of 3 bits, value x digit is at most 105, an
 * int8, and v_pk_mul_lo_u16 forms four of them at once (105 x 257 fits 16 bits: no carry from one
 * byte into the next). I = sum (q * low digit) a + 8 sum (q * high digit) a is then two
 * 16 x 16 x 64 products per 64 elements, and M, the minima spread over their sub-blocks' elements,
 * a third. The operands: activation rows (lane & 15; there are n_m, the others repeat the last and
 * are not stored) by table rows. A lane's 16 elements of K are half of what one 16-byte load of its
 * table row holds, so that lane group kg takes sub-block 4 h + kg whole, in two products, and the
 * even and odd elements stay in the order in which the activations' dwords have them.
 *
 * What bounds it: the pass over the table, 5 TB/s at 262144 x 1536 (the vector kernel's dot
 * products and their scalar operands took 3.4 at 8 rows and 4 us more per row). Quantiser and
 * projection of 8 rows, us, from HBM: 262144 x 1536 73.4 -> 56.4, 128256 x 2560 87.1 -> 47.7,
 * 32000 x 4096 114 -> 38.0. A wavefront owns 32 table rows (two tiles; 128 registers, four
 * wavefronts per SIMD): a tile's loads for the next block are issued as soon as its values are
 * cut, into the registers that those leave. Four tiles at three wavefronts took 59.0 / 48.0 /
 * 46.0, one tile at six (spilled) 81 / 69 / 43. */
typedef int            q4x_i4 __attribute__((ext_vector_type(4)));
typedef unsigned short q4x_us2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int q4x_times(uint32_t bytes, uint32_t digit2) {
    return (int) __builtin_bit_cast(uint32_t, __builtin_bit_cast(q4x_us2, bytes) *
                                                  __builtin_bit_cast(q4x_us2, digit2));
}

template <int NT, int WAVES>
__global__ __launch_bounds__(Q4X_TPB, WAVES) void k_q4k_packed_linear_x86_mfma(
    const uint32_t *__restrict__ packed, long n_out, int nb, const uint32_t *__restrict__ act,
    int n_m, float *__restrict__ y, long ld_y) {
    const int  lane = threadIdx.x & 63, j = lane & 15, kg = lane >> 4;
    const long unit = (long) blockIdx.x * (Q4X_TPB / 64) + threadIdx.x / 64;
    const long row0 = unit * (16 * NT); /* NT tiles of 16 rows, of one group of 64 */
    if (row0 >= n_out)
        return;
    const int       r0     = (int) (row0 & 63);
    const uint32_t *base   = packed + (row0 >> 6) * nb * Q4X_PACK_DWORDS;
    const long      act_ld = (long) nb * Q4X_ACT_DWORDS + Q4X_ACT_TAIL;
    const uint32_t *arow   = act + (long) (j < n_m ? j : n_m - 1) * act_ld + 8 * kg;
    /* byte kg of a dword, into the low byte of both halves / into all four bytes */
    const uint32_t sel_half = 0x0c000c00u | (uint32_t) kg * 0x00010001u;
    const uint32_t sel_all  = (uint32_t) kg * 0x01010101u;

    float d_a[4], acc[NT][4], acc_min[NT][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = 4 * kg + i;
        d_a[i] = __uint_as_float(act[(m < n_m ? m : n_m - 1) * act_ld + (long) nb * Q4X_ACT_DWORDS]);
#pragma unroll
        for (int t = 0; t < NT; ++t)
            acc[t][i] = 0.0f, acc_min[t][i] = 0.0f;
    }
    q4x_u4   q[NT][2], sm[NT]; /* values of sub-blocks kg and 4 + kg; scales, minima */
    uint32_t dd[NT];
    q4x_i4   a[2][2], an[2][2];
    auto load_tile = [&](const uint32_t *blk, int t) {
        const uint32_t *p = blk + 4 * (r0 + 16 * t + j);
        q[t][0] = __builtin_nontemporal_load(reinterpret_cast<const q4x_u4 *>(p + kg * 256));
        q[t][1] = __builtin_nontemporal_load(reinterpret_cast<const q4x_u4 *>(p + (4 + kg) * 256));
        sm[t]   = __builtin_nontemporal_load(reinterpret_cast<const q4x_u4 *>(p + 8 * 256));
        dd[t]   = __builtin_nontemporal_load(blk + 2304 + r0 + 16 * t + j);
    };
    auto load_act = [&](int b, q4x_i4 (&v)[2][2]) {
        const uint32_t *p = arow + (long) b * Q4X_ACT_DWORDS;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v[h][0] = *reinterpret_cast<const q4x_i4 *>(p + 32 * h);
            v[h][1] = *reinterpret_cast<const q4x_i4 *>(p + 32 * h + 4);
        }
    };
#pragma unroll
    for (int t = 0; t < NT; ++t)
        load_tile(base, t);
    load_act(0, a);
    for (int b = 0; b < nb; ++b) {
        /* (the last block loads itself again: no branch between the loads and their waits) */
        const int       bn   = b + 1 < nb ? b + 1 : b;
        const uint32_t *next = base + (long) bn * Q4X_PACK_DWORDS;
        load_act(bn, an);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            q4x_i4      lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0}, mi = {0, 0, 0, 0};
            const float d    = __half2float(__ushort_as_half((unsigned short) (dd[t] & 0xffffu)));
            const float dmin = __half2float(__ushort_as_half((unsigned short) (dd[t] >> 16)));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t sc = __builtin_amdgcn_perm(0u, h ? sm[t].y : sm[t].x, sel_half);
                const uint32_t sl = sc & 0x00070007u, sh = (sc >> 3) & 0x00070007u;
                const int      mn = (int) __builtin_amdgcn_perm(0u, h ? sm[t].w : sm[t].z, sel_all);
                const q4x_i4   mv = {mn, mn, mn, mn};
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint32_t w0 = k ? q[t][h].z : q[t][h].x, w1 = k ? q[t][h].w : q[t][h].y;
                    const uint32_t e0 = w0 & 0x0f0f0f0fu, o0 = (w0 >> 4) & 0x0f0f0f0fu;
                    const uint32_t e1 = w1 & 0x0f0f0f0fu, o1 = (w1 >> 4) & 0x0f0f0f0fu;
                    const q4x_i4   wl = {q4x_times(e0, sl), q4x_times(o0, sl), q4x_times(e1, sl),
                                         q4x_times(o1, sl)};
                    const q4x_i4   wh = {q4x_times(e0, sh), q4x_times(o0, sh), q4x_times(e1, sh),
                                         q4x_times(o1, sh)};
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[h][k], wl, lo, 0, 0, 0);
                    hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[h][k], wh, hi, 0, 0, 0);
                    mi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[h][k], mv, mi, 0, 0, 0);
                }
            }
            load_tile(next, t);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[t][i] = __builtin_fmaf((float) (lo[i] + 8 * hi[i]), __fmul_rn(d, d_a[i]), acc[t][i]);
                acc_min[t][i] =
                    __builtin_fmaf((float) mi[i], __fmul_rn(dmin, d_a[i]), acc_min[t][i]);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
            a[h][0] = an[h][0], a[h][1] = an[h][1];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const long row = row0 + 16 * t + j;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row < n_out && 4 * kg + i < n_m)
                y[(4 * kg + i) * ld_y + row] = __fsub_rn(acc[t][i], acc_min[t][i]);
    }
}

size_t q4k_x86_act_dwords(int n_in) {
    return (size_t) (n_in / 256) * Q4X_ACT_DWORDS + Q4X_ACT_TAIL;
}

void launch_q8k_row_quantize(hipStream_t stream, const float *x, long ld_x, int n_m, int n_in,
                             bool ties_even, uint32_t *act) {
    k_q8k_row_quantize<<<dim3(n_m), dim3(Q4X_TPB), 0, stream>>>(x, ld_x, n_in / 256, ties_even, act);
}

void launch_rmsnorm_q8k_row_rows(hipStream_t stream, const float *x, long ld_x, const float *w,
                                 float eps, int n_rows, int n, float *y, long ld_y, bool ties_even,
                                 uint32_t *act) {
    k_rmsnorm_q8k_row_rows<<<dim3(n_rows), dim3(NORM_TPB), 0, stream>>>(x, ld_x, w, eps, n, y, ld_y,
                                                                      ties_even, act);
}

/* Whether one activation row takes k_q4k_packed_gemv_x86_rows. The form that shares the blocks has a
 * workgroup per 64 table rows, four at a time on each of 256 compute units: just past 1536 (and 1792)
 * a few compute units have a seventh (eighth) to wait for, while the other form's wavefronts, two to a SIMD
 * up to 2048, run at once. Shared / not, us: 24 blocks 116500 (1821 workgroups) 75.2 / 73.9, 28 blocks 100500
 * (1571) 77.8 / 76.7, 48 blocks 100500 127.3 / 122.4, 108000 (1688) 130.5 / 128.6, 115500 (1805) 142.2 / 136.1,
 * 60 blocks 115500 173.7 / 167.5; elsewhere 24 blocks 100500 66.9 / 67.1, 20 blocks 118500 64.4 / 64.7, 36
 * blocks 98000 (1532) 91.6 / 93.7, 113000 (1766) 101.5 / 103.1, 48 blocks 128000 150.0 / 150.6, 140000 163 / 193. */
static bool q4x_whole_rows(long groups, int nb) {
    return (nb >= 22 && groups > 1792 && groups <= (nb < 28 ? 1860 : 1888)) ||
           (nb >= 28 && groups > 1536 && groups <= 1664);
}

void launch_q4k_packed_gemv_q8k(hipStream_t stream, const void *packed, long n_out, int n_in,
                                const uint32_t *act, int n_m, bool pairs, float *y, long ld_y) {
    const uint32_t *p  = static_cast<const uint32_t *>(packed);
    const int       nb = n_in / 256;
    const long      groups = (n_out + 63) / 64;
    const dim3      grid((unsigned) ((groups + 3) / 4)), block(Q4X_TPB);
    auto split = [&](auto m) {
        constexpr int M = decltype(m)::value;
        k_q4k_packed_gemv_x86<M>
            <<<dim3((unsigned) groups), block, (size_t) nb * q4x_split_dwords(M) * sizeof(uint32_t), stream>>>(
                p, n_out, nb, act, y, ld_y);
    };
    /* Up to three rows leave the matrix cores idle for the most part and the vector kernel streams at the
     * same rate or a better one: norm, projection and greedy draw, us, by it / by the matrix cores, 2 rows
     * 33000 x 1024 14.6 / 17.0, 43680 x 3072 25.2 / 28.5, 262144 x 1536 47.6 / 50.5; 3 rows 15.4 / 17.3,
     * 27.2 / 28.7, 49.3 / 51.9, 64048 x 1536 22.0 / 21.5; 4 rows 36736 x 2304 24.9 / 24.7, 124296 x 1536
     * 34.8 / 31.3. Three rows of 24 blocks and more leave room for three workgroups on a compute unit,
     * 768 on the card: what is left over waits, where the matrix cores' 512 of 128 table rows run at once
     * -- 49600 x 6144 48.2 / 46.3, 58000 x 7168 56.6 / 54.7, 65500 x 8192 67.5 / 64.5, but 49100 x 6144
     * (768) 42.1 / 46.1 and 66500 x 6144 55.4 / 61.9. pairs: a tile of sixteen rows' order of
     * accumulation, which comes in eights. */
    if (pairs)
        k_q4k_packed_gemv_x86_rows<Q4X_M_MAX, true><<<grid, block, 0, stream>>>(p, n_out, nb, act, y, ld_y);
    else if (n_m == 1 && q4x_whole_rows(groups, nb))
        k_q4k_packed_gemv_x86_rows<1, false><<<grid, block, 0, stream>>>(p, n_out, nb, act, y, ld_y);
    else if (n_m == 1) /* (at most 64 blocks: what the reference's kernel takes) */
        split(std::integral_constant<int, 1>{});
    else if (n_m == 2 && nb <= Q4X_SPLIT_BLOCKS)
        split(std::integral_constant<int, 2>{});
    else if (n_m == 3 && nb <= Q4X_SPLIT_BLOCKS && !(nb >= 24 && groups > 768 && groups <= 1024))
        split(std::integral_constant<int, 3>{});
    else
        k_q4k_packed_linear_x86_mfma<2, 4><<<dim3((unsigned) ((groups + 1) / 2)), block, 0, stream>>>(
            p, n_out, nb, act, n_m, y, ld_y);
}

} // namespace gs
