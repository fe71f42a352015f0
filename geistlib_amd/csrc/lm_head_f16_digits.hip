/*
 * lm_head_f16_digits.hip -- the portable batch projection over a binary16 table
 * (cpu_scalar_w_quant_m1 / _mN for F16 weights, src/backends/cpu_scalar/weight_resolve.c:186-241,
 * which the x86 backend also runs whenever more than one activation row is projected):
 *   y[m][j] = (float) sum_k (double) x[m][k] * (double) f16(W[j][k])   (double, index order)
 * bit for bit, on the int8 matrix cores.
 *
 * What it rests on. Every product is exact in double, so the reference's result is the exact sum,
 * plus what its n - 1 additions round away, rounded to binary32. The exact sum is an integer
 * problem: a binary16 weight is a multiple of 2^-24, an activation, scaled by its row's largest
 * magnitude, is an integer below 2^46 (but for values 2^22 times smaller than that, whose
 * remainders are bounded). Cut into signed bytes, four for a weight below 127 and six for an
 * activation, the sum is 24 int8 products, which v_mfma_i32_16x16x64_i8 adds exactly. The additions of
 * the reference err by at most n 2^-53 times the largest partial sum, which is at most ||w|| ||x||;
 * where that could carry the sum over a binary32 rounding boundary (2850 of 8 x 128256 outputs), a
 * second kernel looks closer -- the partial sums themselves are 95 times smaller on average --, and
 * what is then still open (about 30) a third one adds in index order.
 *
 * What bounds it. The pass over the table: 2 bytes per weight, 657 MB at 128256 x 2560, 104 us at
 * the rate the memory gives a stream that is read once; it takes 111 to 119. Cutting the weights
 * keeps the vector units busy half of that time (106 instructions per 64 columns and tile), the
 * matrix cores are busy a quarter; both run while the next stages' loads, four per wavefront, are
 * under way. The launches around it are the rest: 7 us for the cut, 11 and 14 for the two behind. With
 * the products in double (v_mfma_f64_4x4x4, half of whose rate eight rows could use) the same pass
 * took 200 us.
 *
 * What a call's data can cost. Rows that are not finite, sums beyond binary32 and activations of few
 * bits are settled on the way. Weight rows of a norm of 126 or more in 256 columns are left to the
 * second kernel, 1.6 us per thousand outputs of 2560 columns: a table full of them takes 8 rows of
 * 128256 1.7 ms.
 */
#include "f32_rounding.h"
#include "lm_head_kernels.h"
#include "rmsnorm_device.h"
#include "sampler_device.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gs {

namespace {

typedef int      i4v __attribute__((ext_vector_type(4)));
typedef float    f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int XD_TPB     = 512; /* threads that cut one activation row */
constexpr int XDIGITS    = 6;   /* signed bytes of an activation */
constexpr int WDIGITS    = 4;   /* ... of a weight */
constexpr int STAGE_K    = 64;  /* columns per matrix-core instruction */
constexpr int AHEAD      = 4;   /* stages whose weights are under way, per wavefront */
constexpr int LDS_STAGES = 160; /* LDS, in KiB: stages times tiles of activations it holds */

/* What the projection needs to know of a cut activation row. */
struct XRow {
    double unit; /* the value of one unit of the integer sum: 2^-24 times the activations' unit; NaN
                  * for a row that holds a NaN, and so is every output of it */
    double norm; /* ||x||, rounded up; infinite for a row that is not finite */
    double rest; /* the sum of what the cut left over of each activation, rounded up */
    double exact_to; /* products whose magnitudes add up to less add without rounding, in any order:
                      * they are multiples of 2^-24 times the largest power of two that the
                      * activations are multiples of, and this is 2^53 of that */
};
static_assert(sizeof(XRow) == F16_XROW_BYTES, "the scratch is sized by the caller");

/* Sum over a workgroup of XD_TPB threads, every thread gets it; s: XD_TPB / 64 entries that no
 * thread still reads. */
__device__ __forceinline__ double xd_block_sum(double v, double *s) {
    v = wave_sum_f64(v);
    if ((threadIdx.x & 63) == 0)
        s[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = s[0];
#pragma unroll
    for (int i = 1; i < XD_TPB / 64; ++i)
        r += s[i];
    return r;
}

/* Eight consecutive floats of a row; vec: its start is 16-byte aligned. */
__device__ __forceinline__ void xd_load8(const float *__restrict__ p, bool vec, float (&v)[8]) {
    if (vec) {
        const f4v a = *reinterpret_cast<const f4v *>(p), b = *reinterpret_cast<const f4v *>(p + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = a[i], v[4 + i] = b[i];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = p[i];
    }
}

/* One workgroup per activation row: the row (NORM: normed first, as k_rmsnorm_rows does it, and
 * written to y) cut into digits for k_f16_linear_digits, its sums and norms. A thread takes eight
 * consecutive columns at a time, the bytes one lane of the projection feeds per digit.
 *
 * Digits: the operand of tile t (of NT) of stage s holds, for lane l of a wavefront, row l % 16
 * and the sixteen columns from 64 s + 16 (l / 16) on. Row 4 g + r of tile t is digit (4 t + r) % 6
 * of activation row g + 4 ((4 t + r) / 6): the result tile then leaves all digits of an activation
 * row in one lane. */
template <bool NORM>
__global__ __launch_bounds__(XD_TPB) void k_x_digits(const float *__restrict__ x, long ld_x,
                                                     const float *__restrict__ wn, float eps, int n,
                                                     float *__restrict__ y, long ld_y, int NT,
                                                     uint8_t *__restrict__ digits, XRow *rows,
                                                     F64Lists list) {
    __shared__ double   s_d[3][XD_TPB / 64];
    __shared__ uint32_t s_u[XD_TPB / 64];
    __shared__ uint32_t s_z[XD_TPB / 64];
    __shared__ float    s_inv;
    const int    m = blockIdx.x, t = threadIdx.x;
    const float *xr = x + (long) m * ld_x;
    float       *yr = NORM ? y + (long) m * ld_y : nullptr;
    const int    n8 = n / 8, n_group = (n + STAGE_K - 1) / STAGE_K * (STAGE_K / 8);
    const bool   vx = ((uintptr_t) xr & 15) == 0;
    if (m == 0 && t == 0)
        *list.n_near = *list.n_open = 0;
    float v[8];
    if (NORM) {
        double a = 0.0;
        for (int i = t; i < n8; i += XD_TPB) {
            xd_load8(xr + 8 * i, vx, v);
#pragma unroll
            for (int q = 0; q < 8; ++q)
                a = __builtin_fma((double) v[q], (double) v[q], a); /* (exact products) */
        }
        a = xd_block_sum(a, s_d[0]);
        if (t == 0) {
            float f;
            if (!rms_inv_is_safe(a, n, eps, f))
                f = rms_inv_sequential(xr, n, eps);
            s_inv = f;
        }
        __syncthreads();
    }
    const float inv = NORM ? s_inv : 0.0f;
    double      sq  = 0.0;
    uint32_t    top = 0; /* the bits of the largest magnitude (a NaN's are larger than any) */
    for (int i = t; i < n8; i += XD_TPB) {
        xd_load8(xr + 8 * i, vx, v);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (NORM) {
                v[q]          = __fmul_rn(__fmul_rn(v[q], inv), wn[8 * i + q]);
                yr[8 * i + q] = v[q];
            }
            sq               = __builtin_fma((double) v[q], (double) v[q], sq);
            const uint32_t b = __float_as_uint(v[q]) & 0x7fffffffu;
            top              = b > top ? b : top;
        }
    }
    top = wave_max_u32(top);
    if ((t & 63) == 0)
        s_u[t >> 6] = top;
    sq = xd_block_sum(sq, s_d[1]); /* (its barrier is s_u's too) */
#pragma unroll
    for (int i = 0; i < XD_TPB / 64; ++i)
        top = s_u[i] > top ? s_u[i] : top;
    const bool finite = top < 0x7f800000u;
    /* |x| < 2^e; an activation becomes the integer nearest to x 2^(46 - e), below 2^46 */
    const long long tb = __double_as_longlong((double) __uint_as_float(top));
    const int    e = top ? (int) ((tb >> 52) & 0x7ff) - 1022 : 0;
    const double scale = __longlong_as_double((long long) (1023 + 46 - e) << 52);
    const int    g = m & 3, p0 = XDIGITS * (m >> 2);
    double       rest = 0.0;
    long long    any  = 0; /* the integers' bits */
    for (int i = t; i < n_group; i += XD_TPB) {
        uint32_t lo[XDIGITS] = {}, hi[XDIGITS] = {};
        if (i < n8 && finite) {
            if (NORM) { /* (this thread's own stores) */
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    v[q] = yr[8 * i + q];
            } else {
                xd_load8(xr + 8 * i, vx, v);
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const double f = (double) v[q] * scale;
                const double r = f + 0x1.8p52; /* the integer, in the low bits */
                rest += fabs(f - (r - 0x1.8p52));
                long long k = __double_as_longlong(r) - __double_as_longlong(0x1.8p52);
                any |= k;
#pragma unroll
                for (int d = 0; d < XDIGITS; ++d) {
                    const int b = (int) (int8_t) k;
                    k = (k - b) >> 8;
                    if (q < 4)
                        lo[d] |= ((uint32_t) b & 0xffu) << (8 * q);
                    else
                        hi[d] |= ((uint32_t) b & 0xffu) << (8 * (q - 4));
                }
            }
        }
        const int s = i >> 3, kg = (i >> 1) & 3, half = i & 1;
#pragma unroll
        for (int d = 0; d < XDIGITS; ++d) {
            const int p = p0 + d;
            uint8_t  *o = digits + ((((long) s * NT + (p >> 2)) * 64 + kg * 16 + 4 * g + (p & 3)) * 16 +
                                   8 * half);
            *reinterpret_cast<uint2 *>(o) = make_uint2(lo[d], hi[d]);
        }
    }
    /* 64 less the number of bits that are zero at the end of all integers; 0 if they are zeros */
    const uint32_t ends = wave_max_u32(any ? 64u - (uint32_t) __builtin_ctzll((unsigned long long) any) : 0u);
    if ((t & 63) == 0)
        s_z[t >> 6] = ends;
    rest = xd_block_sum(rest, s_d[2]); /* (its barrier is s_z's too) */
    if (t == 0) {
        uint32_t z = s_z[0];
        for (int i = 1; i < XD_TPB / 64; ++i)
            z = s_z[i] > z ? s_z[i] : z;
        XRow &o = rows[m];
        const double unit = __longlong_as_double((long long) (1023 - 46 + e) << 52);
        o.unit = top > 0x7f800000u ? __builtin_nan("") : unit * 0x1p-24;
        o.norm = finite ? sqrt(sq) * (1.0 + 0x1p-40) : (double) __builtin_inff();
        o.rest = rest * unit * (1.0 + 0x1p-40);
        o.exact_to = rest == 0.0 ? ldexp(unit, 53 - 24 + 64 - (int) z) : 0.0;
    }
}

/* (float) s, and whether every order of the additions leads there, err bounding what they round
 * away. Products are exact and their sums far within double's range: a sum that is not finite had
 * a product that is not, and is the same in any order. */
__device__ __forceinline__ bool order_is_free(double s, double err, float &f) {
    if (fabs(s) < __builtin_inf())
        return f32_rounding_is_safe(s, err, f);
    f = (float) s;
    return true;
}

/* v_cvt_i32_f32: towards zero, NaN to 0, what int does not hold to its ends (as a cast, undefined) */
__device__ __forceinline__ uint32_t to_int(float f) {
    uint32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(f));
    return r;
}

/* The digits of a lane's sixteen weights (eight dwords q): a weight times 2^24 is a whole number,
 * and adding 0x808080 moves the carries of the three lower signed bytes to their left neighbours, so
 * that each byte less 128 is a digit. The sum is exact in binary32 below 127: a weight of 2^-6 or
 * more has its eleven bits above the 2^7 that the constant ends on. Byte n of four weights then goes
 * to dword i of operand n. */
__device__ __forceinline__ void weight_digits(const uint32_t (&q)[8], i4v (&d)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t t[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const h2v w  = __builtin_bit_cast(h2v, q[2 * i + k]);
            t[2 * k]     = to_int(__builtin_fmaf((float) w[0], 0x1p24f, (float) 0x808080));
            t[2 * k + 1] = to_int(__builtin_fmaf((float) w[1], 0x1p24f, (float) 0x808080));
        }
        const uint32_t a01 = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u); /* bytes 0, 0, 1, 1 */
        const uint32_t a23 = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u);
        const uint32_t b01 = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u); /* bytes 2, 2, 3, 3 */
        const uint32_t b23 = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
        d[0][i] = (int) (__builtin_amdgcn_perm(a23, a01, 0x05040100u) ^ 0x80808080u);
        d[1][i] = (int) (__builtin_amdgcn_perm(a23, a01, 0x07060302u) ^ 0x80808080u);
        d[2][i] = (int) (__builtin_amdgcn_perm(b23, b01, 0x05040100u) ^ 0x80808080u);
        d[3][i] = (int) __builtin_amdgcn_perm(b23, b01, 0x07060302u);
    }
}

/* A wavefront's weights under way, as they are read: lane l gets columns 8 (l / 8) .. + 7 of a
 * stage of row l % 8 and of row 8 + l % 8, so that each load takes eight whole 128-byte lines. (A
 * load of sixteen half lines, which is what the matrix cores' operand looks like, brings this
 * stream 4.1 TB/s instead of 6.7.) */
struct Ring {
    uint32_t q[AHEAD][8];
};
struct Rows {
    const uint16_t *a, *b; /* the lane's two rows, from its columns of a stage on */
};

/* Stage s behind rows r. Not FULL: columns behind the row's end, `last` or more from r, repeat its
 * last eight (their activations are zero). */
template <bool FULL>
__device__ __forceinline__ void ring_load(const Rows &r, int s, int last, uint32_t (&q)[8]) {
    int c = s * STAGE_K;
    if (!FULL)
        c = c < last ? c : last;
    const u4v a = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(r.a + c));
    const u4v b = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(r.b + c));
#pragma unroll
    for (int i = 0; i < 4; ++i)
        q[i] = a[i], q[4 + i] = b[i];
}
/* ... as the matrix cores take them: lane l has row l % 16 and the sixteen columns from
 * 16 (l / 16) on, eight to each half of o. Lanes l and l ^ 8 swap what the other one's row is. */
__device__ __forceinline__ void ring_take(const uint32_t (&q)[8], uint32_t (&o)[8]) {
    constexpr int ROR8 = 0x128, LOW = 0x3, HIGH = 0xc; /* lanes 0..7 / 8..15 of every sixteen */
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        o[i]     = (uint32_t) __builtin_amdgcn_update_dpp((int) q[i], (int) q[4 + i], ROR8, 0xf, HIGH, false);
        o[4 + i] = (uint32_t) __builtin_amdgcn_update_dpp((int) q[4 + i], (int) q[i], ROR8, 0xf, LOW, false);
    }
}

/* One tile of 16 weight rows against the cut activations. A lane of column group kg holds the sums
 * of its weight row l % 16 and the activation rows kg, kg + 4, ... The outputs of a weight row that
 * could hold a magnitude of 127 or more go to the second kernel: one with a norm of 126 or more in
 * some turn of the ring (256 columns). */
template <int NT, int TPB, bool LDSX, bool FULL>
__device__ __forceinline__ void digits_tile(const Rows &rows, const Rows &rows_next, long row_id,
                                            long n_out, int n_in, i4v *s_x,
                                            const i4v *__restrict__ xdig, int &buf,
                                            const XRow *__restrict__ xrow, int n_m,
                                            float *__restrict__ y, long ld_y, F64Lists list,
                                            Ring &ring) {
    const int lane = threadIdx.x & 63, kg = lane >> 4, last = n_in - 8 - 8 * (lane >> 3);
    const int n_stage = (n_in + STAGE_K - 1) / STAGE_K;
    constexpr int TURN_X = AHEAD * NT * 64; /* operands of a turn of the ring */
    i4v       acc[WDIGITS][NT];
    const int j  = lane & 15;
    float     w2 = 0.0f, turn_w2 = 0.0f; /* ||w||^2 of row j of the tile, and the largest of a turn */
#pragma unroll
    for (int d = 0; d < WDIGITS; ++d)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            acc[d][t] = i4v{0, 0, 0, 0};
    for (int s0 = 0; s0 < n_stage; s0 += AHEAD) {
        /* a place of the ring that has been used is free for the stage AHEAD from there, of this
         * tile or of the next */
        const bool      over = s0 + AHEAD >= n_stage;
        const int       s1   = over ? 0 : s0 + AHEAD;
        const Rows      src  = {(over ? rows_next.a : rows.a) + s1 * STAGE_K,
                                (over ? rows_next.b : rows.b) + s1 * STAGE_K};
        /* the activations of this turn, and the next turn's on their way */
        const i4v *xd = LDSX ? s_x + s0 * NT * 64 : s_x + buf * TURN_X;
        i4v        xn[LDSX ? 1 : (TURN_X + TPB - 1) / TPB];
        f4v        nrm = {0.0f, 0.0f, 0.0f, 0.0f};
        if (!LDSX) {
#pragma unroll
            for (int i = 0; i < (TURN_X + TPB - 1) / TPB; ++i) {
                const int at = s1 * NT * 64 + (int) threadIdx.x + i * TPB;
                xn[i]        = xdig[at < n_stage * NT * 64 ? at : 0];
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (FULL || s0 + u < n_stage) {
                i4v      d[WDIGITS];
                uint32_t q[8];
                ring_take(ring.q[u], q);
                weight_digits(q, d);
                /* ||w||^2 on the diagonal of the tile times itself */
                const h8v h0 = __builtin_bit_cast(h8v, (u4v){q[0], q[1], q[2], q[3]});
                const h8v h1 = __builtin_bit_cast(h8v, (u4v){q[4], q[5], q[6], q[7]});
                nrm = __builtin_amdgcn_mfma_f32_16x16x32_f16(h0, h0, nrm, 0, 0, 0);
                nrm = __builtin_amdgcn_mfma_f32_16x16x32_f16(h1, h1, nrm, 0, 0, 0);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const i4v a = xd[(u * NT + t) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < WDIGITS; ++n)
                        acc[n][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, d[n], acc[n][t], 0, 0, 0);
                }
            }
            if (FULL || s1 + u < n_stage)
                ring_load<FULL>(src, u, last - s1 * STAGE_K, ring.q[u]);
            __builtin_amdgcn_sched_barrier(0); /* (stages mixed together would not fit the registers) */
        }
        /* the lane of column group j / 4 holds, in register j % 4, the square of row j */
        const float v0 = (j & 2) ? ((j & 1) ? nrm[3] : nrm[2]) : ((j & 1) ? nrm[1] : nrm[0]);
        w2 += v0;
        turn_w2 = __builtin_fmaxf(turn_w2, v0);
        if (!LDSX) {
            buf ^= 1;
#pragma unroll
            for (int i = 0; i < (TURN_X + TPB - 1) / TPB; ++i)
                if ((i + 1) * TPB <= TURN_X || (int) threadIdx.x + i * TPB < TURN_X)
                    s_x[buf * TURN_X + threadIdx.x + i * TPB] = xn[i];
            lds_barrier();
        }
    }
    w2      = __shfl(w2, (j >> 2) * 16 + j);
    turn_w2 = __shfl(turn_w2, (j >> 2) * 16 + j);
    const bool digits_hold = turn_w2 < 16000.0f && w2 < __builtin_inff(); /* (no NaN either) */
    /* rounded up by more than the binary32 sum's error and than what subnormal weights, were the
     * matrix cores to drop them, could add */
    const double wn = (double) __builtin_sqrtf(w2) * (1.0 + 1e-4 + (double) n_in * 0x1p-22) +
                      __builtin_sqrt((double) n_in) * 0x1p-14;
    /* (opaque from here on: the compiler would work the addresses out once, before the loop over
     * the tiles, and keep them in scratch memory) */
    int m0 = kg;
    asm volatile("" : "+v"(m0), "+s"(xrow), "+s"(y), "+s"(list.near));
#pragma unroll
    for (int r = 0; r < (4 * NT) / XDIGITS; ++r) {
        const int m = m0 + 4 * r;
        if (m >= n_m || row_id >= n_out)
            continue;
        const XRow &xr = xrow[m];
        long long   T[XDIGITS];
#pragma unroll
        for (int d = 0; d < XDIGITS; ++d) {
            const int p = XDIGITS * r + d, t = p >> 2, i = p & 3;
            T[d] = ((long long) acc[3][t][i] << 24) + ((long long) acc[2][t][i] << 16) +
                   ((long long) acc[1][t][i] << 8) + acc[0][t][i];
        }
        /* the sum of up to 96 bits in two exact halves, then in double: four roundings */
        const double hi  = (double) ((T[5] << 8) + T[4]);
        const double mid = (double) ((T[3] << 8) + T[2]);
        const double lo  = (double) ((T[1] << 8) + T[0]);
        const double sum = __builtin_fma(hi, 0x1p32, __builtin_fma(mid, 0x1p16, lo)) * xr.unit;
        const double err = (double) (n_in + 16) * 0x1p-53 * 1.01 * wn * xr.norm + 128.0 * xr.rest;
        float        f;
        if (!order_is_free(sum, err, f) || !digits_hold)
            list.near[atomicAdd(list.n_near, 1)] = make_int2((int) row_id, m);
        y[m * ld_y + row_id] = f;
        __builtin_amdgcn_sched_barrier(0);
    }
}

/* One workgroup per compute unit, its wavefronts taking tiles of 16 weight rows in turn (tile by
 * tile over the workgroups first, so that a table of any size uses every compute unit). The weights
 * come straight to the registers, four stages ahead of the arithmetic, the activations' operands from
 * LDS, which holds them all for the life of the workgroup (LDSX), and no wavefront waits for another
 * behind the one barrier. Rows too long for that (more than 5120 columns of up to 4 activation
 * rows, 3392 of up to 8, 1664 of up to 16) have theirs pass through LDS, a turn of the ring at a
 * time, in two buffers, for the wavefronts of the workgroup in step; read from the caches instead,
 * they took 240 us for 8 x 65536 x 4096 and 380 us for 16 x 128256 x 2560 (now 205 and 264). */
template <int NT, int TPB, bool LDSX, bool FULL>
__global__ __launch_bounds__(TPB) void k_f16_linear_digits(
    const uint16_t *__restrict__ w, long n_out, int n_in, const i4v *__restrict__ xdig,
    const XRow *__restrict__ xrow, int n_m, float *__restrict__ y, long ld_y, F64Lists list) {
    extern __shared__ i4v s_x[];
    const int  lane = threadIdx.x & 63;
    const int  wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long n_tile = (n_out + 15) / 16, step = (long) gridDim.x * (TPB / 64);
    long       tile   = (long) blockIdx.x + (long) wave * gridDim.x;
    const int  n_stage = (n_in + STAGE_K - 1) / STAGE_K;
    auto rows_of = [&](long t) {
        const long      r = t * 16 + (lane & 7), end = n_out - 1;
        const uint16_t *c = w + 8 * (lane >> 3);
        return Rows{c + (r < end ? r : end) * (long) n_in, c + (r + 8 < end ? r + 8 : end) * (long) n_in};
    };
    Ring ring;
    {
        const Rows r = rows_of(tile);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (FULL || u < n_stage)
                ring_load<FULL>(r, u, n_in - 8 - 8 * (lane >> 3), ring.q[u]);
    }
    for (int i = threadIdx.x; i < (LDSX ? n_stage : AHEAD < n_stage ? AHEAD : n_stage) * NT * 64; i += TPB)
        s_x[i] = xdig[i];
    __syncthreads();
    /* (in step: as many tiles for every wavefront, the last ones of some beyond the table) */
    int buf = 0;
    for (long t0 = LDSX ? tile : (long) blockIdx.x; t0 < n_tile; t0 += step, tile += step) {
        const Rows rows = rows_of(tile), next = rows_of(tile + step);
        digits_tile<NT, TPB, LDSX, FULL>(rows, next, tile * 16 + (lane & 15), n_out, n_in, s_x, xdig,
                                         buf, xrow, n_m, y, ld_y, list, ring);
    }
}

/* Every output on the list: rows longer than the integer sums hold. */
__global__ void k_f16_linear_list_all(long n_out, int n_m, F64Lists list) {
    const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_out * n_m)
        list.near[i] = make_int2((int) (i / n_m), (int) (i % n_m));
    if (i == 0)
        *list.n_near = (int) (n_out * n_m), *list.n_open = 0;
}

/* One output's products added in index order by a wavefront: its lanes form 64 products at a time and
 * every lane runs the chain. */
__device__ __forceinline__ float sum_in_order(const uint16_t *__restrict__ wr,
                                              const float *__restrict__ xm, int n_in) {
    const int lane = threadIdx.x & 63;
    double    acc  = 0.0; /* (never -0: the zeros behind the row's end change nothing) */
    for (int k0 = 0; k0 < n_in; k0 += 64) {
        const int    k = k0 + lane < n_in ? k0 + lane : 0;
        const double w = (double) (float) __builtin_bit_cast(_Float16, wr[k]);
        const uint2  p = __builtin_bit_cast(uint2, k0 + lane < n_in ? (double) xm[k] * w : 0.0);
#pragma unroll
        for (int i = 0; i < 64; ++i)
            acc += __builtin_bit_cast(double, make_uint2(readlane_u32(p.x, i), readlane_u32(p.y, i)));
    }
    return (float) acc;
}

/* A closer look at the outputs near a rounding boundary, a wavefront each. The bound that listed
 * them is cheap, not tight: it takes every partial sum for ||w|| ||x||, which is 95 times what it is
 * on average. Here the lanes add eight products each per 512 columns, a scan puts their sums
 * together, and u sum |S_k| over all partial sums S_k, which the lanes then know, bounds what the
 * reference's additions round away; of 2850 listed outputs (8 x 128256, 2560 columns) about 30
 * stay open. 14.6 MB in rows scattered over the table: five loads of a row in flight at once.
 * Activations of few bits, an int8's or a bfloat16's, put many sums right on a boundary, but their
 * additions round nothing away (XRow::exact_to): left open all the same, they made a batch of
 * integers up to 127 take 1300 us (8 x 128256 x 2560), now 213. What is open goes on a list for the
 * kernel behind this one, but of short rows, whose chain takes less than that launch, and beyond the
 * list's end: 256 outputs are two rounds of that kernel, 18 us, and a chain of 2560 additions here
 * is 30, 4096 of them side by side (every one of 16 x 20000 x 2560 open: 5800 us, with a list that holds
 * all 20300). */
constexpr int LOOK_TPB   = 256;
constexpr int LOOK_COLS  = 8 * 64; /* of a row per round of the wavefront */
constexpr int LOOK_AHEAD = 5;      /* rounds whose loads are requested together */
__global__ __launch_bounds__(LOOK_TPB) void k_f16_linear_look(const uint16_t *__restrict__ w,
                                                              int n_in, const float *__restrict__ x,
                                                              long ld_x,
                                                              const XRow *__restrict__ xrow,
                                                              float *__restrict__ y, long ld_y,
                                                              F64Lists list, int open_max) {
    const int lane = threadIdx.x & 63, count = *list.n_near;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int it = (int) blockIdx.x * (LOOK_TPB / 64) + wave; it < count;
         it += (int) gridDim.x * (LOOK_TPB / 64)) {
        const int2      mine = list.near[it];
        const uint16_t *wr = w + (long) mine.x * n_in;
        const float    *xm = x + (long) mine.y * ld_x;
        const bool      vx = ((uintptr_t) xm & 15) == 0;
        /* (a list that is full is left alone: additions to one word by the ten thousand take their
         * time. Asked for here, where nothing waits for it) */
        const int       seen = __hip_atomic_load(list.n_open, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double    exact_to = xrow ? xrow[mine.y].exact_to : 0.0;
        double          base = 0.0, own = 0.0, all = 0.0, top = 0.0;
        for (int k0 = 0; k0 < n_in; k0 += LOOK_COLS * LOOK_AHEAD) {
            h8v   h[LOOK_AHEAD];
            float v[LOOK_AHEAD][8];
#pragma unroll
            for (int g = 0; g < LOOK_AHEAD; ++g) {
                const int k = k0 + g * LOOK_COLS + 8 * lane;
                h[g]        = *reinterpret_cast<const h8v *>(wr + (k < n_in ? k : 0));
                xd_load8(xm + (k < n_in ? k : 0), vx, v[g]);
            }
#pragma unroll
            for (int g = 0; g < LOOK_AHEAD; ++g) {
                if (k0 + g * LOOK_COLS >= n_in)
                    break;
                const bool in = k0 + g * LOOK_COLS + 8 * lane < n_in;
                double     p[8], s = 0.0;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    s += in ? (double) v[g][i] * (double) (float) h[g][i] : 0.0;
                    p[i] = s;
                    own += fabs(s);
                }
                const double incl = wave_scan_f64_dpp(s), before = base + (incl - s);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    all += in ? fabs(before + p[i]) : 0.0;
                base += __shfl(incl, 63);
                top = fmax(top, fmax(fabs(base), fabs(incl)));
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            own += __shfl_xor(own, d);
            all += __shfl_xor(all, d);
            top = fmax(top, __shfl_xor(top, d));
        }
        /* own and the scans' additions (63 and one per round, of values up to twice the largest)
         * are this sum's error, all the reference's. (A product is at most the sums in front of and
         * behind it: their magnitudes add up to 2 own at most.) */
        const double rounds = (double) ((n_in + LOOK_COLS - 1) / LOOK_COLS);
        float        f;
        const bool   ok = order_is_free(
                              base, (own + all + 160.0 * rounds * top) * 0x1p-53 * (1.0 + 0x1p-20), f) ||
                          2.0 * own * (1.0 + 0x1p-30) < exact_to;
        if (!ok) { /* (uniform) */
            int at = open_max;
            if (seen < open_max && lane == 0)
                at = atomicAdd(list.n_open, 1);
            at = __builtin_amdgcn_readfirstlane(at);
            if (at < open_max) {
                if (lane == 0)
                    list.open[at] = mine;
                continue;
            }
            f = sum_in_order(wr, xm, n_in);
        }
        if (lane == 0)
            y[mine.y * ld_y + mine.x] = f;
    }
}

/* The outputs on the list in index order, as the reference adds them, a workgroup each. One chain of
 * n dependent additions is what such a sum takes (32 us for 2560 columns); here the sixteen
 * wavefronts add a sixteenth of the products each, side by side, from every value the sum can be
 * expected to have where their part begins: 128 neighbouring doubles around the parts' plain sums,
 * two to a lane. The first wavefront knows its start, so its end is known, and with it which of the
 * next one's chains was the true one. A start that is none of the 128 -- the sum had come close to
 * zero there, or the additions had rounded to one side -- has its part added once more, alone. The
 * result is the reference's chain whatever the guesses were. */
constexpr int LISTED_TPB   = 1024;
constexpr int LISTED_PARTS = LISTED_TPB / 64;
constexpr int LISTED_CAND  = 2; /* starts per lane */
constexpr int LISTED_COLS  = 4096; /* products in LDS at a time */

__global__ __launch_bounds__(LISTED_TPB) void k_f16_linear_listed(
    const uint16_t *__restrict__ w, int n_in, const float *__restrict__ x, long ld_x,
    float *__restrict__ y, long ld_y, F64Lists list) {
    __shared__ __align__(16) double s_prod[LISTED_COLS];
    __shared__ double s_end[LISTED_PARTS][64 * LISTED_CAND];
    __shared__ double s_sum[LISTED_PARTS];
    const int lane = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int count = *list.n_open < F64_OPEN_MAX ? *list.n_open : F64_OPEN_MAX;
    for (int it = blockIdx.x; it < count; it += gridDim.x) { /* (uniform over the workgroup) */
        const int2      mine = list.open[it];
        const uint16_t *wr   = w + (long) mine.x * n_in;
        const float    *xm   = x + (long) mine.y * ld_x;
        const bool      vx   = ((uintptr_t) xm & 15) == 0;
        double          sum  = 0.0; /* the reference's sum before column k0 */
        for (int k0 = 0; k0 < n_in; k0 += LISTED_COLS) {
            const int n_here = n_in - k0 < LISTED_COLS ? n_in - k0 : LISTED_COLS;
            /* a part is whole pairs of products; n_here is a multiple of eight */
            const int len = ((n_here + 2 * LISTED_PARTS - 1) / (2 * LISTED_PARTS)) * 2;
            const int b   = part * len < n_here ? part * len : n_here;
            const int e   = b + len < n_here ? b + len : n_here;
            for (int k = 8 * threadIdx.x; k < n_here; k += 8 * LISTED_TPB) {
                float v[8];
                xd_load8(xm + k0 + k, vx, v);
                const h8v h = *reinterpret_cast<const h8v *>(wr + k0 + k);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    s_prod[k + i] = (double) v[i] * (double) (float) h[i];
            }
            __syncthreads();
            double a = 0.0;
            for (int k = b + lane; k < e; k += 64)
                a += s_prod[k];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1)
                a += __shfl_xor(a, d);
            if (lane == 0)
                s_sum[part] = a;
            __syncthreads();
            double start = sum;
            for (int q = 0; q < part; ++q)
                start += s_sum[q];
            const long long at = __double_as_longlong(start);
            double          c[LISTED_CAND];
#pragma unroll
            for (int i = 0; i < LISTED_CAND; ++i)
                c[i] = __longlong_as_double(at + (LISTED_CAND * lane + i - 32 * LISTED_CAND));
            const double2 *pp = reinterpret_cast<const double2 *>(s_prod + b);
            const int      n_pair = (e - b) >> 1;
#pragma unroll 8
            for (int k = 0; k < n_pair; ++k) {
                const double2 q = pp[k];
#pragma unroll
                for (int i = 0; i < LISTED_CAND; ++i)
                    c[i] += q.x;
#pragma unroll
                for (int i = 0; i < LISTED_CAND; ++i)
                    c[i] += q.y;
            }
#pragma unroll
            for (int i = 0; i < LISTED_CAND; ++i)
                s_end[part][LISTED_CAND * lane + i] = c[i];
            __syncthreads();
            /* every thread follows the parts: the same work, and no broadcast behind it */
            double guess = sum;
            for (int q = 0; q < LISTED_PARTS; ++q) {
                const long long off = __double_as_longlong(sum) - __double_as_longlong(guess) +
                                      32 * LISTED_CAND;
                guess += s_sum[q];
                if (off >= 0 && off < 64 * LISTED_CAND) {
                    sum = s_end[q][off];
                } else {
                    const int qb = q * len < n_here ? q * len : n_here;
                    const int qe = qb + len < n_here ? qb + len : n_here;
#pragma unroll 16
                    for (int k = qb; k < qe; ++k)
                        sum += s_prod[k];
                }
            }
            __syncthreads(); /* (products and ends are read before the next are written) */
        }
        if (threadIdx.x == 0)
            y[mine.y * ld_y + mine.x] = (float) sum;
    }
}

template <int NT, int TPB>
void launch_digits(hipStream_t stream, const uint16_t *w, long n_out, int n_in, const i4v *xdig,
                   const XRow *xrow, int n_m, float *y, long ld_y, const F64Lists &list) {
    const long n_tile  = (n_out + 15) / 16;
    const dim3 grid((unsigned) (n_tile < 256 ? n_tile : 256)), block(TPB);
    const int  n_stage = (n_in + STAGE_K - 1) / STAGE_K;
    const bool full    = n_in % (AHEAD * STAGE_K) == 0;
    if (n_stage * NT > LDS_STAGES) {
        k_f16_linear_digits<NT, TPB, false, false><<<grid, block, 2 * AHEAD * NT * 1024, stream>>>(
            w, n_out, n_in, xdig, xrow, n_m, y, ld_y, list);
        return;
    }
    const size_t lds = (size_t) n_stage * NT * 1024;
    auto k = full ? k_f16_linear_digits<NT, TPB, true, true> : k_f16_linear_digits<NT, TPB, true, false>;
    /* (more than a launch gets unasked; where it is refused so is the launch, which the caller sees) */
    if (lds > 64 * 1024)
        (void) hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, LDS_STAGES * 1024);
    k<<<grid, block, lds, stream>>>(w, n_out, n_in, xdig, xrow, n_m, y, ld_y, list);
}

/* The activation rows' operands: tiles of 16 digit rows per stage. Four rows of activations per
 * lane group of the result at most, six digits each. */
int digit_tiles(int n_m) { return n_m <= 4 ? 2 : n_m <= 8 ? 3 : 6; }

} // namespace

size_t f16_linear_act_bytes(int n_in) {
    return ((size_t) (n_in + STAGE_K - 1) / STAGE_K) * 6 * 1024 + F64_M_MAX * sizeof(XRow);
}

static void f16_linear_pass(hipStream_t stream, const uint16_t *w_f16, long n_out, int n_in,
                            const float *x, long ld_x, int n_m, const F64Scratch &ws, float *y,
                            long ld_y) {
    const XRow *xrow = static_cast<const XRow *>(ws.act);
    const i4v  *xdig = reinterpret_cast<const i4v *>(xrow + F64_M_MAX);
    if (n_in > F16_DIGITS_MAX_IN)
        k_f16_linear_list_all<<<dim3((unsigned) ((n_out * n_m + 255) / 256)), dim3(256), 0, stream>>>(
            n_out, n_m, ws.list);
    else if (n_m <= 4)
        launch_digits<2, 768>(stream, w_f16, n_out, n_in, xdig, xrow, n_m, y, ld_y, ws.list);
    else if (n_m <= 8)
        launch_digits<3, 768>(stream, w_f16, n_out, n_in, xdig, xrow, n_m, y, ld_y, ws.list);
    else
        launch_digits<6, 512>(stream, w_f16, n_out, n_in, xdig, xrow, n_m, y, ld_y, ws.list);
    /* A wavefront's chain of 512 additions takes 6 us, a launch 4 and the parts 2 at least: rows of up
     * to 512 columns are done with the closer look (16 x 64, 2 rows, called from Python: 12.5 us, with
     * the third kernel 15.6). */
    const int open_max = n_in <= 512 ? 0 : F64_OPEN_MAX;
    k_f16_linear_look<<<dim3(1024), dim3(LOOK_TPB), 0, stream>>>(
        w_f16, n_in, x, ld_x, n_in > F16_DIGITS_MAX_IN ? nullptr : xrow, y, ld_y, ws.list, open_max);
    if (open_max == 0)
        return;
    k_f16_linear_listed<<<dim3(128), dim3(LISTED_TPB), 0, stream>>>(w_f16, n_in, x, ld_x, y, ld_y, ws.list);
}

void launch_f16_linear_f64(hipStream_t stream, const uint16_t *w_f16, long n_out, int n_in,
                           const float *x, long ld_x, int n_m, const F64Scratch &ws, float *y,
                           long ld_y) {
    XRow    *xrow = static_cast<XRow *>(ws.act);
    uint8_t *xdig = reinterpret_cast<uint8_t *>(xrow + F64_M_MAX);
    if (n_in <= F16_DIGITS_MAX_IN)
        k_x_digits<false><<<dim3(n_m), dim3(XD_TPB), 0, stream>>>(x, ld_x, nullptr, 0.0f, n_in, nullptr,
                                                                 0, digit_tiles(n_m), xdig, xrow,
                                                                 ws.list);
    f16_linear_pass(stream, w_f16, n_out, n_in, x, ld_x, n_m, ws, y, ld_y);
}

void launch_rmsnorm_f16_linear_f64(hipStream_t stream, const float *h, long ld_h, const float *wn,
                                   float eps, float *normed, long ld_n, const uint16_t *w_f16,
                                   long n_out, int n_in, int n_m, const F64Scratch &ws, float *y,
                                   long ld_y) {
    XRow    *xrow = static_cast<XRow *>(ws.act);
    uint8_t *xdig = reinterpret_cast<uint8_t *>(xrow + F64_M_MAX);
    if (n_in <= F16_DIGITS_MAX_IN)
        k_x_digits<true><<<dim3(n_m), dim3(XD_TPB), 0, stream>>>(h, ld_h, wn, eps, n_in, normed, ld_n,
                                                                digit_tiles(n_m), xdig, xrow,
                                                                ws.list);
    else
        launch_rmsnorm_rows(stream, h, ld_h, wn, eps, n_m, n_in, normed, ld_n);
    f16_linear_pass(stream, w_f16, n_out, n_in, normed, ld_n, n_m, ws, y, ld_y);
}

} // namespace gs
