/*
 * lm_head.hip -- the two steps between the last transformer layer and the sampler
 * (src/archs/transformer/forward/head.c:94-129 of the reference), for gfx950:
 *
 *   k_rmsnorm_rows   cpu_scalar_rmsnorm               src/backends/cpu_scalar/elementwise.c:241-280
 *   k_f16_gemv       f16_gemv_m1 (tied F16 lm_head)   src/backends/cpu_x86/kernel_f16_gemv.c:34-64
 *
 * Both reproduce the reference's results bit for bit, which fixes the order of every sum.
 *
 * k_f16_gemv. The reference adds the products of a row in sixteen chains of fused multiply-adds
 * (two 8-lane AVX accumulators: element k belongs to chain k % 16 and is added at step k / 16),
 * then folds the chains in a fixed tree. A chain is sequential, so one lane owns eight chains of
 * one weight row -- the 16 bytes it needs per step are exactly one accumulator's 8 weights --
 * and two neighbouring lanes own a row. A wavefront therefore works on 32 rows at a time, and
 * reading 16 bytes per lane straight from those rows would touch 32 different lines per load.
 * Instead the wavefront streams the rows through a private LDS tile: it loads 128 bytes of each
 * of its 32 rows with fully coalesced 16-byte loads (8 lanes per row), two stages ahead in
 * registers, writes them to the tile (row pitch 144 bytes against bank conflicts), and each lane
 * reads its own 16 bytes per step back. No workgroup barrier is involved: the tile belongs to
 * one wavefront, whose LDS operations execute in order. The activations of the stage take the
 * same way (they come from L2). The kernel is bound by the one pass over the weights: 2 bytes
 * per multiply-add for one activation row, 2 / n_m bytes with n_m rows, whose accumulators
 * (8 per row and lane) share each converted weight.
 */
#include "lm_head_kernels.h"
#include "rmsnorm_device.h"

#include <hip/hip_fp16.h>

namespace gs {

namespace {

constexpr int LM_TPB       = 256;
constexpr int LM_WAVE      = 64;
constexpr int LM_WAVES     = LM_TPB / LM_WAVE;
constexpr int ROWS_WAVE    = 32;                   /* two lanes per weight row */
constexpr int ROWS_BLOCK   = ROWS_WAVE * LM_WAVES; /* 128 */
constexpr int STAGE_BYTES  = 128;                  /* of a row per stage */
constexpr int STAGE_COLS   = 64;                   /* ... which is 64 binary16 weights */
constexpr int STAGE_LOADS  = 4;                    /* 32 rows x 8 segments / 64 lanes */
constexpr int TILE_PITCH   = STAGE_BYTES + 16;     /* bytes */
constexpr int TILE_BYTES   = ROWS_WAVE * TILE_PITCH;
/* EB = bytes per weight: 2 (binary16) or 1 (int8 with a scale per row). A stage then holds
 * 128 / EB columns, 8 / EB steps of 16, and each lane stages 2 / EB activations per row. */
template <int EB>
struct Geom {
    static constexpr int COLS  = STAGE_BYTES / EB;
    static constexpr int STEPS = COLS / 16;
    static constexpr int XL    = COLS / LM_WAVE;
};

__device__ __forceinline__ float dadd(float a, float b) { return __fadd_rn(a, b); }

/* The weights of one stage for this lane: segment (lane & 7) of rows 8 i + (lane >> 3). */
struct StageRegs {
    uint4 w[STAGE_LOADS];
};

template <int MT, int XL>
struct StageX {
    float x[MT][XL];
};

/* Which weight row a wavefront's virtual row r (0..31) is. Plain: 32 consecutive rows per
 * wavefront task. Sampler layout: task (chunk, t) is thread t of chunk `chunk` of the sampler's
 * top-k scan (chunks of 8192 logits, thread t owns the float4 groups 4 * (j * 256 + t), j < 8),
 * so that the maximum over the task's 32 results is that thread's maximum. */
template <bool SL>
__device__ __forceinline__ long virtual_row(long task, int r) {
    if (!SL)
        return task * ROWS_WAVE + r;
    const long chunk = task >> 8, t = task & 255;
    return chunk * 8192 + 4 * ((long) (r >> 2) * 256 + t) + (r & 3);
}

template <int EB, bool SL>
__device__ __forceinline__ void stage_load(const uint8_t *__restrict__ w, long task, long n_out,
                                           int n_in, int stage, int lane, StageRegs &g) {
    const int seg = lane & 7;
    const int col = stage * Geom<EB>::COLS + seg * (16 / EB);
#pragma unroll
    for (int i = 0; i < STAGE_LOADS; ++i) {
        const long row = virtual_row<SL>(task, 8 * i + (lane >> 3));
        g.w[i]         = make_uint4(0u, 0u, 0u, 0u);
        if (row < n_out && col < n_in) {
            /* read once, and far more than the caches hold: non-temporal */
            typedef uint32_t nt_u4 __attribute__((ext_vector_type(4)));
            const nt_u4 t = __builtin_nontemporal_load(
                reinterpret_cast<const nt_u4 *>(w + (row * n_in + col) * EB));
            g.w[i] = make_uint4(t.x, t.y, t.z, t.w);
        }
    }
}

template <int EB, int MT>
__device__ __forceinline__ void stage_load_x(const float *__restrict__ x, long ld_x, int n_m,
                                             int n_in, int stage, int lane,
                                             StageX<MT, Geom<EB>::XL> &gx) {
#pragma unroll
    for (int q = 0; q < Geom<EB>::XL; ++q) {
        const int col = stage * Geom<EB>::COLS + q * LM_WAVE + lane;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int mm = m < n_m ? m : n_m - 1; /* rows beyond n_m repeat the last, unstored */
            gx.x[m][q]   = col < n_in ? x[mm * ld_x + col] : 0.0f;
        }
    }
}

/* One step of the chains: eight weights of this lane's row and half against the activations of
 * the same columns. MASKED: lanes with keep == false leave their chains alone. */
template <int EB, int MT, bool MASKED>
__device__ __forceinline__ void gemv_step(const uint8_t *tile, const float (*xs)[Geom<EB>::COLS],
                                          int my_row, int half, int t, bool keep,
                                          float (&acc)[MT][8]) {
    float wf[8];
    if (EB == 2) {
        const uint4 q =
            *reinterpret_cast<const uint4 *>(tile + my_row * TILE_PITCH + t * 32 + half * 16);
        const float2 f01 = __half22float2(*reinterpret_cast<const __half2 *>(&q.x));
        const float2 f23 = __half22float2(*reinterpret_cast<const __half2 *>(&q.y));
        const float2 f45 = __half22float2(*reinterpret_cast<const __half2 *>(&q.z));
        const float2 f67 = __half22float2(*reinterpret_cast<const __half2 *>(&q.w));
        wf[0] = f01.x, wf[1] = f01.y, wf[2] = f23.x, wf[3] = f23.y;
        wf[4] = f45.x, wf[5] = f45.y, wf[6] = f67.x, wf[7] = f67.y;
    } else {
        const uint2 q =
            *reinterpret_cast<const uint2 *>(tile + my_row * TILE_PITCH + t * 16 + half * 8);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wf[i]     = (float) (int) (int8_t) (q.x >> (8 * i));
            wf[4 + i] = (float) (int) (int8_t) (q.y >> (8 * i));
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const float4 xa = *reinterpret_cast<const float4 *>(&xs[m][t * 16 + half * 8]);
        const float4 xb = *reinterpret_cast<const float4 *>(&xs[m][t * 16 + half * 8 + 4]);
        const float  xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float f = __builtin_fmaf(wf[i], xv[i], acc[m][i]);
            acc[m][i]     = (!MASKED || keep) ? f : acc[m][i];
        }
    }
}

/* The work of one workgroup; `scales` != NULL (int8 weights): y = sum * scales[row]. */
template <int EB, int MT, bool SL>
__device__ __forceinline__ void gemv_body(const uint8_t *__restrict__ w,
                                          const float *__restrict__ scales, long n_out, int n_in,
                                          const float *__restrict__ x, long ld_x, int n_m,
                                          float *__restrict__ y, long ld_y, const GemvFuse &fuse) {
    constexpr int COLS = Geom<EB>::COLS, STEPS = Geom<EB>::STEPS, XL = Geom<EB>::XL;
    __shared__ __align__(16) uint8_t s_tile[LM_WAVES][TILE_BYTES];
    __shared__ __align__(16) float   s_x[LM_WAVES][MT][COLS];
    const int  lane = threadIdx.x & (LM_WAVE - 1), wave = threadIdx.x / LM_WAVE;
    const long task = (long) blockIdx.x * LM_WAVES + wave;
    if (virtual_row<SL>(task, 0) >= n_out) { /* (no workgroup barrier below) */
        if (SL && lane < n_m && task < (long) fuse.n_chunks * 256)
            fuse.tmax[((long) lane * fuse.n_chunks + (task >> 8)) * 256 + (task & 255)] =
                __builtin_nanf(""); /* a scanning thread without an element is never chosen */
        return;
    }
    uint8_t *tile = s_tile[wave];
    float(*xs)[COLS] = s_x[wave];
    const int my_row = lane >> 1, half = lane & 1;

    float acc[MT][8];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            acc[m][i] = 0.0f;

    const int n_stage = (n_in + COLS - 1) / COLS;
    StageRegs      g0, g1;
    StageX<MT, XL> x0, x1;
    stage_load<EB, SL>(w, task, n_out, n_in, 0, lane, g0);
    if (n_stage > 1)
        stage_load<EB, SL>(w, task, n_out, n_in, 1, lane, g1);
    stage_load_x<EB, MT>(x, ld_x, n_m, n_in, 0, lane, x0);
    if (n_stage > 1)
        stage_load_x<EB, MT>(x, ld_x, n_m, n_in, 1, lane, x1);
    /* One stage: registers -> tile (this waits for the loads issued two stages ago), the same
     * registers are reloaded with the stage after next, then the steps. Two register sets take
     * turns, so nothing is copied. */
    auto do_stage = [&](int s, StageRegs &g, StageX<MT, XL> &gx) {
#pragma unroll
        for (int i = 0; i < STAGE_LOADS; ++i)
            *reinterpret_cast<uint4 *>(tile + (8 * i + (lane >> 3)) * TILE_PITCH + (lane & 7) * 16) =
                g.w[i];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int q = 0; q < XL; ++q)
                xs[m][q * LM_WAVE + lane] = gx.x[m][q];
        if (s + 2 < n_stage) {
            stage_load<EB, SL>(w, task, n_out, n_in, s + 2, lane, g);
            stage_load_x<EB, MT>(x, ld_x, n_m, n_in, s + 2, lane, gx);
        }
        /* steps of this stage: whole blocks of 16 columns, and at the end of the row possibly
         * a block of 8, which only extends chains 0..7 (the lanes with half == 0) */
        const int left = n_in - s * COLS;
        if (left >= COLS) {
#pragma unroll
            for (int t = 0; t < STEPS; ++t)
                gemv_step<EB, MT, false>(tile, xs, my_row, half, t, true, acc);
        } else {
            const int  full  = left / 16;
            const bool tail8 = (left & 15) == 8;
            for (int t = 0; t < full; ++t)
                gemv_step<EB, MT, false>(tile, xs, my_row, half, t, true, acc);
            if (tail8)
                gemv_step<EB, MT, true>(tile, xs, my_row, half, full, half == 0, acc);
        }
    };
    for (int s = 0; s < n_stage; s += 2) {
        do_stage(s, g0, x0);
        if (s + 1 < n_stage)
            do_stage(s + 1, g1, x1);
    }
    /* (chain j + chain j+8), (lane i + lane i+4), ((0+1) + (2+3)): kernel_f16_gemv.c:25-32, 59 */
    const long row = virtual_row<SL>(task, my_row);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = dadd(acc[m][i], __shfl_xor(acc[m][i], 1, LM_WAVE));
        const float q0 = dadd(v[0], v[4]), q1 = dadd(v[1], v[5]);
        const float q2 = dadd(v[2], v[6]), q3 = dadd(v[3], v[7]);
        float sum = dadd(dadd(q0, q1), dadd(q2, q3));
        if (EB == 1) /* q8w_gemv_m1: y[r] = s * scales[r], kernel_f16_gemv.c:125 */
            sum = __fmul_rn(sum, row < n_out ? scales[row] : 0.0f);
        if (half == 0 && row < n_out && m < n_m)
            y[m * ld_y + row] = sum;
        if (SL) {
            /* the scanning thread's maximum over its elements of the row (NaN ignored, as the
             * scan's v_max3_f32 does) */
            float mx = row < n_out ? sum : -__builtin_inff();
#pragma unroll
            for (int d = 1; d < LM_WAVE; d <<= 1)
                mx = __builtin_fmaxf(mx, __shfl_xor(mx, d, LM_WAVE));
            if (lane == 0 && m < n_m)
                fuse.tmax[((long) m * fuse.n_chunks + (task >> 8)) * 256 + (task & 255)] = mx;
        } else if (fuse.gmax != nullptr && m == 0) { /* (uniform) */
            float mx = row < n_out ? sum : -__builtin_inff();
#pragma unroll
            for (int d = 1; d < LM_WAVE; d <<= 1)
                mx = __builtin_fmaxf(mx, __shfl_xor(mx, d, LM_WAVE));
            if (lane == 0)
                fuse.gmax[task] = mx;
        }
    }
}

} // namespace

template <int MT, bool SL>
__global__ __launch_bounds__(LM_TPB) void k_f16_gemv(const uint16_t *__restrict__ w, long n_out,
                                                     int n_in, const float *__restrict__ x,
                                                     long ld_x, int n_m, float *__restrict__ y,
                                                     long ld_y, GemvFuse fuse) {
    gemv_body<2, MT, SL>(reinterpret_cast<const uint8_t *>(w), nullptr, n_out, n_in, x, ld_x, n_m,
                         y, ld_y, fuse);
}

/* q8w_gemv_m1 (kernel_f16_gemv.c:95-127): the same chains over int8 weights, times the row's
 * scale. Half the bytes per weight, so twice the columns per stage. One and two activation rows; more
 * go to the matrix cores (k_q8w_gemv_mfma: two rows 65 us there, 58 here, for 128256 x 2560). */
template <int MT, bool SL>
__global__ __launch_bounds__(LM_TPB) void k_q8w_gemv(const int8_t *__restrict__ wq,
                                                     const float *__restrict__ scales, long n_out,
                                                     int n_in, const float *__restrict__ x,
                                                     long ld_x, int n_m, float *__restrict__ y,
                                                     long ld_y, GemvFuse fuse) {
    gemv_body<1, MT, SL>(reinterpret_cast<const uint8_t *>(wq), scales, n_out, n_in, x, ld_x, n_m,
                         y, ld_y, fuse);
}

/* q8w_gemv_m1 for three to eight activation rows, on the matrix cores. v_mfma_f32_4x4x1 performs, for
 * sixteen blocks of four lanes, one fused multiply-add per output, rounded once (subnormals kept:
 * compared with fmaf over every range of exponents), so a chain stays a chain: an accumulator per
 * chain takes the columns 16 t + j in order as the reference's do. A lane holds a table row (its
 * weight is the instruction's second operand); of the first operand one block of four activations
 * is broadcast to all blocks, so one register carries sixteen columns of four activation rows and
 * the instruction's block selector picks the column. Output register i of a lane: activation row i
 * against the lane's table row.
 *
 * A workgroup has 64 table rows, a wavefront of it four of the sixteen chains (its quarter of every
 * sixteen columns): four times the wavefronts that whole chains would give, which a table of 32000
 * rows needs to fill the chip. 256 columns are staged in LDS as dwords [column / 4][row] -- written and
 * read without bank conflicts --, two stages take turns, and two more are on their way in registers.
 *
 * What bounds it: the table's bytes (128256 x 2560, 4 rows 66 us, 5.0 TB/s), and from five rows on the
 * matrix cores too (63e12 of these multiply-adds a second in a loop of nothing else: 42 of the 93 us
 * of 8 rows; the vector unit's rate is half that). The vector form, with an LDS read for every four
 * multiply-adds and eight rows' work for five, waited for LDS: 92 us for 4 rows, 152 for 8;
 * 32000 x 3072, 3 rows 44 -> 25, 8 rows 78 -> 30. */
typedef float mfma_f4 __attribute__((ext_vector_type(4)));
template <int J>
__device__ __forceinline__ void chain_mfma(float x, float w, mfma_f4 &acc) {
    acc = __builtin_amdgcn_mfma_f32_4x4x1f32(x, w, acc, 4, J, 0);
}
/* Four columns, one of each of the wavefront's chains: d holds the lane's weights, x[g] the activations
 * of rows 4 g .. 4 g + 3 of four such steps, of which this is number U. */
template <int G, int U>
__device__ __forceinline__ void chains_step(uint32_t d, const float (&x)[G], mfma_f4 (&acc)[G][4]) {
    float w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        w[e] = (float) (int) (int8_t) (d >> (8 * e));
#pragma unroll
    for (int g = 0; g < G; ++g) {
        chain_mfma<4 * U + 0>(x[g], w[0], acc[g][0]);
        chain_mfma<4 * U + 1>(x[g], w[1], acc[g][1]);
        chain_mfma<4 * U + 2>(x[g], w[2], acc[g][2]);
        chain_mfma<4 * U + 3>(x[g], w[3], acc[g][3]);
    }
}
constexpr int MF_ROWS  = 64;  /* table rows of a workgroup */
constexpr int MF_COLS  = 256; /* columns of a stage */
constexpr int MF_PITCH = MF_ROWS + 1; /* dwords: rows 4 apart of 16 column groups fall on 64 banks */
__device__ __forceinline__ void mf_barrier() { /* orders LDS only: loads stay on their way */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <int G>
__global__ __launch_bounds__(LM_TPB, 4) void k_q8w_gemv_mfma(const int8_t *__restrict__ wq,
                                                             const float *__restrict__ scales,
                                                             long n_out, int n_in,
                                                             const float *__restrict__ x, long ld_x,
                                                             int n_m, float *__restrict__ y, long ld_y) {
    __shared__ union {
        uint32_t tile[2][MF_COLS / 4][MF_PITCH];
        float    chain[4][16][MF_ROWS]; /* the chains of four activation rows, at the end */
    } s;
    const int  tid = threadIdx.x, lane = tid & (LM_WAVE - 1);
    const int  wave = __builtin_amdgcn_readfirstlane(tid / LM_WAVE);
    const long row0 = (long) blockIdx.x * MF_ROWS;
    mfma_f4    acc[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc[g][e] = mfma_f4{0.0f, 0.0f, 0.0f, 0.0f};
    /* Rows beyond the table repeat its last, activation rows beyond n_m theirs, columns past the row's
     * end (n_in is a multiple of 16) its last sixteen: none of them is used. */
    const int     seg = tid & 15;
    const int8_t *wp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long r = row0 + 16 * i + (tid >> 4);
        wp[i]        = wq + (r < n_out ? r : n_out - 1) * n_in;
    }
    const float *xp[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int m = 4 * g + (lane & 3);
        xp[g]       = x + (m < n_m ? m : n_m - 1) * ld_x + 4 * wave + ((lane >> 2) & 3);
    }
    struct Regs {
        uint4 w[4];
    } r0, r1;
    auto load = [&](int st, Regs &r) {
        int col = st * MF_COLS + 16 * seg;
        col     = col < n_in ? col : n_in - 16;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            typedef uint32_t nt_u4 __attribute__((ext_vector_type(4)));
            const nt_u4 t = __builtin_nontemporal_load(reinterpret_cast<const nt_u4 *>(wp[i] + col));
            r.w[i]        = make_uint4(t.x, t.y, t.z, t.w);
        }
    };
    float xc[4][G], xn[4][G];
    auto  load_x = [&](int st) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            int col = st * MF_COLS + 64 * q + 16 * (lane >> 4);
            col     = col < n_in ? col : n_in - 16;
#pragma unroll
            for (int g = 0; g < G; ++g)
                xn[q][g] = xp[g][col];
        }
    };
    auto store = [&](int st, const Regs &r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t *t = &s.tile[st & 1][4 * seg][16 * i + (tid >> 4)];
            t[0 * MF_PITCH] = r.w[i].x;
            t[1 * MF_PITCH] = r.w[i].y;
            t[2 * MF_PITCH] = r.w[i].z;
            t[3 * MF_PITCH] = r.w[i].w;
        }
    };
    const int n_stage = (n_in + MF_COLS - 1) / MF_COLS;
    load(0, r0);
    if (n_stage > 1)
        load(1, r1);
    load_x(0);
    store(0, r0);
    if (n_stage > 2)
        load(2, r0);
    mf_barrier();
    /* Stage st is in LDS; `next` holds the one behind it, the other registers the one after. */
    auto stage = [&](int st, Regs &next) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int g = 0; g < G; ++g)
                xc[q][g] = xn[q][g];
        if (st + 1 < n_stage) {
            load_x(st + 1);
            store(st + 1, next); /* (read last before the barrier behind the stage before this) */
        }
        if (st + 3 < n_stage)
            load(st + 3, next);
        const uint32_t *t    = &s.tile[st & 1][wave][lane];
        const int       left = n_in - st * MF_COLS;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            /* (a branch per 64 columns: the compiler would convert a whole stage ahead) */
            if (64 * q >= left)
                break;
            chains_step<G, 0>(t[(16 * q + 0) * MF_PITCH], xc[q], acc);
            if (64 * q + 16 < left)
                chains_step<G, 1>(t[(16 * q + 4) * MF_PITCH], xc[q], acc);
            if (64 * q + 32 < left)
                chains_step<G, 2>(t[(16 * q + 8) * MF_PITCH], xc[q], acc);
            if (64 * q + 48 < left)
                chains_step<G, 3>(t[(16 * q + 12) * MF_PITCH], xc[q], acc);
        }
        mf_barrier();
    };
    for (int st = 0; st < n_stage; st += 2) {
        stage(st, r1);
        if (st + 1 < n_stage)
            stage(st + 1, r0);
    }
    /* wavefront i folds activation row i's chains: (chain j + chain j+8), (i + i+4),
     * ((0+1) + (2+3)), as gemv_body */
    const long  row   = row0 + lane;
    const float scale = row < n_out ? scales[row] : 0.0f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (g)
            mf_barrier();
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s.chain[i][4 * wave + e][lane] = acc[g][e][i];
        mf_barrier();
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = dadd(s.chain[wave][j][lane], s.chain[wave][j + 8][lane]);
        const float q0 = dadd(v[0], v[4]), q1 = dadd(v[1], v[5]);
        const float q2 = dadd(v[2], v[6]), q3 = dadd(v[3], v[7]);
        const float sum = __fmul_rn(dadd(dadd(q0, q1), dadd(q2, q3)), scale);
        if (row < n_out && 4 * g + wave < n_m)
            y[(4 * g + wave) * ld_y + row] = sum;
    }
}

/* The projection for several activation rows. Here a lane owns all sixteen chains of one weight
 * row (a wavefront works on 64 rows), so the activations of a step are the same for every lane
 * and come from scalar registers: each converted weight feeds n_m multiply-adds whose second
 * operand costs neither LDS traffic nor vector registers. The weights take the same way through
 * a private LDS tile as in k_f16_gemv. */
constexpr int ROWS_WAVE_B  = 64;
constexpr int ROWS_BLOCK_B = ROWS_WAVE_B * LM_WAVES;
constexpr int STAGE_LOADS_B = 8; /* 64 rows x 8 segments / 64 lanes */

struct StageRegsB {
    uint4 w[STAGE_LOADS_B];
};

__device__ __forceinline__ void stage_load_b(const uint16_t *__restrict__ w, long row0, long n_out,
                                             int n_in, int stage, int lane, StageRegsB &g) {
    const int col = stage * STAGE_COLS + (lane & 7) * 8;
#pragma unroll
    for (int i = 0; i < STAGE_LOADS_B; ++i) {
        const long row = row0 + 8 * i + (lane >> 3);
        g.w[i]         = make_uint4(0u, 0u, 0u, 0u);
        if (row < n_out && col < n_in) {
            typedef uint32_t nt_u4 __attribute__((ext_vector_type(4)));
            const nt_u4 t =
                __builtin_nontemporal_load(reinterpret_cast<const nt_u4 *>(w + row * n_in + col));
            g.w[i] = make_uint4(t.x, t.y, t.z, t.w);
        }
    }
}

/* Eight chains (one accumulator of the reference) of this lane's row against the activations
 * x[m][col .. col + 8), which are uniform over the wavefront. */
template <int MT>
__device__ __forceinline__ void gemv_half_step(const uint8_t *row_tile, int byte_off,
                                               const float *__restrict__ x, long ld_x, int n_m,
                                               int col, float (&acc)[MT][16], int chain0) {
    const uint4  q   = *reinterpret_cast<const uint4 *>(row_tile + byte_off);
    const float2 f01 = __half22float2(*reinterpret_cast<const __half2 *>(&q.x));
    const float2 f23 = __half22float2(*reinterpret_cast<const __half2 *>(&q.y));
    const float2 f45 = __half22float2(*reinterpret_cast<const __half2 *>(&q.z));
    const float2 f67 = __half22float2(*reinterpret_cast<const __half2 *>(&q.w));
    float        wf[8] = {f01.x, f01.y, f23.x, f23.y, f45.x, f45.y, f67.x, f67.y};
    /* keep the conversion a separate instruction: folded into a mixed-precision multiply-add it
     * is repeated per activation row, and that instruction takes no scalar operand, so every
     * activation would be copied to a vector register first */
#pragma unroll
    for (int i = 0; i < 8; ++i)
        asm("" : "+v"(wf[i]));
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const float *xm = x + (long) (m < n_m ? m : n_m - 1) * ld_x + col; /* uniform address */
#pragma unroll
        for (int i = 0; i < 8; ++i)
            acc[m][chain0 + i] = __builtin_fmaf(wf[i], xm[i], acc[m][chain0 + i]);
    }
}

template <int MT>
__global__ __launch_bounds__(LM_TPB) void k_f16_gemv_batched(const uint16_t *__restrict__ w,
                                                             long n_out, int n_in,
                                                             const float *__restrict__ x, long ld_x,
                                                             int n_m, float *__restrict__ y,
                                                             long ld_y) {
    __shared__ __align__(16) uint8_t s_tile[LM_WAVES][ROWS_WAVE_B * TILE_PITCH];
    const int  lane = threadIdx.x & (LM_WAVE - 1);
    const int  wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LM_WAVE);
    const long row0 = (long) blockIdx.x * ROWS_BLOCK_B + wave * ROWS_WAVE_B;
    if (row0 >= n_out)
        return;
    uint8_t       *tile     = s_tile[wave];
    const uint8_t *row_tile = tile + lane * TILE_PITCH;

    float acc[MT][16];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            acc[m][i] = 0.0f;

    const int  n_stage = (n_in + STAGE_COLS - 1) / STAGE_COLS;
    StageRegsB g0, g1;
    stage_load_b(w, row0, n_out, n_in, 0, lane, g0);
    if (n_stage > 1)
        stage_load_b(w, row0, n_out, n_in, 1, lane, g1);
    for (int s = 0; s < n_stage; ++s) {
#pragma unroll
        for (int i = 0; i < STAGE_LOADS_B; ++i)
            *reinterpret_cast<uint4 *>(tile + (8 * i + (lane >> 3)) * TILE_PITCH + (lane & 7) * 16) =
                g0.w[i];
        g0 = g1;
        if (s + 2 < n_stage)
            stage_load_b(w, row0, n_out, n_in, s + 2, lane, g1);
        const int col0 = s * STAGE_COLS;
        const int left = n_in - col0;
        if (left >= STAGE_COLS) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                gemv_half_step<MT>(row_tile, t * 32, x, ld_x, n_m, col0 + t * 16, acc, 0);
                gemv_half_step<MT>(row_tile, t * 32 + 16, x, ld_x, n_m, col0 + t * 16 + 8, acc, 8);
            }
        } else {
            const int full = left / 16;
            for (int t = 0; t < full; ++t) {
                gemv_half_step<MT>(row_tile, t * 32, x, ld_x, n_m, col0 + t * 16, acc, 0);
                gemv_half_step<MT>(row_tile, t * 32 + 16, x, ld_x, n_m, col0 + t * 16 + 8, acc, 8);
            }
            if ((left & 15) == 8) /* the block of eight extends chains 0..7 */
                gemv_half_step<MT>(row_tile, full * 32, x, ld_x, n_m, col0 + full * 16, acc, 0);
        }
    }
    const long row = row0 + lane;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = dadd(acc[m][i], acc[m][i + 8]);
        const float q0 = dadd(v[0], v[4]), q1 = dadd(v[1], v[5]);
        const float q2 = dadd(v[2], v[6]), q3 = dadd(v[3], v[7]);
        const float sum = dadd(dadd(q0, q1), dadd(q2, q3));
        if (row < n_out && m < n_m)
            y[m * ld_y + row] = sum;
    }
}

/* One workgroup per row. The reference adds the squares in double in index order; the order of
 * a double sum only shows in the binary32 result when 1 / sqrt(mean + eps) lies within the
 * sum's error of the middle between two binary32 values. The workgroup adds in a fixed parallel
 * order and, in that rare case, one thread repeats the sum in the reference's order. */
template <int TPB, int PER>
__global__ __launch_bounds__(TPB) void k_rmsnorm_rows(const float *__restrict__ x, long ld_x,
                                                      const float *__restrict__ w, float eps, int n,
                                                      float *__restrict__ y, long ld_y) {
    __shared__ NormShared s_norm;
    const int    tid = threadIdx.x;
    const float *xr  = x + (long) blockIdx.x * ld_x;
    float       *yr  = y + (long) blockIdx.x * ld_y;
    float        v[PER];
    const float  inv = block_rmsnorm<TPB, PER>(xr, w, n, eps, v, s_norm);
#pragma unroll
    for (int k = 0; k < PER; ++k)
        if (k * TPB + tid < n)
            yr[k * TPB + tid] = v[k];
    for (int i = PER * TPB + tid; i < n; i += TPB)
        yr[i] = __fmul_rn(__fmul_rn(xr[i], inv), w[i]);
}

void launch_rmsnorm_rows(hipStream_t stream, const float *x, long ld_x, const float *w, float eps,
                         int n_rows, int n, float *y, long ld_y) {
    auto go = [&](auto kernel, int tpb) {
        kernel<<<dim3(n_rows), dim3(tpb), 0, stream>>>(x, ld_x, w, eps, n, y, ld_y);
    };
    /* No more threads than hold a short row, and beyond the 512 rows that are at work at a time with
     * 1024 threads each, 256: many rows want many workgroups, few long ones all threads. 4096 rows
     * of 64 elements 4.9 us (16.6 with 1024 threads), of 1024 6.9 (18.0), of 2560 13.4 (20.7); 512
     * rows of 2560 4.8 (5.5 with 256), of 4096 4.9 (7.2). */
    if (n <= 256)
        go(k_rmsnorm_rows<64, 4>, 64);
    else if (n <= 1024)
        go(k_rmsnorm_rows<256, 4>, 256);
    else if (n_rows > 512 && n <= 4096)
        go(k_rmsnorm_rows<256, 16>, 256);
    else
        go(k_rmsnorm_rows<NORM_TPB, NORM_PER>, NORM_TPB);
}

bool f16_gemv_can_fuse(int n_m) { return n_m >= 1 && n_m <= 2; }

void launch_f16_gemv(hipStream_t stream, const uint16_t *w_f16, long n_out, int n_in,
                     const float *x, long ld_x, int n_m, float *y, long ld_y,
                     const GemvFuse *fuse) {
    const dim3 block(LM_TPB);
    const dim3 grid((unsigned) ((n_out + ROWS_BLOCK - 1) / ROWS_BLOCK));
    const dim3 grid_b((unsigned) ((n_out + ROWS_BLOCK_B - 1) / ROWS_BLOCK_B));
    GemvFuse   none{};
    if (fuse && fuse->tmax) { /* (the caller has asked f16_gemv_can_fuse) */
        const dim3 grid_s((unsigned) (fuse->n_chunks * 256 / LM_WAVES));
        if (n_m <= 1)
            k_f16_gemv<1, true><<<grid_s, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y, *fuse);
        else
            k_f16_gemv<2, true><<<grid_s, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y, *fuse);
        return;
    }
    if (n_m <= 1)
        k_f16_gemv<1, false><<<grid, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y, none);
    else if (n_m <= 2)
        k_f16_gemv<2, false><<<grid, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y, none);
    else if (n_m <= 4) /* (with 8 rows the batched kernel's 128 accumulators leave no room) */
        k_f16_gemv_batched<4><<<grid_b, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y);
    else
        k_f16_gemv<8, false><<<grid, block, 0, stream>>>(w_f16, n_out, n_in, x, ld_x, n_m, y, ld_y, none);
}

/* f16_to_q8w (kernel_f16_gemv.c:66-93): per row scale = max|w| / 127, q = lrintf(w * (127 /
 * max|w|)) clamped to +-127. One workgroup per row. */
__global__ __launch_bounds__(LM_TPB) void k_f16_to_q8w(const uint16_t *__restrict__ w, int n_in,
                                                       int8_t *__restrict__ wq,
                                                       float *__restrict__ scales) {
    __shared__ float s_max[LM_TPB];
    const int        tid = threadIdx.x;
    const uint16_t  *wr  = w + (long) blockIdx.x * n_in;
    float            a   = 0.0f;
    for (int k = tid; k < n_in; k += LM_TPB) {
        const float v = fabsf(__half2float(*reinterpret_cast<const __half *>(wr + k)));
        a             = v > a ? v : a; /* (a NaN never replaces the maximum, as in the reference) */
    }
    s_max[tid] = a;
    __syncthreads();
    for (int step = LM_TPB / 2; step > 0; step >>= 1) {
        if (tid < step)
            s_max[tid] = s_max[tid + step] > s_max[tid] ? s_max[tid + step] : s_max[tid];
        __syncthreads();
    }
    const float amax = s_max[0];
    const float id   = amax > 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
    if (tid == 0)
        scales[blockIdx.x] = __fdiv_rn(amax, 127.0f);
    int8_t *qr = wq + (long) blockIdx.x * n_in;
    for (int k = tid; k < n_in; k += LM_TPB) {
        const float v = __fmul_rn(__half2float(*reinterpret_cast<const __half *>(wr + k)), id);
        int         q = __float2int_rn(v); /* lrintf: to nearest, ties to even */
        q             = q > 127 ? 127 : q;
        q             = q < -127 ? -127 : q;
        qr[k]         = (int8_t) q;
    }
}

void launch_f16_to_q8w(hipStream_t stream, const uint16_t *w_f16, long n_out, int n_in, int8_t *wq,
                       float *scales) {
    k_f16_to_q8w<<<dim3((unsigned) n_out), dim3(LM_TPB), 0, stream>>>(w_f16, n_in, wq, scales);
}

void launch_q8w_gemv(hipStream_t stream, const int8_t *wq, const float *scales, long n_out,
                     int n_in, const float *x, long ld_x, int n_m, float *y, long ld_y,
                     const GemvFuse *fuse) {
    const dim3 block(LM_TPB);
    const dim3 grid((unsigned) ((n_out + ROWS_BLOCK - 1) / ROWS_BLOCK));
    GemvFuse   none{};
    if (fuse && fuse->tmax) {
        const dim3 grid_s((unsigned) (fuse->n_chunks * 256 / LM_WAVES));
        if (n_m <= 1)
            k_q8w_gemv<1, true><<<grid_s, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y, *fuse);
        else
            k_q8w_gemv<2, true><<<grid_s, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y, *fuse);
        return;
    }
    if (n_m <= 1)
        k_q8w_gemv<1, false><<<grid, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y,
                                                         fuse ? *fuse : none);
    else if (n_m <= 2)
        k_q8w_gemv<2, false><<<grid, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y, none);
    else {
        const dim3 grid_m((unsigned) ((n_out + MF_ROWS - 1) / MF_ROWS));
        if (n_m <= 4)
            k_q8w_gemv_mfma<1><<<grid_m, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y);
        else
            k_q8w_gemv_mfma<2><<<grid_m, block, 0, stream>>>(wq, scales, n_out, n_in, x, ld_x, n_m, y, ld_y);
    }
}

} // namespace gs
