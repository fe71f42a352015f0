/*
 * sampler_greedy.h -- argmax over a row of logits (sampler.c:52-62) in one launch.
 */
#ifndef GEIST_SAMPLER_GREEDY_H
#define GEIST_SAMPLER_GREEDY_H

namespace gs {

template <int NV, bool PEN, bool PLAIN>
__device__ __forceinline__ void greedy_chunk(const RowView &rv, int row, int chunk, int n_rows,
                                             int base, int end, int32_t *__restrict__ out,
                                             uint32_t *s_cnt16, const FusedScan &fs) {
    const int  tid = threadIdx.x;
    const bool collects = chunk == rv.n_chunks - 1;
    HistPrefetch pf;
    if (PEN)
        pf = history_prefetch(rv, row, n_rows);
    float4       v[NV];
    const float *rowp = rv.logits + (long) row * rv.ld;
    if (PLAIN) {
        const float4 *p = reinterpret_cast<const float4 *>(rowp + base) + tid;
        if (rv.stream_loads) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
                v[j] = load_streaming(p + j * TPB);
        } else {
#pragma unroll
            for (int j = 0; j < NV; ++j)
                v[j] = p[j * TPB];
        }
    } else {
        load_raw<NV>(rv, rowp, base, end, v);
    }
    float first = 0.0f;
    if (collects)
        first = rowp[0];
    if (tid == 0)
        fs.s_arrive[0] = 0;
    if (PEN) {
        history_clear<NV * TPB * 4>(s_cnt16);
        history_count(rv, row, pf, base, end, s_cnt16);
    } else {
        lds_barrier();
    }
    float tm = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        transform_group<PEN, !PLAIN>(rv, row, s_cnt16, 4 * (j * TPB + tid), base, end, v[j]);
        tm = max3f(tm, max3f(v[j].x, v[j].y, v[j].z), v[j].w);
    }
    if (base + 4 * tid >= end)
        tm = __builtin_nanf("");
    const uint32_t bk   = wave_max_u32(f2key(tm));
    uint64_t       best = wave_first_of<NV, PLAIN>(v, bk, base, end);
    if ((tid & (WAVE - 1)) == 0)
        fs.s_red[tid / WAVE] = best;
    const bool last = wave_arrives_last(fs.s_arrive);
    if (last) {
        best = fs.s_red[0];
#pragma unroll
        for (int w = 1; w < NWAVES; ++w)
            best = fs.s_red[w] > best ? fs.s_red[w] : best;
        if (!best) /* an all-NaN chunk reports key 0 at its first index */
            best = pack_best(0u, (uint32_t) base);
    }
    if (!collects) {
        if (last && (tid & (WAVE - 1)) == 0)
            meet_store(fs.slots + (long) row * rv.n_chunks + chunk, best, fs.local);
        return;
    }
    const uint64_t bb = row_best_meet<NV, PEN>(rv, row, chunk, n_rows, best, last, fs, s_cnt16);
    if (tid == 0) {
        /* a NaN at index 0 is never displaced by the strict '>' of the reference; after the
         * transforms it stays NaN, so the raw value decides (unless token 0 is forbidden) */
        const bool nan0 = first != first && (!rv.allowed || allowed_at(rv, row, 0));
        out[row]        = nan0 ? 0 : (int32_t) best_idx(bb);
    }
}

/* grid (chunks, rows): every workgroup reports its chunk's maximum with its first index into the
 * chunk's meeting slot and leaves; the one of the row's last chunk, which starts last, waits for
 * the others' (row_best_meet: bounded, past the bound it reads the row itself) and writes the id.
 *
 * What bounds it: one row is a launch and two round trips to memory, a large batch the bytes (256 x
 * 262144: 268 MB in 45.1 us, 5.9 TB/s). A scan that stored the chunks' and the threads' maxima and a
 * second launch that combined them were 51.3 us there, 6.5 against 4.2 for 1 x 32000, 10.7 against
 * 7.9 for 64 x 128256 and 14.3 against 11.8 with 2048 tokens of penalties. One store and no
 * read-modify-write per workgroup: nobody waits but the one that writes the id. (Rows of fewer than
 * eight on one XCD each, as the temperature draw has them: within 0.1 us either way, 7 x 128256
 * 4.3 against 4.0; not done.) */
template <int NV, bool PEN>
__global__ __launch_bounds__(TPB) void k_greedy(RowView rv, int32_t *__restrict__ out, MeetSpace meet) {
    __shared__ __align__(16) uint32_t s_cnt16[PEN ? NV * TPB * 2 : 1];
    __shared__ uint64_t s_red[NWAVES], s_bb;
    __shared__ uint32_t s_arrive[1];
    const int tid = threadIdx.x;
    int       row, chunk;
    xcd_row_chunk(row, chunk);
    {
        const uint32_t wg = blockIdx.y * gridDim.x + blockIdx.x, n_wg = gridDim.x * gridDim.y;
        for (uint32_t i = wg * TPB + tid; i < meet.stale_count; i += n_wg * TPB)
            meet.stale[i] = 0;
    }
    int base, end;
    chunk_bounds<NV>(rv, chunk, base, end);
    FusedScan fs;
    fs.tmax       = nullptr;
    fs.chunk_best = nullptr;
    fs.slots      = meet.slots;
    fs.wait_limit = meet.wait_limit;
    fs.local      = meet.local;
    fs.s_red      = s_red;
    fs.s_bb       = &s_bb;
    fs.s_arrive   = s_arrive;
    const bool plain = rv.vec_ok && end - base == NV * TPB * 4 && !(rv.softcap > 0.0f) &&
                       rv.allowed == nullptr;
    if (plain)
        greedy_chunk<NV, PEN, true>(rv, row, chunk, rv.n_rows, base, end, out, s_cnt16, fs);
    else
        greedy_chunk<NV, PEN, false>(rv, row, chunk, rv.n_rows, base, end, out, s_cnt16, fs);
}

} // namespace gs
#endif
