// Log-sum-exp merge of the chunk partials of one (batch element, head) by one wave: eight
// output dims per lane, one 16-byte piece of each chunk's bf16 accumulator row.
#ifndef YVEX_ROCM_KERNELS_MERGE_ROWS_H
#define YVEX_ROCM_KERNELS_MERGE_ROWS_H

#include "mfma.h"

// One of the 16 rotations of every row of 16 lanes.
template <int kLanes>
__device__ inline float rotated16(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + kLanes, 0xf, 0xf,
                                                              true));
}

__device__ inline float wave_max(float v)
{
    v = fmaxf(v, rotated16<8>(v));
    v = fmaxf(v, rotated16<4>(v));
    v = fmaxf(v, rotated16<2>(v));
    v = fmaxf(v, rotated16<1>(v));
    return max_xor32(max_xor16(v));
}

__device__ inline float wave_sum(float v)
{
    v += rotated16<8>(v);
    v += rotated16<4>(v);
    v += rotated16<2>(v);
    v += rotated16<1>(v);
    return sum_xor32(sum_xor16(v));
}

// The statistics of 64 chunks are one load, a chunk per lane, and so are their weights; the rows
// come sixteen chunks per trip, every load of a trip independent of the others (chunks past the
// end alias the last one with weight zero): one memory round trip per sixteen chunks.  With every
// lane loading and weighing the statistics of every chunk for itself the merge of 16 x 128 rows of
// 512 dims over 3 to 16 chunks took 6.7 us, this 6.1 us; over 16 chunks each (33 MB of partials) both
// take 8.0 us.
//   stats(c):       (running maximum in log2 units, denominator) of chunk c
//   piece(c):       the lane's 16 bytes of chunk c's row, c the same in all lanes
//   meanwhile():    work of the caller that runs while the first loads are in flight
template <class Stats, class Piece, class Meanwhile>
__device__ inline void merge_chunk_rows(uint32_t chunks, uint32_t lane, Stats stats, Piece piece,
                                        Meanwhile meanwhile, float &top, float &total, float (&acc)[8])
{
    top = -INFINITY;
    total = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    float weight = 0.f;
    for (uint32_t c0 = 0; c0 < chunks; c0 += 16u) {
        u32x2 ml = {0u, 0u};
        if ((c0 & 63u) == 0u) ml = stats(min(c0 + lane, chunks - 1u));
        u32x4 row[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) row[j] = piece(min(c0 + (uint32_t)j, chunks - 1u));
        __builtin_amdgcn_sched_barrier(0);  // every load is on its way
        if (c0 == 0u) meanwhile();
        if ((c0 & 63u) == 0u) {
            const uint32_t mx = ml.x, dx = ml.y;
            const float m = c0 + lane < chunks ? __builtin_bit_cast(float, mx) : -INFINITY;
            const float m_new = fmaxf(top, wave_max(m));
            const float keep = fast_exp2(top - m_new);  // 0 at the start (top = -inf)
            weight = fast_exp2(m - m_new);
            total = total * keep + wave_sum(c0 + lane < chunks ? weight * __builtin_bit_cast(float, dx) : 0.f);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] *= keep;
            top = m_new;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float w = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), (int)((c0 & 63u) + (uint32_t)j)));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i + 0] += w * bf16_to_f32((uint16_t)(row[j][i] & 0xffffu));
                acc[2 * i + 1] += w * bf16_to_f32((uint16_t)(row[j][i] >> 16));
            }
        }
    }
}

// The head's sink logit joins the softmax with a zero value row
// (src/graph/core.c:471-508): it only enlarges the denominator.  Returns false for a sink
// that is not finite.
__device__ inline bool merge_sink(float sink_logit, float &top, float &total, float (&acc)[8])
{
    const float sink = sink_logit * 1.4426950408889634f;  // log2 units, as the maxima
    const float m_new = fmaxf(top, sink);
    const float keep = fast_exp2(top - m_new);
    total = total * keep + fast_exp2(sink - m_new);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] *= keep;
    top = m_new;
    return isfinite(sink);
}

#endif  // YVEX_ROCM_KERNELS_MERGE_ROWS_H
