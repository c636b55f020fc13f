// The fp32 walk of the rows of an item whose parts left the range: what gqa_f32_halved.h falls back to.
#ifndef YVEX_ROCM_KERNELS_GQA_F32_AGAIN_H
#define YVEX_ROCM_KERNELS_GQA_F32_AGAIN_H

#include <hip/hip_runtime.h>

#include "../kernel_params.h"
#include "gqa_f32_walk.h"
#include "mfma.h"

namespace {

// What a run of keys contributes to row `row` of its tile (the maximum in log2 units).
template <int kBlocks>
__device__ __forceinline__ void leave_partial(float *part_acc, float *part_ml, uint32_t slot, uint32_t row, int half,
                                              const floatx16 (&o)[kBlocks], float m, float l)
{
    const uint64_t at = (uint64_t)slot * YVEX_ROCM_PREFILL_ROWS + row;
    if (half == 0) {
        part_ml[at * 2u] = m;
        part_ml[at * 2u + 1u] = l;
    }
    float *acc = part_acc + at * (32u * kBlocks) + half * 4;
#pragma unroll
    for (int b = 0; b < kBlocks; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<floatx4 *>(acc + b * 32 + g * 8) =
                (floatx4){o[b][g * 4], o[b][g * 4 + 1], o[b][g * 4 + 2], o[b][g * 4 + 3]};
}

// Row `row` of a tile, of which the bits of lower (rows 0 to 63) and upper (64 to 127) failed.
__device__ __forceinline__ bool row_failed(uint64_t lower, uint64_t upper, uint32_t row)
{
    return ((row < 64u ? lower : upper) >> (row & 63u) & 1ull) != 0ull;
}

// The item, or the run, once more in fp32, its rows packed as they are.  Only the rows that failed (bits of
// `failed`, 32 rows to a word) are left: the others have been, and what a row gives does
// not depend on whether another one fails.  Head by head, with the tokens of a head in its tiles, it took
// as many walks as heads share a tile (every row failed, 1777 tokens of 40/8 heads of 128 1420 us, 1000 of 24/4 of 256
// 2260; now 424 and 447, in one launch 313 and 291).  A function of its own, whose registers are not found by spilling
// the walk's (64 tokens behind 20000 at 24/4 heads of 256 209 us, inlined 211 to 215; the others alike).  It takes the
// kernel's arguments from where they lie; `arguments` is the kernel's to find, a function that is called is not
// given the place.
typedef __attribute__((address_space(3))) unsigned char local_bytes;
typedef __attribute__((address_space(4))) const yvex_rocm_gqa_f32_halved_params constant_params;
template <int kDim>
__device__ __attribute__((noinline)) void
walk_again(constant_params *arguments, local_bytes *shared, u32x4 failed, bool cut, uint32_t slot_, uint32_t row_head_,
           uint32_t tile_row_, uint32_t tile_end_, uint32_t first_tile_, uint32_t tiles_)
{
    auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    const uint64_t at = (uint64_t)arguments;
    constant_params &p = *(constant_params *)((uint64_t)uniform((uint32_t)(at >> 32)) << 32 | uniform((uint32_t)at));
    const uint32_t slot = uniform(slot_), row_head = uniform(row_head_), tile_row = uniform(tile_row_);
    const uint32_t tile_end = uniform(tile_end_), first_tile = uniform(first_tile_), tiles = uniform(tiles_);
    const bool partial = uniform(cut) != 0u;
    const uint32_t pack = p.walk.pack;
    const uint64_t lower = (uint64_t)uniform(failed[1]) << 32 | uniform(failed[0]);
    const uint64_t upper = (uint64_t)uniform(failed[3]) << 32 | uniform(failed[2]);
    yvex_rocm_gqa_f32_params f = {};
    f.q = (const float *)p.walk.q;
    f.k = (const float *)p.walk.k;
    f.v = (const float *)p.walk.v;
    f.out = (float *)p.walk.out;
    f.lse = p.walk.lse;
    f.status = p.walk.status;
    f.query_tokens = p.walk.query_tokens;
    f.kv_tokens = p.walk.kv_tokens;
    f.query_start = p.walk.query_start;
    f.query_heads = p.walk.query_heads;
    f.kv_heads = p.walk.kv_heads;
    f.q_stride = p.walk.q_stride;
    f.k_stride = p.walk.k_stride;
    f.v_stride = p.walk.v_stride;
    f.scale = p.scale;
    f.causal = (int32_t)p.walk.causal;
    float *const part_acc = p.walk.part_acc, *const part_ml = p.walk.part_ml;
    const GqaTile<kDim / 32> tile(f, (float *)(unsigned char *)shared, (int)threadIdx.x);
    // the rows as they are packed; a wave without one that failed only stages (its lanes' words are the same)
    const uint64_t word = tile.wave < 2 ? lower : upper;
    const bool idle = (uint32_t)(tile.wave % 2 == 0 ? word : word >> 32) == 0u;
    typedef typename GqaTile<kDim / 32>::Place Place;
    tile.walk(row_head * pack / (p.walk.query_heads / p.walk.kv_heads), tile_end - tile_row, idle,
              [&](uint32_t row) {
                  const uint32_t token = (tile_row + row) / pack;
                  return Place{token, row_head * pack + (tile_row + row - token * pack)};
              },
              first_tile, partial ? first_tile + tiles : ~0ull >> 8,
              [&](const Place &place, uint32_t row, floatx16(&o)[kDim / 32], float m, float l) {
                  if (!row_failed(lower, upper, row)) return;
                  if (partial)
                      leave_partial(part_acc, part_ml, slot, row, tile.half, o, m * YVEX_LOG2E, l);
                  else
                      tile.publish(place.head, place.token, o, m, l);
              });
}

}  // namespace

#endif  // YVEX_ROCM_KERNELS_GQA_F32_AGAIN_H
