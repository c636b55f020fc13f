// EXACT_F32 grouped-query attention on the matrix cores of gfx950 (wave64): the fp32 walk of items of 128 query
// tokens of one query head (gqa_f32_walk.h), which needs no workspace, and the walk over keys and values split
// beforehand (gqa_f32_halved.h).
//
// The one-launch form stays with fp32 products.  Split products in it take 150 us instead of 310 (1777 tokens of
// 40/8 heads of 128), but with one power of two to eight rows they lost what lay 2^20 and more below the largest of
// the eight, and split as the walk over halves splits them every workgroup would make the splits for itself again.
//
// grid = query_heads * ceil(query_tokens / 128), the longest (last) query tiles first;
// block = 256 (512 at head dimension 256).
#include <hip/hip_runtime.h>

#include "../kernel_params.h"
#include "gqa_f32_halved.h"
#include "gqa_f32_walk.h"
#include "run_merge.h"

namespace {

// Items (one head, one tile of queries) are numbered heaviest first.  A scheduled launch
// hands every workgroup a row of items (the count, then the items, 16 bytes: one scalar
// load); otherwise the workgroup runs the one item its number stands for.
// Without lists the hardware gives workgroup b of the first 2 * pair_units to compute
// unit b % pair_units, and a unit's time follows the key tiles it walks: the second workgroup
// of a unit takes the second tier of items in reverse, and the unit that got the heaviest item
// gets the lightest of them (equal sums for causal walks).
template <typename Walk>
__device__ void run_items(const yvex_rocm_gqa_f32_params &p, float *shared)
{
    uint32_t count = 1u;
    u32x4 row = {0u, 0u, 0u, 0u};
    if (p.lists != nullptr) {
        typedef __attribute__((address_space(4))) const u32x4 constant_u32x4;
        row = *(constant_u32x4 *)(uintptr_t)(p.lists + (uint64_t)blockIdx.x * 8u);
        count = min(row.x & 0xffffu, 7u);
    }
    const uint32_t paired = blockIdx.x >= p.pair_units && blockIdx.x < 2u * p.pair_units
                                ? 3u * p.pair_units - 1u - blockIdx.x
                                : blockIdx.x;
    for (uint32_t j = 1u; j <= count; ++j) {
        const uint32_t word = j >> 1 == 0u ? row.x : j >> 1 == 1u ? row.y : j >> 1 == 2u ? row.z : row.w;
        const uint32_t id = p.lists != nullptr ? (word >> ((j & 1u) * 16u)) & 0xffffu : paired;
        // (opaque, so that what depends on the lane is not kept in registers from item to item)
        int thread = (int)threadIdx.x;
        __asm__ volatile("" : "+v"(thread));
        Walk(p, shared, thread).item(id);
        // every wave is done with the tiles in LDS before the next item stages its own
        if (j < count) __syncthreads();
    }
}

// Merge of the runs of cut items.
template <int kDim>
__device__ __forceinline__ void merge_f32(const yvex_rocm_prefill_params &p, floatx4 *acc_of, float2 *ml_of)
{
    merge_runs<kDim>(p, acc_of, ml_of, [&](uint64_t row, uint32_t d, const floatx4 &acc, float top, float sum) {
        if (!(sum > 0.f) || !isfinite(sum) || !isfinite(top)) return flag_status(p.status, YVEX_ROCM_DEVICE_NUMERIC);
        floatx4 o;
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = acc[i] / sum;
            bad |= !isfinite(o[i]);
        }
        *reinterpret_cast<floatx4 *>((float *)p.out + row * kDim + d) = o;
        if (bad) flag_status(p.status, YVEX_ROCM_DEVICE_NUMERIC);
        if (p.lse && d == 0u) p.lse[row] = top * YVEX_LN2 + logf(sum);
    });
}

constexpr int larger(int a, int b) { return a > b ? a : b; }

}  // namespace

// `waves`: waves per SIMD the register budget is sized for.
#define YVEX_GQA_F32_TILE_KERNEL(name, walk, threads, waves)                                                  \
    extern "C" __global__ void __launch_bounds__(threads) __attribute__((amdgpu_waves_per_eu(waves, waves)))   \
    name(const yvex_rocm_gqa_f32_params p)                                                                      \
    {                                                                                                           \
        __shared__ __attribute__((aligned(16))) float lds[2 * walk::kStageFloats];                              \
        run_items<walk>(p, lds);                                                                                \
    }

YVEX_GQA_F32_TILE_KERNEL(yvex_rocm_gqa_f32_tile_64, GqaTile<2>, 256, 2)
YVEX_GQA_F32_TILE_KERNEL(yvex_rocm_gqa_f32_tile_128, GqaTile<4>, 256, 2)
// pairs of waves split the head dimension
YVEX_GQA_F32_TILE_KERNEL(yvex_rocm_gqa_f32_tile_256, GqaTilePair, 512, 2)

#define YVEX_GQA_F32_HALVED_KERNELS(dim, waves)                                                                   \
    extern "C" __global__ void __launch_bounds__(256)                                                             \
    yvex_rocm_gqa_f32_halve_##dim(const yvex_rocm_gqa_f32_halved_params p)                                        \
    {                                                                                                             \
        __shared__ __attribute__((aligned(16))) unsigned char lds[HalvedTile<dim>::kBytes];                       \
        HalveRows<dim>::run(p, lds);                                                                              \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(waves, waves)))          \
    yvex_rocm_gqa_f32_halved_##dim(const yvex_rocm_gqa_f32_halved_params p)                                       \
    {                                                                                                             \
        typedef GqaHalved<dim> Halved;                                                                            \
        __shared__ __attribute__((aligned(16))) unsigned char                                                     \
            lds[larger((int)sizeof(Halved::Shared), (int)sizeof(float) * 2 * GqaTile<dim / 32>::kStageFloats)];   \
        Halved(p, *reinterpret_cast<Halved::Shared *>(lds), (int)threadIdx.x).run();                              \
    }                                                                                                             \
    extern "C" __global__ void __launch_bounds__(256)                                                             \
    yvex_rocm_gqa_f32_merge_##dim(const yvex_rocm_gqa_f32_halved_params p)                                        \
    {                                                                                                             \
        __shared__ floatx4 acc_of[256];                                                                           \
        __shared__ float2 ml_of[256];                                                                             \
        merge_f32<dim>(p.walk, acc_of, ml_of);                                                                    \
    }

// two workgroups per unit; one at 256, whose accumulators and queries take 256 registers a lane
YVEX_GQA_F32_HALVED_KERNELS(64, 2)
YVEX_GQA_F32_HALVED_KERNELS(128, 2)
YVEX_GQA_F32_HALVED_KERNELS(256, 1)
