// Row arithmetic shared by the prefill kernels (kernel_params.h: packed rows, items).
#ifndef YVEX_ROCM_KERNELS_PREFILL_ROWS_H
#define YVEX_ROCM_KERNELS_PREFILL_ROWS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../kernel_params.h"

// token of packed row `row`: a division by `pack` (2 to 16 query heads) as a multiplication by its
// rounded-up inverse, exact below 2^28 rows
__device__ inline uint32_t token_of(const yvex_rocm_prefill_params &p, uint32_t row)
{
    return p.pack == 1u ? row : __umulhi(row, p.pack_inverse);
}

// kv head of a row head
__device__ inline uint32_t kv_head_of(const yvex_rocm_prefill_params &p, uint32_t row_head)
{
    return p.row_heads == p.kv_heads ? row_head : row_head * p.kv_heads / p.row_heads;
}

#endif  // YVEX_ROCM_KERNELS_PREFILL_ROWS_H
