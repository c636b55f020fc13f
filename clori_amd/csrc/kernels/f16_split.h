// F32 values as the sum of two f16 values, for products on the f16 matrix cores.
#ifndef YVEX_ROCM_KERNELS_F16_SPLIT_H
#define YVEX_ROCM_KERNELS_F16_SPLIT_H

#include "mfma.h"

namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ floatx16 mfma_32x32x16_f16(halfx8 a, halfx8 b, floatx16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Biased exponent that a query row whose largest magnitude has these bits is scaled by: 2^(141 - e)
// brings it to [2^14, 2^15).  A row below 2^-62 is scaled as one of that size (so that 2^(e - 141) times a
// score's unit stays a normal number), one of 2^51 and more as one of that.
constexpr uint32_t kExponentLeast = 64u, kExponentMost = 177u;

__device__ __forceinline__ uint32_t row_exponent(uint32_t max_bits)
{
    return min(max(max_bits >> 23, kExponentLeast), kExponentMost);
}

__device__ __forceinline__ float power_of_two(uint32_t biased) { return __builtin_bit_cast(float, biased << 23); }

__device__ __forceinline__ float down_factor(uint32_t e) { return power_of_two(268u - e); }
__device__ __forceinline__ float up_factor(uint32_t e) { return power_of_two(e - 14u); }

template <int kValue>
struct Index {
    static constexpr int value = kValue;
};
// f(Index<0>), f(Index<1>) ... f(Index<kCount - 1>): the slots of a trip are more than a loop is unrolled for
template <int kCount, int kFrom = 0, typename F>
__device__ __forceinline__ void for_each(const F &f)
{
    if constexpr (kFrom < kCount) {
        f(Index<kFrom>());
        for_each<kCount, kFrom + 1>(f);
    }
}

// Two values times `factor` as pairs of halves: four instructions, one rounding each (the compiler takes
// seven).  The compiler sees no instructions here and inserts no wait states: the values must not come
// straight from a transcendental instruction (whose result the next but one may read first), and the
// results not go straight into an MFMA or a lane exchange (two instructions in between).
__device__ __forceinline__ void split_pair_by_lane(float a, float b, float factor, uint32_t &hi, uint32_t &lo)
{
    __asm__ volatile("v_fma_mixlo_f16 %0, %2, %4, 0\n\t"
                     "v_fma_mixhi_f16 %0, %3, %4, 0\n\t"
                     "v_fma_mixlo_f16 %1, %2, %4, -%0 op_sel_hi:[0,0,1]\n\t"
                     "v_fma_mixhi_f16 %1, %3, %4, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
                     : "=&v"(hi), "=&v"(lo)
                     : "v"(a), "v"(b), "v"(factor));
}

// x / y given r = 1 / y: one step of Newton's method from x r, which leaves the nearest value but for rare
// halfway cases (a division takes four times as many instructions; a row has head_dim of them).
__device__ __forceinline__ float quotient(float x, float y, float r)
{
    const float q = x * r;
    return fmaf(fmaf(-q, y, x), r, q);
}

}  // namespace

#endif  // YVEX_ROCM_KERNELS_F16_SPLIT_H
