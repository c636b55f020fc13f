// Merge of the partials that runs of keys leave (kernel_params.h: yvex_rocm_prefill_params).
#ifndef YVEX_ROCM_KERNELS_RUN_MERGE_H
#define YVEX_ROCM_KERNELS_RUN_MERGE_H

#include "mfma.h"
#include "prefill_rows.h"

#include "../kernel_params.h"

// Log-sum-exp merge of the runs of the split items and publication of their rows: publish(token * query_heads +
// head, first dim, accumulators, maximum in log2 units, denominator).  head_dim / 4
// threads per row and group, four lanes of the row each; the runs of a row are dealt to
// merge_groups (1 or 4) groups of threads, merged within each in the order of the runs and then
// group by group.  grid = tail_items * YVEX_ROCM_PREFILL_ROWS * head_dim / 4 * merge_groups / 256,
// block = 256.
// A trip of eight runs is a trip to memory, and few tokens leave few rows to hide it: 9 tokens of
// 40/8 heads of 128 in 32 runs took 6.5 us with one group (four trips one after the other): the call
// 20.1 us, now 17.4 us.
template <int kHeadDim, class Publish>
__device__ __forceinline__ void merge_runs(const yvex_rocm_prefill_params &p, floatx4 *acc_of, float2 *ml_of,
                                           const Publish &publish)
{
    constexpr uint32_t kRows = YVEX_ROCM_PREFILL_ROWS, kThreads = kHeadDim / 4;
    constexpr int kWidth = 8;  // runs in flight per trip
    const uint32_t groups = p.merge_groups, member = threadIdx.x / kThreads, d = (threadIdx.x % kThreads) * 4u;
    const uint32_t group = member & (groups - 1u);
    const uint32_t packed = blockIdx.x * (256u / kThreads / groups) + member / groups;
    const uint32_t tail = packed / kRows, in_tile = packed % kRows;
    const uint32_t item = p.whole_items + tail;
    const uint32_t row = (p.query_tiles - 1u - item / p.row_heads) * kRows + in_tile;
    const bool live = row < p.rows;
    const uint64_t first = (uint64_t)tail * p.splits * kRows + in_tile;
    const uint32_t each = (p.splits + groups - 1u) / groups;
    const uint32_t begin = min(group * each, p.splits), end = live ? min(begin + each, p.splits) : begin;
    float top = -INFINITY, sum = 0.f;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t s0 = begin; s0 < end; s0 += (uint32_t)kWidth) {
        float m[kWidth], l[kWidth];
        floatx4 part[kWidth];
#pragma unroll
        for (int i = 0; i < kWidth; ++i) {
            // runs past the end alias the last one, with weight zero
            const uint64_t at = first + (uint64_t)min(s0 + (uint32_t)i, end - 1u) * kRows;
            m[i] = p.part_ml[at * 2u];
            l[i] = p.part_ml[at * 2u + 1u];
            part[i] = *reinterpret_cast<const floatx4 *>(p.part_acc + at * kHeadDim + d);
        }
        float m_new = top;
#pragma unroll
        for (int i = 0; i < kWidth; ++i) {
            if (s0 + (uint32_t)i >= end) m[i] = -INFINITY, l[i] = 0.f;
            m_new = fmaxf(m_new, m[i]);
        }
        const float keep = m_new == -INFINITY ? 1.f : fast_exp2(top - m_new);
        sum *= keep;
        acc *= keep;
#pragma unroll
        for (int i = 0; i < kWidth; ++i) {
            if (m[i] == -INFINITY) {  // no rows were left: no key was seen, or only scores that are NaN
                sum += l[i];
                continue;
            }
            const float w = fast_exp2(m[i] - m_new);
            sum += w * l[i];
            acc += w * part[i];
        }
        top = m_new;
    }
    if (groups != 1u) {
        acc_of[threadIdx.x] = acc;
        ml_of[threadIdx.x] = make_float2(top, sum);
        __syncthreads();
        if (group != 0u || !live) return;
        for (uint32_t other = 1u; other < groups; ++other) {
            const float2 ml = ml_of[threadIdx.x + other * kThreads];
            if (ml.x == -INFINITY) {
                sum += ml.y;
                continue;
            }
            const float m_new = fmaxf(top, ml.x), keep = fast_exp2(top - m_new), w = fast_exp2(ml.x - m_new);
            sum = sum * keep + w * ml.y;
            acc = acc * keep + w * acc_of[threadIdx.x + other * kThreads];
            top = m_new;
        }
    }
    if (!live) return;
    const uint32_t token = token_of(p, row), head = (item % p.row_heads) * p.pack + (row - token * p.pack);
    publish((uint64_t)token * p.query_heads + head, d, acc, top, sum);
}

#endif  // YVEX_ROCM_KERNELS_RUN_MERGE_H
