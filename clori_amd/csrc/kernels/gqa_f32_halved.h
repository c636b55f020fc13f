// EXACT_F32 attention over keys and values that were split into parts of 16 bits beforehand.
//
// The 16-bit matrix instructions do 16 times the fp32 one's work per cycle.  A product of two F32 values is three of
// f16 parts in the scores and six of bf16 parts in the update (the splitting of an operand into parts of fewer
// bits with F32 accumulation is a published method, Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", 2019).
//
// Scores.  An F32 value times a power of two as the sum of two f16 values, hi = its nearest and lo = the nearest of
// what hi leaves, a product as hi hi + hi lo + lo hi.  A key value is scaled by 2^7 whatever lies beside it, a query
// row by a power of two of its own.  Both halves together keep half an F32 last place of a value, but
// no less than 2^-25 after scaling: 2^-32 of a key value, 2^(x-39) of a query value where the row's largest lies in
// [2^x, 2^(x+1)).  What that can move a score by, in log2 units, is at most
//     2^-32 unit sum |q|  +  2^(x-39) unit 2^9 (query values below 2^(x-16)),    unit = scale log2(e),
// as a finite key value is below 2^9 (a larger one becomes infinite, hi and lo of opposite signs, and every
// score of it NaN).  A row for which either could exceed 2^-23 gets scores that are NaN.  N(0,1) rows stay
// below by 2^5.  A row of NaNs is walked in fp32.  So a score depends on its own query and key only, and a weight is
// off by 1e-7 of itself at most beside the roundings that a sum of F32 products has as well.
//
// Update.  A weight and a value as the sum of three bf16 values each, 24 bits at F32's range of exponents, and
// the six products of 2^-16 and more: off by 2^-23 of a product at most, however small or large its factors are
// (a weight below 2^-102 keeps 2^-126 of the row's largest).  With f16 halves here (three products, 122 us instead
// of 147 for 1777 tokens of 40/8 heads of 128) the weights had to carry the exponents of the values: beside a value
// of 2^30, or behind a sink of a weight of 1 and a value near zero, the other weights lost their bits.
//
// Against 64 bits, largest error of an element relative to sum w |v| of it, head dimensions 64 / 128 / 256 (fp32 walk):
// N(0,1) rows, other rows of 2^20 and 2^40 beside them unseen, 5.0e-7 / 6.4e-7 / 5.6e-7 (8.3e-7 / 1.1e-6 / 7.6e-7);
// such rows, channels and components seen 1.4e-6 / 1.4e-6 / 1.7e-6 (3.0e-6 / 2.4e-6 / 2.7e-6); behind sinks of 2^11
// to 2^23 times the other weights 3.9e-6 / 3.8e-6 / 6.5e-6 (7.4e-6 / 1.0e-5 / 1.2e-5).
//
// The splits are made once by a launch of their own (halve_rows) that leaves every tile of 32 keys as the walk wants
// it in LDS: the walk's tiles are filled by loads that write LDS directly, its registers
// hold no rows on their way, and a trip is bound by its MFMAs.  Items, packed rows and runs of keys are those of
// the bf16 prefill (kernel_params.h), with steps of 32 keys.
//
// What bounds the walk is power.  At 128 it runs at 1.52 to 1.57 GHz with the matrix cores busy 71 to 75 % of the
// cycles: 1777 tokens of 40/8 heads 131 of 140 us, 2048 tokens 165 of 175, 260 TFLOP/s of F32 products, 1.17 PFLOP/s
// of 16-bit ones, where a large bf16 product reaches 1.29 on this part.  At 256, one wave per SIMD, 1.91 GHz and
// 51 %: the first operands of a trip come behind its barrier (2048 tokens of 24/4 heads 231 of 240 us).
#ifndef YVEX_ROCM_KERNELS_GQA_F32_HALVED_H
#define YVEX_ROCM_KERNELS_GQA_F32_HALVED_H

#include "../kernel_params.h"
#include "f16_split.h"
#include "gqa_f32_again.h"
#include "gqa_f32_halve_rows.h"
#include "gqa_f32_walk.h"
#include "mfma.h"
#include "prefill_rows.h"

namespace {

// The walk.  A workgroup of four waves of 32 packed rows owns one item or one run of its keys.  Products are
// transposed (S^T = K Q^T, O^T += V^T P^T, 32x32x16), so a lane owns one row and 16 of a tile's 32
// keys, and the weights are the operand of the second product where they are.
//
// The trip of tile t is one sequence of slots, an MFMA each: first S^T of tile t+1, then the update
// with tile t; behind the MFMAs ride the loads of K(t+2) and V(t+1), the exponentials of tile t and their
// split, and the maximum of tile t+1.  An MFMA leaves room for about 24 cycles of vector work (whole
// instructions take 4 to 5, the exponential and the conversions 8 to 9), so a pair of weights is
// five steps of less than that.
template <int kDim>
struct GqaHalved {
    typedef HalvedTile<kDim> Tile;
    static constexpr int kBlocks = kDim / 32, kSteps = kDim / 16, kKeys = Tile::kKeys;
    static constexpr int kRows = YVEX_ROCM_PREFILL_ROWS, kPlane = Tile::kPlane;
    static constexpr int kKeyLoads = Tile::kKeyBytes / 4096;  // 1 KB loads per wave and K tile
    static constexpr int kValueLoads = Tile::kValueBytes / 4096;
    static constexpr int kScoreSlots = 3 * kSteps, kSlots = kScoreSlots + 6 * 2 * kBlocks;
    static constexpr int kLazy = 6;  // weights are at most 2^kLazy: a maximum is raised when it is exceeded by that
    static constexpr int kRing = 4;  // operands on their way from LDS

    struct Shared {
        __attribute__((aligned(16))) unsigned char k[2][Tile::kKeyBytes];
        __attribute__((aligned(16))) unsigned char v[2][Tile::kValueBytes];
    };

    const yvex_rocm_gqa_f32_halved_params &p;
    Shared &lds;
    const int lane, wave, column, half;
    uint32_t first_tile, tiles;      // of this workgroup's run
    int visible;                     // last key the lane's row sees, from the run's first on
    i32x4 rsrc;                      // the kv head's tiles
    uint32_t lds_base, k_unit, v_unit[2];
    halfx8 q_hi[kSteps], q_lo[kSteps];
    float q_factor;                  // of the lane's row: scores in log2 units per product as the MFMAs sum them
    floatx16 out[kBlocks];
    float top, neg_top, sum;         // the maximum that weights are relative to (log2 units), this half's denominator

    __device__ GqaHalved(const yvex_rocm_gqa_f32_halved_params &params, Shared &shared, int thread)
        : p(params), lds(shared), lane(thread & 63), wave(__builtin_amdgcn_readfirstlane(thread >> 6)),
          column(thread & 31), half((thread >> 5) & 1)
    {
    }

    // 1 KB load j of this wave for the K or V tile `tile` into buffer `buf`; tiles past the last are the
    // last once more, so that a trip has no branches.
    __device__ __forceinline__ void stage(uint32_t tile, uint32_t to, uint32_t at, uint32_t mine) const
    {
        lds_dma_b128(lds_base + to + mine, rsrc, (uint32_t)lane * 16u,
                     (uint32_t)__builtin_amdgcn_readfirstlane(
                         (int)((first_tile + min(tile, tiles - 1u)) * (uint32_t)Tile::kBytes + at + mine)));
    }
    __device__ __forceinline__ void stage_keys(uint32_t tile, int buf, int j) const
    {
        stage(tile, (uint32_t)(buf * Tile::kKeyBytes), 0u, (uint32_t)((wave * kKeyLoads + j) * 1024));
    }
    __device__ __forceinline__ void stage_values(uint32_t tile, int buf, int j) const
    {
        stage(tile, (uint32_t)(2 * Tile::kKeyBytes + buf * Tile::kValueBytes), (uint32_t)Tile::kKeyBytes,
              (uint32_t)((wave * kValueLoads + j) * 1024));
    }

    __device__ __forceinline__ u32x4 key_operand(int buf, int step, int plane) const
    {
        return *reinterpret_cast<const u32x4 *>(lds.k[buf] + k_unit + step * 1024 + plane * kPlane);
    }
    // operand m = u * kBlocks + block
    __device__ __forceinline__ u32x4 value_operand(int buf, int m, int plane) const
    {
        const int u = m / kBlocks, b = m % kBlocks;
        return *reinterpret_cast<const u32x4 *>(lds.v[buf] + v_unit[b & 1] + u * kDim * 32 + b * 512 +
                                                plane * kPlane);
    }
    // Operand n of a trip: lo and hi of the steps of S^T, hi of them once more, then the three planes of a step of the
    // update from the last on.
    template <int n>
    __device__ __forceinline__ u32x4 operand(int k_buf, int v_buf) const
    {
        if constexpr (n < 2 * kSteps) return key_operand(k_buf, n / 2, 1 - n % 2);
        else if constexpr (n < kScoreSlots) return key_operand(k_buf, n - 2 * kSteps, 0);
        else return value_operand(v_buf, (n - kScoreSlots) / 3, 2 - (n - kScoreSlots) % 3);
    }
    static constexpr int kOperands = kScoreSlots + 3 * 2 * kBlocks;

    // Step `part` (0, 1, 2) of the split of two F32 values into three bf16 values each: the nearest of what is left.
    __device__ static __forceinline__ uint32_t third(int part, float &a, float &b)
    {
        uint32_t pair = pack_bf16x2(a, b);
        if (part < 2) {
            a -= __builtin_bit_cast(float, pair << 16);
            b -= __builtin_bit_cast(float, pair & 0xffff0000u);
        }
        __asm__ volatile("" : "+v"(pair), "+v"(a), "+v"(b));
        return pair;
    }

    __device__ __forceinline__ void mask(floatx16 &s, uint32_t tile) const
    {
        int seen = visible - (int)(tile * kKeys) - 4 * half;
        __asm__ volatile("" : "+v"(seen));  // (the sixteen sums are not to be kept in registers)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 8 * (i / 4) + i % 4 <= seen ? s[i] : -INFINITY;
    }

    // the largest score
    __device__ static __forceinline__ float peak_of(const floatx16 &s)
    {
        float peak = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) peak = fmaxf(peak, s[i]);
        return peak;
    }
    // The largest of four and what came before, without fmaxf's canonical forms.  The compiler sees no
    // instructions here: the scores must have been complete for some MFMAs.
    __device__ static __forceinline__ void peak_step(const floatx16 &s, int g, float &peak)
    {
        __asm__ volatile("v_max3_f32 %0, %0, %1, %2\n\t"
                         "v_max3_f32 %0, %0, %3, %4"
                         : "+v"(peak)
                         : "v"(s[4 * g]), "v"(s[4 * g + 1]), "v"(s[4 * g + 2]), "v"(s[4 * g + 3]));
    }

    // Brings the maximum of the rows where a tile's peak (over both halves of a row) exceeds it by more than
    // 2^kLazy to that peak.  The other rows of the wave keep theirs, bit for bit: what a row gives
    // does not depend on the rows beside it.
    __device__ __forceinline__ void adjust(float peak)
    {
        const float raised = peak > top + (float)kLazy ? peak : top;
        // a row that has seen nothing yet keeps the maximum -inf
        const float keep = raised == -INFINITY ? 1.f : fast_exp2(top - raised);
        sum *= keep;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) out[b][i] *= keep;
        top = raised;
        neg_top = raised == -INFINITY ? 0.f : -raised;
    }

    // The trip of tile t; kAt = t % 2; `peak`: of tile t in this lane's half of its row (log2 units).
    template <int kAt>
    __device__ __forceinline__ void trip(uint32_t t, uint32_t wave_tiles, uint32_t unmasked, floatx16 &s_cur,
                                         floatx16 &s_next, float &peak)
    {
        constexpr int kNext = kAt ^ 1;
        // K(t+1) and V(t) have landed (this wave's loads, then everybody's); every wave is done with
        // K(t) and V(t-1)
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        __syncthreads();
        if (t >= wave_tiles) {
            // nothing of this tile is visible to the wave: it only keeps staging
#pragma unroll
            for (int j = 0; j < kKeyLoads; ++j) stage_keys(t + 2u, kAt, j);
#pragma unroll
            for (int j = 0; j < kValueLoads; ++j) stage_values(t + 1u, kNext, j);
            return;
        }
        u32x4 ring[kRing];
        for_each<kRing>([&](auto n) __attribute__((always_inline)) {
            ring[decltype(n)::value] = operand<decltype(n)::value>(kNext, kAt);
        });
        uint32_t weights[3][8];
        float part_sum = 0.f, next_peak = -INFINITY;
        bool raise = false;
        // the maximum of this tile's rows
        auto settle_step = [&](int k) __attribute__((always_inline)) {
            if (k == 0) peak = max_xor32(peak);
            if (k == 1) raise = __builtin_amdgcn_ballot_w64(peak > top + (float)kLazy) != 0ull;
        };
        // pair k / 5 of the weights: the two exponentials, then their parts
        auto weigh_step = [&](int k) __attribute__((always_inline)) {
            const int w = k / 5 * 2;
            if (k % 5 < 2) {
                float weight = fast_exp2(fmaf(s_cur[w + k % 5], q_factor, neg_top));
                part_sum += weight;
                __asm__ volatile("" : "+v"(weight), "+v"(part_sum));
                s_cur[w + k % 5] = weight;
            } else {
                float a = s_cur[w], b = s_cur[w + 1];
                weights[k % 5 - 2][k / 5] = third(k % 5 - 2, a, b);
                s_cur[w] = a;
                s_cur[w + 1] = b;
            }
        };
        constexpr int kSettled = 3;  // slots before the weights can be formed
        auto slot = [&](auto index) __attribute__((always_inline)) {
            constexpr int i = decltype(index)::value;
            if constexpr (i < kScoreSlots) {
                // lo hi and hi lo of all steps while the sum is small, then hi hi: a third of the roundings that count
                // (2-norm from 64 bits, 24/4 heads of 256: 100 tokens 2.9e-7 -> 2.0e-7, fp32 walk 2.7e-7; 1000 tokens
                // 4.4e-7 -> 3.3e-7, 4.6e-7; for an operand more to read a step, 119 -> 120 us)
                constexpr int m = i < 2 * kSteps ? i / 2 : i - 2 * kSteps;
                const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                s_next = mfma_32x32x16_f16(__builtin_bit_cast(halfx8, ring[i % kRing]),
                                           i < 2 * kSteps && i % 2 != 0 ? q_lo[m] : q_hi[m], i == 0 ? zero : s_next);
                ring[i % kRing] = operand<i + kRing>(kNext, kAt);
            } else {
                // value and weight parts 3 1, 2 2, 2 1, 1 3, 1 2, 1 1
                constexpr int m = (i - kScoreSlots) / 6, term = (i - kScoreSlots) % 6, first = m / kBlocks * 4;
                constexpr int plane = term == 0 ? 0 : term < 3 ? 1 : 2, n = kScoreSlots + 3 * m + plane;
                constexpr int part = term == 0 ? 0 : term < 3 ? 2 - term : 5 - term;
                const uint32_t(&w)[8] = weights[part];
                out[m % kBlocks] = mfma_32x32x16(as_bf16x8(ring[n % kRing]),
                                                 as_bf16x8((u32x4){w[first], w[first + 1], w[first + 2], w[first + 3]}),
                                                 out[m % kBlocks]);
                if constexpr ((term == 0 || term == 2 || term == 5) && n + kRing < kOperands)
                    ring[n % kRing] = operand<n + kRing>(kNext, kAt);
            }
            if constexpr (i < kKeyLoads) stage_keys(t + 2u, kAt, i);
            else if constexpr (i < kKeyLoads + kValueLoads) stage_values(t + 1u, kNext, i - kKeyLoads);
            ride<i, 2, 0, 2>(settle_step);
            // the first eight weights before the update's first MFMA, the others before its second half
            ride<i, 20, kSettled, kScoreSlots>(weigh_step);
            ride<i, 20, kScoreSlots, kScoreSlots + 6 * kBlocks - 1>(
                [&](int k) __attribute__((always_inline)) { weigh_step(20 + k); });
            ride<i, 4, kScoreSlots + 6 * kBlocks, kSlots>(
                [&](int g) __attribute__((always_inline)) { peak_step(s_next, g, next_peak); });
            __builtin_amdgcn_sched_barrier(0);
        };
        __builtin_amdgcn_sched_barrier(0);
        for_each<kSettled>(slot);
        if (raise) adjust(peak);
        __builtin_amdgcn_sched_barrier(0);
        for_each<kSlots, kSettled>(slot);
        sum += part_sum;
        if (t + 1u >= unmasked && t + 1u < wave_tiles) {
            mask(s_next, t + 1u);
            next_peak = peak_of(s_next);
        }
        peak = next_peak * q_factor;
    }

    // Steps of a kind, spread over slots [kFrom, kTo).
    template <int kSlot, int kCount, int kFrom, int kTo, typename F>
    __device__ static __forceinline__ void ride(const F &step)
    {
        for_each<kCount>([&](auto k) __attribute__((always_inline)) {
            if constexpr (kFrom + decltype(k)::value * (kTo - kFrom) / kCount == kSlot) step(decltype(k)::value);
        });
    }

    __device__ __forceinline__ void load_queries(const float *row)
    {
        floatx4 x[kSteps][2];
        float most = 0.f;
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int j = 0; j < 2; ++j) x[s][j] = *reinterpret_cast<const floatx4 *>(row + 16 * s + 4 * j);
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) most = fmaxf(most, fabsf(x[s][j / 4][j % 4]));
        const uint32_t e = row_exponent(__builtin_bit_cast(uint32_t, max_xor32(most)));
        const float up = up_factor(e), unit = p.scale * YVEX_LOG2E;  // 2^x / 2^14, a score's log2 units
        // (NaN where the halves' floors could move a score: the row is then not finite, and is walked in fp32)
        q_factor = up * (unit * (1.f / Tile::kKeyFactor));
        if (__builtin_amdgcn_ballot_w64(!(up * unit * (float)(kDim << 14) <= 128.f)) != 0ull) {
            float l1 = 0.f, tiny = 0.f;
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v = fabsf(x[s][j / 4][j % 4]);
                    l1 += v;
                    tiny += v != 0.f && v < 0.25f * up ? 1.f : 0.f;
                }
            if (!(sum_xor32(l1) * unit <= 512.f && sum_xor32(tiny) * up * unit <= 0x1p-7f))
                q_factor = __builtin_nanf("");
        }
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                split_pair_by_lane(x[s][j / 2][2 * (j % 2)], x[s][j / 2][2 * (j % 2) + 1], down_factor(e), hi[j],
                                   lo[j]);
            q_hi[s] = __builtin_bit_cast(halfx8, (u32x4){hi[0], hi[1], hi[2], hi[3]});
            q_lo[s] = __builtin_bit_cast(halfx8, (u32x4){lo[0], lo[1], lo[2], lo[3]});
        }
    }

    __device__ __forceinline__ void run()
    {
        const yvex_rocm_prefill_params &w = p.walk;
        uint32_t item = blockIdx.x, split = 0u;
        const bool partial = item >= w.whole_items;
        if (partial) {
            split = (item - w.whole_items) / w.tail_items;
            item = w.whole_items + (item - w.whole_items) % w.tail_items;
        } else if (item >= p.pair_units && item < 2u * p.pair_units) {
            // the second workgroup of a unit takes the second tier of items in reverse
            item = 3u * p.pair_units - 1u - item;
        }
        const uint32_t level = item / w.row_heads, row_head = item - level * w.row_heads;
        const uint32_t kv_head = kv_head_of(w, row_head);
        const uint32_t tile_row = (w.query_tiles - 1u - level) * kRows, tile_end = min(w.rows, tile_row + kRows);
        const uint32_t row0 = tile_row + (uint32_t)wave * 32u;
        auto last_of = [&](uint32_t row) {
            return w.causal ? min(w.kv_tokens, w.query_start + token_of(w, row) + 1u) : w.kv_tokens;
        };
        tiles = (last_of(tile_end - 1u) + kKeys - 1u) / kKeys;
        first_tile = 0u;
        if (partial) {
            const uint32_t per_split = (tiles + w.splits - 1u) / w.splits;
            first_tile = min(tiles, split * per_split);
            tiles = min(per_split, tiles - first_tile);
            if (tiles == 0u) first_tile = 0u;  // a run without steps
        }
        const int first_key = (int)(first_tile * kKeys);
        const bool wave_active = row0 < w.rows && tiles != 0u;
        const int wave_first_sees = (int)last_of(min(row0, w.rows - 1u)) - first_key;  // keys, as a count
        const int wave_last_sees = (int)last_of(min(row0 + 32u, w.rows) - 1u) - first_key;
        const uint32_t wave_tiles =
            wave_active && wave_last_sees > 0 ? min(tiles, (uint32_t)(wave_last_sees + kKeys - 1) / kKeys) : 0u;
        const uint32_t unmasked = wave_first_sees > 0 ? (uint32_t)wave_first_sees / kKeys : 0u;
        const uint32_t row = min(row0 + (uint32_t)column, w.rows - 1u), token = token_of(w, row);
        const uint32_t head = row_head * w.pack + (row - token * w.pack);
        visible = (int)last_of(row) - 1 - first_key;

        const uint64_t head_bytes = (uint64_t)p.kv_tiles * Tile::kBytes;
        rsrc = raw_buffer(p.tiles + kv_head * head_bytes, (uint32_t)head_bytes);
        lds_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address_of(lds.k[0]));
        k_unit = (uint32_t)(half * 32 + column) * 16u;
#pragma unroll
        for (int b = 0; b < 2; ++b)
            v_unit[b] = (uint32_t)((half * kDim + Tile::value_unit(32 * b + column)) * 16 - b * 512);
        top = -INFINITY;
        neg_top = 0.f;
        sum = 0.f;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) out[b][i] = 0.f;

        if (tiles != 0u) walk_tiles(wave_tiles, unmasked, (const float *)w.q + (uint64_t)token * w.q_stride +
                                                              (uint64_t)head * kDim + 8 * half);

        const bool own = row0 + (uint32_t)column < w.rows;
        sum = sum_xor32(sum);
        // (a run none of whose keys the row sees leaves a maximum of -inf and nothing)
        bool good = isfinite(sum) && (partial && top == -INFINITY ? sum == 0.f : sum > 0.f && isfinite(top));
        const float inverse = 1.0f / sum;
        if (!partial) {
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) out[b][i] = quotient(out[b][i], sum, inverse);
        }
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) good &= isfinite(out[b][i]);
        // the rows of every wave that are left to the fp32 walk, as bits: a word of each wave, behind the rows
        uint32_t *verdict = reinterpret_cast<uint32_t *>(lds.v[2]) - 4;
        const uint64_t bad = __builtin_amdgcn_ballot_w64(own && !good);
        const uint32_t failed = (uint32_t)bad | (uint32_t)(bad >> 32);
        __syncthreads();  // the tiles in LDS are done with
        lay_rows_down();
        if (lane == 0) verdict[wave] = failed;
        __syncthreads();
        const u32x4 verdicts = *reinterpret_cast<u32x4 *>(verdict);
        const uint32_t slot = partial ? (item - w.whole_items) * w.splits + split : 0u;
        const bool leave = own && half == 0 && (failed >> column & 1u) == 0u;
        if (row0 < w.rows && partial) {
            const uint64_t first = (uint64_t)slot * kRows + (row0 - tile_row);
            publish_rows(row0, failed, [&](uint32_t, uint32_t r) { return w.part_acc + (first + r) * kDim; });
            if (leave) {
                float *ml = w.part_ml + 2u * (first + (uint32_t)column);
                ml[0] = top;
                ml[1] = sum;
            }
        } else if (row0 < w.rows) {
            publish_rows(row0, failed, [&](uint32_t row_, uint32_t) {
                const uint32_t token_ = token_of(w, row_);
                return (float *)w.out +
                       ((uint64_t)token_ * w.query_heads + (row_head * w.pack + (row_ - token_ * w.pack))) * kDim;
            });
            if (leave && w.lse) w.lse[(uint64_t)token * w.query_heads + head] = top * YVEX_LN2 + logf(sum);
        }
        if ((verdicts[0] | verdicts[1] | verdicts[2] | verdicts[3]) != 0u) {
            __syncthreads();  // every wave is done with the rows and the verdicts
            local_bytes *shared = (local_bytes *)(void *)&lds;
            constant_params *arguments = (constant_params *)__builtin_amdgcn_kernarg_segment_ptr();
            walk_again<kDim>(arguments, shared, verdicts, partial, slot, row_head, tile_row, tile_end, first_tile,
                             tiles);
        }
    }

    // The wave's 32 rows go through its part of LDS, 16-byte units of a row dealt by its number so that
    // both sides spread over the banks.  They are laid down before the vote: kept in registers over it,
    // which the call of the fallback takes, they were spilled and fetched back, 5.4 us at the end of a
    // workgroup and 27 MB of scratch written (1777 tokens of 40 heads of 128).
    static constexpr uint32_t kUnits = kDim / 4;
    __device__ __forceinline__ floatx4 *laid_rows() const
    {
        static_assert(4 * 32 * kDim * 4 <= sizeof(Shared) - 16, "rows end before the verdicts");
        return reinterpret_cast<floatx4 *>(lds.k[0]) + (uint32_t)wave * 32u * kUnits;
    }
    __device__ __forceinline__ void lay_rows_down() const
    {
        floatx4 *rows = laid_rows();
#pragma unroll
        for (uint32_t b = 0; b < (uint32_t)kBlocks; ++b)
#pragma unroll
            for (uint32_t g = 0; g < 4; ++g)
                rows[(uint32_t)column * kUnits + ((8u * b + 2u * g + (uint32_t)half) ^ ((uint32_t)column & 15u))] =
                    (floatx4){out[b][4 * g], out[b][4 * g + 1], out[b][4 * g + 2], out[b][4 * g + 3]};
    }
    template <typename To>
    __device__ __forceinline__ void publish_rows(uint32_t row0, uint32_t failed, const To &to) const
    {
        const floatx4 *rows = laid_rows();
#pragma unroll
        for (uint32_t i = 0; i < kUnits / 2u; ++i) {
            const uint32_t r = (i * 64u + (uint32_t)lane) / kUnits, unit = (i * 64u + (uint32_t)lane) % kUnits;
            const floatx4 x = rows[r * kUnits + (unit ^ (r & 15u))];
            if (row0 + r < p.walk.rows && (failed >> r & 1u) == 0u)
                *reinterpret_cast<floatx4 *>(to(row0 + r, r) + 4u * unit) = x;
        }
    }

    __device__ __forceinline__ void walk_tiles(uint32_t wave_tiles, uint32_t unmasked, const float *query)
    {
#pragma unroll
        for (int j = 0; j < kKeyLoads; ++j) stage_keys(0u, 0, j);
#pragma unroll
        for (int j = 0; j < kKeyLoads; ++j) stage_keys(1u, 1, j);
#pragma unroll
        for (int j = 0; j < kValueLoads; ++j) stage_values(0u, 0, j);
        load_queries(query);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        __syncthreads();
        floatx16 s_even, s_odd;
#pragma unroll
        for (int i = 0; i < 16; ++i) s_even[i] = 0.f;
#pragma unroll
        for (int m = 0; m < kSteps; ++m) {
            s_even = mfma_32x32x16_f16(__builtin_bit_cast(halfx8, key_operand(0, m, 1)), q_hi[m], s_even);
            s_even = mfma_32x32x16_f16(__builtin_bit_cast(halfx8, key_operand(0, m, 0)), q_lo[m], s_even);
        }
#pragma unroll
        for (int m = 0; m < kSteps; ++m)
            s_even = mfma_32x32x16_f16(__builtin_bit_cast(halfx8, key_operand(0, m, 0)), q_hi[m], s_even);
        if (unmasked == 0u) mask(s_even, 0u);
        float peak = peak_of(s_even) * q_factor;
        // (two copies of a trip; a third for an odd last tile takes as long: 139 to 142 us at 1777 tokens of 128, 119
        // at 1000 of 256)
        for (uint32_t t = 0u;;) {
            trip<0>(t, wave_tiles, unmasked, s_even, s_odd, peak);
            if (++t == tiles) break;
            trip<1>(t, wave_tiles, unmasked, s_odd, s_even, peak);
            if (++t == tiles) break;
        }
        // nothing may still be in flight into LDS
        __builtin_amdgcn_s_waitcnt(0x0f70);
    }
};

}  // namespace

#endif  // YVEX_ROCM_KERNELS_GQA_F32_HALVED_H
