// EXACT_F32 attention tiles on the f16 matrix cores: every F32 product as three f16 products.
//
// An F32 value times a power of two is written as the sum of two f16 values, hi = its nearest and
// lo = the nearest of what hi leaves: 22 bits and a sign, and x y = hi hi + hi lo + lo hi up to
// 2^-22 of it, less than what an F32 accumulation of such products rounds away.  The f16 matrix
// instruction does 16 times the fp32 one's work per cycle, so three of them take 3/16 of its time.
// Powers of two bring the values into f16's range: a query row (its part of the head dimension), and
// each group of eight key or value rows of a tile, has its own, chosen so that its largest magnitude
// lies in [2^14, 2^15); a value 2^-k of the largest keeps 2^-23 of itself up to k = 16, and 2^-39 of the
// largest below that.  The distance from 64 bits is smaller than that of the fp32 MFMA walk (fewer
// roundings on the way to a sum): 3.2e-7 in the 2-norm where that has 5.2e-7 (1777 tokens, 40/8 heads of 128,
// N(0,1) rows).  The factors of the keys go into the factor that the scores take anyway, the
// factors of the values into the weights as they are split.
#ifndef YVEX_ROCM_KERNELS_GQA_F32_HALVES_H
#define YVEX_ROCM_KERNELS_GQA_F32_HALVES_H

#include "../kernel_params.h"
#include "f16_split.h"
#include "gqa_f32_walk.h"
#include "mfma.h"

namespace {

// One workgroup = one item: 128 consecutive query tokens of one query head, a team of four waves of 32
// queries (kParts = 1), or two teams that split the head dimension (kParts = 2, head dimension
// 256): waves w and w + 4 share 32 queries, each computes what its kPartDim dimensions contribute to the
// scores, the parts are exchanged through LDS, and each accumulates its own part of the output.
//
// Products are transposed (S^T = K Q^T, O^T += V^T P^T, 32x32x16), so a lane owns one query column
// and 16 of a tile's 32 keys, and the weights are the operand of the second product where they are.
// Key and value rows are fetched into registers, split there (each wave eight rows of a tile) and
// written to LDS as operands: 16-byte units of eight halves that lie as the lanes read them.
//
// The trip of tile t is one pipelined sequence of slots, an MFMA each: first S^T of tile t+1, then
// the update with tile t, with everything else riding behind them: the exponentials of tile t and their
// split, the split of K(t+2) and V(t+1), the maximum of tile t+1.  What bounds it is the vector work beside
// the MFMAs (48 of 32 cycles each): about 1700 cycles of a trip at 128, half of them the splits, each of
// which every workgroup makes for itself.  Fp32 MFMA walk / this one, us: 1777 tokens of 40/8 heads
// of 128 313 / 150 (215 TFLOP/s), 300 behind 5000 774 / 316; 2000 of 16/4 of 64 167 / 80; 1000 of 24/4 of
// 256 297 / 130, 333 behind 2222 716 / 275.
template <int kPartDim, int kParts>
struct GqaHalves {
    static constexpr int kDim = kPartDim * kParts, kBlocks = kPartDim / 32, kSteps = kPartDim / 16;
    static constexpr int kKeys = 32, kQueries = 128;
    static constexpr int kPlane = kKeys * kPartDim * 2;  // bytes of one half (hi or lo) of a team's K or V tile
    static constexpr int kTile = 2 * kPlane;             // hi, then lo
    static constexpr int kValueStages = kParts == 1 ? 2 : 1;
    static constexpr int kPieces = kPartDim / 32;        // 16-byte pieces of a K (or V) tile per lane
    static constexpr int kOctets = kPartDim / 64;        // units of K per lane
    static constexpr int kVLanes = kPartDim / 4;         // lanes side by side on a value row
    static constexpr int kExchange = 64 * 16 * 4;        // what one wave hands its partner of the other team
    static constexpr int kHalfSlots = 3 * kSteps, kSlots = 2 * kHalfSlots;
    // weights are at most 2^kLazy (a maximum is raised when it is exceeded by that), so times
    // 2^kWeightShift they stay inside f16
    static constexpr int kLazy = 6, kWeightShift = 15 - kLazy;
    // steps of a split: the largest magnitude, its exponent, the halves
    static constexpr int kReduceSteps = 3, kSplitSteps = kPieces + kReduceSteps + 2 * kPieces;

    struct Shared {
        // K: units (octet of dims, key);  V: units (16 keys u, lane half, dim) of eight keys in the order
        // of the score registers, swizzled (value_unit)
        __attribute__((aligned(16))) unsigned char k[2][kParts][kTile];
        __attribute__((aligned(16))) unsigned char v[kValueStages][kParts][kTile];
        __attribute__((aligned(16))) unsigned char exchange[kParts == 1 ? 16 : 8 * kExchange];
        __attribute__((aligned(16))) float key_factor[2][kParts][4];  // per group of eight keys
        __attribute__((aligned(16))) uint32_t value_exponent[kValueStages][kParts][4];
        uint32_t failed;
    };

    const yvex_rocm_gqa_f32_params &p;
    Shared &lds;
    const int lane, wave, column, half, quarter, part;

    // the rows of a tensor that are still to be fetched
    struct Cursor {
        uint64_t at, left;  // address and bytes
        uint64_t tile;      // bytes from tile to tile
    };
    Cursor k_cursor, v_cursor;
    uint32_t k_offset, v_offset, v_row;     // of this lane's pieces in a tile
    uint32_t k_unit, v_unit[2], v_place;    // this lane's units: K operand, V operand of even and odd blocks, V split
    halfx8 q_hi[kSteps], q_lo[kSteps];
    float q_factor;
    floatx16 out[kBlocks];
    float top, neg_top, sum;   // the maximum that weights are relative to (log2 units), this half's denominator
    int reference;             // the exponent that the accumulators are relative to
    bool extreme;
    int visible;               // last key this lane's query sees
    floatx4 piece[kPieces];    // K or V on its way

    __device__ GqaHalves(const yvex_rocm_gqa_f32_params &params, Shared &shared, int thread)
        : p(params), lds(shared), lane(thread & 63), wave(__builtin_amdgcn_readfirstlane(thread >> 6)),
          column(thread & 31), half((thread >> 5) & 1), quarter(wave & 3), part(wave >> 2)
    {
    }

    __device__ __forceinline__ Cursor rows_of(const float *rows, uint64_t stride, uint64_t kv_head) const
    {
        Cursor c;
        c.at = (uint64_t)(uintptr_t)(rows + kv_head * kDim);
        c.left = ((p.kv_tokens - 1) * stride + kDim) * 4;
        c.tile = kKeys * stride * 4;
        return c;
    }

    // The descriptor of the next tile; rows past the last read as zero.
    __device__ static __forceinline__ __amdgpu_buffer_rsrc_t advance(Cursor &c)
    {
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(uintptr_t)c.at, 0, (int)(uint32_t)min(c.left, (uint64_t)0xffffffffu), 0x00027000);
        c.at += c.tile;
        c.left -= min(c.left, c.tile);
        return rsrc;
    }

    // A wave takes eight key rows of a tile: lane (octet of dims, key), so that its units are written side by
    // side; and eight value rows: lane (quad of dims, kPieces consecutive keys).
    __device__ __forceinline__ void fetch_keys()
    {
        const __amdgpu_buffer_rsrc_t rsrc = advance(k_cursor);
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
            piece[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                rsrc, (int)(k_offset + 256 * (j / 2) + 16 * (j % 2)), 0, 0));
    }
    __device__ __forceinline__ void fetch_values()
    {
        const __amdgpu_buffer_rsrc_t rsrc = advance(v_cursor);
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
            piece[j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                rsrc, (int)(v_offset + (uint32_t)j * v_row), 0, 0));
    }

    // The split of the pieces in steps that ride behind the MFMAs of a trip.
    struct Split {
        float factor;
        uint32_t most, exponent;
        uint32_t hi[4], lo[4];
    };

    __device__ __forceinline__ void measure_step(int k, Split &s)
    {
        if (k < kPieces) {
            const uint32_t a = largest(piece[k][0], piece[k][1], piece[k][2]);
            s.most = largest(piece[k][3], __builtin_bit_cast(float, a),
                             k == 0 ? 0.f : __builtin_bit_cast(float, s.most));
        } else if (k == kPieces) {
            // (two wait states between the assembly above and a lane exchange, which the compiler cannot see)
            __asm__ volatile("s_nop 1" : "+v"(s.most));
            s.most = dpp_max<0x112>(dpp_max<0x111>(s.most));  // row_shr 1, 2
        } else if (k == kPieces + 1) {
            s.most = dpp_max<0x118>(dpp_max<0x114>(s.most));  // row_shr 4, 8: the last lane of a row has its largest
        } else {
            s.most = dpp_max<0x143>(dpp_max<0x142>(s.most));  // row_bcast 15, 31
            const uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)s.most, 63);
            s.exponent = group_exponent(bits);
            extreme |= bits >> 23 > kExponentMost;
            s.factor = down_factor(s.exponent);
        }
        __asm__ volatile("" : "+v"(s.most));
    }

    __device__ __forceinline__ void keys_step(int k, int stage, Split &s)
    {
        if (k < kPieces + kReduceSteps) return measure_step(k, s);
        k -= kPieces + kReduceSteps;  // two of the lane's values
        const floatx4 &x = piece[k / 2];
        split_pair(x[2 * (k % 2)], x[2 * (k % 2) + 1], s.factor, s.hi[k % 4], s.lo[k % 4]);
        if (k % 4 != 3) return;
        unsigned char *unit = lds.k[stage][part] + ((lane >> 3) * 32 + 8 * quarter + (lane & 7)) * 16 + k / 4 * 4096;
        *reinterpret_cast<u32x4 *>(unit) = (u32x4){s.hi[0], s.hi[1], s.hi[2], s.hi[3]};
        *reinterpret_cast<u32x4 *>(unit + kPlane) = (u32x4){s.lo[0], s.lo[1], s.lo[2], s.lo[3]};
        if (k == 2 * kPieces - 1 && lane == 0) lds.key_factor[stage][part][quarter] = up_factor(s.exponent);
    }

    // Where the unit of `dim` lies among those of its keys: lanes that write units four dims apart,
    // and lanes that read neighbouring ones, meet every bank once.
    __device__ static __forceinline__ int value_unit(int dim) { return dim ^ ((dim >> 4) & 3); }

    __device__ __forceinline__ void values_step(int k, int stage, Split &s)
    {
        if (k < kPieces + kReduceSteps) return measure_step(k, s);
        k -= kPieces + kReduceSteps;  // two of the lane's keys, of one dim
        constexpr int pairs = kPieces / 2;
        const int i = k / pairs, j = 2 * (k % pairs);
        split_pair(piece[j][i], piece[j + 1][i], s.factor, s.hi[k % pairs], s.lo[k % pairs]);
        if (k % pairs != pairs - 1) return;
        unsigned char *unit = lds.v[stage][part] + (v_place ^ (uint32_t)(i * 16));
        if constexpr (pairs == 2) {
            *reinterpret_cast<u32x2 *>(unit) = (u32x2){s.hi[0], s.hi[1]};
            *reinterpret_cast<u32x2 *>(unit + kPlane) = (u32x2){s.lo[0], s.lo[1]};
        } else {
            *reinterpret_cast<uint32_t *>(unit) = s.hi[0];
            *reinterpret_cast<uint32_t *>(unit + kPlane) = s.lo[0];
        }
        if (k == 2 * kPieces - 1 && lane == 0) lds.value_exponent[stage][part][quarter] = s.exponent;
    }

    __device__ __forceinline__ void split_keys(int stage)
    {
        Split s = {};
#pragma unroll
        for (int k = 0; k < kSplitSteps; ++k) keys_step(k, stage, s);
    }
    __device__ __forceinline__ void split_values(int stage)
    {
        Split s = {};
#pragma unroll
        for (int k = 0; k < kSplitSteps; ++k) values_step(k, stage, s);
    }

    __device__ __forceinline__ halfx8 key_operand(int stage, int step, int plane) const
    {
        return *reinterpret_cast<const halfx8 *>(lds.k[stage][part] + k_unit + step * 1024 + plane * kPlane);
    }
    // operand m = u * kBlocks + block
    __device__ __forceinline__ halfx8 value_operand(int stage, int m, int plane) const
    {
        const int u = m / kBlocks, b = m % kBlocks;
        return *reinterpret_cast<const halfx8 *>(lds.v[stage][part] + v_unit[b & 1] + u * kPartDim * 32 + b * 512 +
                                                 plane * kPlane);
    }

    __device__ __forceinline__ void mask(floatx16 &s, uint32_t tile) const
    {
        const int seen = visible - (int)(tile * kKeys);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 8 * (i / 4) + 4 * half + i % 4 <= seen ? s[i] : -INFINITY;
    }

    // the largest of four scores, with what came before
    __device__ static __forceinline__ float peak_of(const floatx16 &s, const floatx4 &factor, int g, float peak)
    {
        const float m = fmaxf(fmaxf(fmaxf(s[4 * g], s[4 * g + 1]), s[4 * g + 2]), s[4 * g + 3]);
        return fmaxf(peak, kParts == 1 ? m * factor[g] : m);
    }

    // Raises the maximum when a tile's exceeds it by more than 2^kLazy.
    __device__ __forceinline__ void settle(float peak)
    {
        peak = max_xor32(peak);
        if (__builtin_amdgcn_ballot_w64(peak > top + (float)kLazy) != 0ull) {
            // key 0 is visible to every query, so the maximum is finite from the first tile on
            const float raised = fmaxf(top, peak), keep = fast_exp2(top - raised);
            sum *= keep;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) out[b][i] *= keep;
            top = raised;
            neg_top = -raised;
        }
    }

    // scores of one tile from the K stage, as the partner's part is to be added (kParts = 2) in log2 units
    __device__ __forceinline__ void hand_over(const floatx16 &s) const
    {
        unsigned char *mine = lds.exchange + wave * kExchange + lane * 16;
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<floatx4 *>(mine + g * 1024) =
                (floatx4){s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
    }
    __device__ __forceinline__ void take_over(floatx16 &s, int g) const
    {
        const floatx4 other =
            *reinterpret_cast<const floatx4 *>(lds.exchange + (wave ^ 4) * kExchange + lane * 16 + g * 1024);
#pragma unroll
        for (int r = 0; r < 4; ++r) s[4 * g + r] += other[r];
    }

    // The trip of tile t; kAt = t % 2.
    template <int kAt>
    __device__ __forceinline__ void trip(uint32_t t, uint32_t wave_tiles, uint32_t unmasked, floatx16 &s_cur,
                                         floatx16 &s_next, floatx4 &f_cur, floatx4 &f_next)
    {
        constexpr int kNext = kAt ^ 1, kVAt = kParts == 1 ? kAt : 0, kVNext = kParts == 1 ? kNext : 0;
        // K(t+1) and V(t) are in LDS, every wave is done with K(t) and V(t-1)
        __syncthreads();
        if (t >= wave_tiles) {
            // nothing of this tile is visible to the wave: it only keeps staging
            if constexpr (kParts == 1) {
                split_keys(kAt);
                fetch_values();
                split_values(kVNext);
                fetch_keys();
            } else {
                split_values(kVAt);
                fetch_keys();
                __syncthreads();
                split_keys(kAt);
                fetch_values();
            }
            return;
        }
        const floatx4 factors = *reinterpret_cast<const floatx4 *>(lds.key_factor[kNext][part]);
        halfx8 hi[2], lo[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            lo[k] = key_operand(kNext, k, 1);
            hi[k] = key_operand(kNext, k, 0);
        }
        float weight_factor[4];
        auto weigh_values = [&]() __attribute__((always_inline)) {
            const u32x4 exponents = *reinterpret_cast<const u32x4 *>(lds.value_exponent[kVAt][part]);
            int e[4], most = 0;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                e[g] = __builtin_amdgcn_readfirstlane((int)exponents[g]);
                most = max(most, e[g]);
            }
            if (most > reference) {
                // one power of two of room, so that the accumulators seldom move
                const int raised = most + 1;
#pragma unroll
                for (int b = 0; b < kBlocks; ++b)
#pragma unroll
                    for (int i = 0; i < 16; ++i) out[b][i] = __builtin_amdgcn_ldexpf(out[b][i], reference - raised);
                reference = raised;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g)
                weight_factor[g] = power_of_two((uint32_t)max(127 + kWeightShift + e[g] - reference, 0));
        };
        if constexpr (kParts == 1) weigh_values();
        f_next = factors * q_factor;

        uint32_t p_hi[8], p_lo[8];
        float part_sum = 0.f, peak = -INFINITY;
        Split split = {};
        // a weight and, with every second, their halves
        auto weigh_step = [&](int e) __attribute__((always_inline)) {
            const float x = kParts == 1 ? fmaf(s_cur[e], f_cur[e / 4], neg_top) : s_cur[e] + neg_top;
            s_cur[e] = fast_exp2(x);
            part_sum += s_cur[e];
            if (e & 1) {
                // (behind the sum: the exponential's result has been read once)
                __asm__ volatile("" : "+v"(s_cur[e]), "+v"(part_sum));
                split_pair(s_cur[e - 1], s_cur[e], weight_factor[e / 4], p_hi[e / 2], p_lo[e / 2]);
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        for_each<kSlots>([&](auto slot) __attribute__((always_inline)) {
            constexpr int i = decltype(slot)::value;
            constexpr int m = (i % kHalfSlots) / 3, term = i % 3;
            if constexpr (i < kHalfSlots) {
                const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                s_next = mfma_32x32x16_f16(term == 0 ? lo[m % 2] : hi[m % 2], term == 1 ? q_lo[m] : q_hi[m],
                                           i == 0 ? zero : s_next);
            } else {
                constexpr int first = m / kBlocks * 4;
                u32x4 words;
                if constexpr (term == 1)
                    words = (u32x4){p_lo[first], p_lo[first + 1], p_lo[first + 2], p_lo[first + 3]};
                else
                    words = (u32x4){p_hi[first], p_hi[first + 1], p_hi[first + 2], p_hi[first + 3]};
                out[m % kBlocks] = mfma_32x32x16_f16(term == 0 ? lo[m % 2] : hi[m % 2],
                                                     __builtin_bit_cast(halfx8, words), out[m % kBlocks]);
            }
            // the operands two steps on: of K, then of V
            if constexpr (term != 1) {
                constexpr int n = m + 2 + (i < kHalfSlots ? 0 : kSteps);
                if constexpr (n < kSteps)
                    (term == 0 ? lo : hi)[m % 2] = key_operand(kNext, n, term == 0);
                else if constexpr (n < 2 * kSteps && (kParts == 1 || i >= kHalfSlots))
                    (term == 0 ? lo : hi)[m % 2] = value_operand(kVAt, n - kSteps, term == 0);
            }
            // steps of a kind, spread over a range of slots
            auto ride = [&](auto steps, auto from, auto to, const auto &step) __attribute__((always_inline)) {
                constexpr int count = decltype(steps)::value, begin = decltype(from)::value, end = decltype(to)::value;
                for_each<count>([&](auto k) __attribute__((always_inline)) {
                    if constexpr (begin + decltype(k)::value * (end - begin) / count == i) step(decltype(k)::value);
                });
            };
            auto peak_step = [&](int g) __attribute__((always_inline)) {
                if constexpr (kParts == 2) take_over(s_next, g);
                peak = peak_of(s_next, f_next, g, peak);
                __asm__ volatile("" : "+v"(peak));
            };
            constexpr int kQuarter = kHalfSlots / 4;
            if constexpr (kParts == 1) {
                ride(Index<8>(), Index<0>(), Index<2 * kQuarter>(), weigh_step);
                ride(Index<kSplitSteps>(), Index<kQuarter>(), Index<kHalfSlots>(),
                     [&](int k) __attribute__((always_inline)) { keys_step(k, kAt, split); });
                if constexpr (i == kHalfSlots) fetch_values();
                ride(Index<8>(), Index<3 * kQuarter>(), Index<6 * kQuarter>(),
                     [&](int k) __attribute__((always_inline)) { weigh_step(8 + k); });
                ride(Index<4>(), Index<5 * kQuarter>(), Index<6 * kQuarter>(), peak_step);
                ride(Index<kSplitSteps>(), Index<6 * kQuarter>(), Index<kSlots>(),
                     [&](int k) __attribute__((always_inline)) { values_step(k, kVNext, split); });
            } else {
                ride(Index<kSplitSteps>(), Index<0>(), Index<kHalfSlots>(),
                     [&](int k) __attribute__((always_inline)) { values_step(k, kVAt, split); });
                if constexpr (i == kHalfSlots - 1) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) s_next[r] *= f_next[r / 4];
                    hand_over(s_next);
                    fetch_keys();
                    __syncthreads();  // the parts of the scores, and V(t)
                    weigh_values();
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        lo[k] = value_operand(kVAt, k, 1);
                        hi[k] = value_operand(kVAt, k, 0);
                    }
#pragma unroll
                    for (int k = 0; k < 8; ++k) weigh_step(k);
                    // (between the assembly of the split and the MFMA that reads its result)
                    __asm__ volatile("s_nop 1" : "+v"(p_hi[3]), "+v"(p_lo[3]));
                }
                ride(Index<8>(), Index<4 * kQuarter>(), Index<6 * kQuarter>(),
                     [&](int k) __attribute__((always_inline)) { weigh_step(8 + k); });
                ride(Index<4>(), Index<5 * kQuarter>(), Index<6 * kQuarter>(), peak_step);
                ride(Index<kSplitSteps>(), Index<6 * kQuarter>(), Index<kSlots>(),
                     [&](int k) __attribute__((always_inline)) { keys_step(k, kAt, split); });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (kParts == 1) fetch_keys();
        else fetch_values();
        sum += part_sum;
        if (t + 1 < wave_tiles) {
            if (t + 1 >= unmasked) {
                mask(s_next, t + 1);
                peak = -INFINITY;
#pragma unroll
                for (int g = 0; g < 4; ++g) peak = peak_of(s_next, f_next, g, peak);
            }
            settle(peak);
        }
    }

    // One item.  False when some result is not finite or an input lies outside the range: then
    // nothing was stored and the item is to be walked in fp32.  Every wave gets the same answer.
    __device__ __forceinline__ bool item(uint64_t id)
    {
        if (((p.k_stride | p.v_stride) >> 24) != 0) return false;  // a tile's rows span 4 GiB
        const uint64_t tiles_q = (p.query_tokens + kQueries - 1) / kQueries;
        const uint64_t head = id % p.query_heads;
        const uint64_t q_tile = tiles_q - 1 - id / p.query_heads;
        const uint64_t kv_head = head / (p.query_heads / p.kv_heads);
        const uint64_t q0 = q_tile * kQueries + (uint64_t)quarter * 32u;
        // rows past the last query repeat it: they compute, they are not stored
        const uint64_t token = min(q0 + (uint64_t)column, p.query_tokens - 1);
        const uint64_t group_last =
            p.causal ? min(p.kv_tokens, p.query_start + min((q_tile + 1) * kQueries, p.query_tokens)) : p.kv_tokens;
        const uint64_t wave_last =
            p.causal ? min(p.kv_tokens, p.query_start + min(q0 + 32u, p.query_tokens)) : p.kv_tokens;
        const uint32_t tiles = (uint32_t)((group_last + kKeys - 1) / kKeys);
        const uint32_t wave_tiles = q0 < p.query_tokens ? (uint32_t)((wave_last + kKeys - 1) / kKeys) : 0u;
        // tiles whose keys every query of the wave sees
        const uint32_t unmasked = (last_visible(p, p.query_start + min(q0, p.query_tokens - 1)) + 1u) / kKeys;
        visible = (int)last_visible(p, p.query_start + token);
        extreme = false;
        reference = 0;
        top = -INFINITY;
        neg_top = 0.f;
        sum = 0.f;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) out[b][i] = 0.f;

        k_cursor = rows_of(p.k, p.k_stride, kv_head);
        v_cursor = rows_of(p.v, p.v_stride, kv_head);
        v_row = (uint32_t)p.v_stride * 4u;
        k_offset = (uint32_t)(8 * quarter + (lane & 7)) * (uint32_t)p.k_stride * 4u +
                   (uint32_t)(part * kPartDim * 4 + (lane >> 3) * 32);
        v_offset = (uint32_t)(8 * quarter + lane / kVLanes * kPieces) * v_row +
                   (uint32_t)(part * kPartDim * 4 + lane % kVLanes * 16);
        k_unit = (uint32_t)(half * 32 + column) * 16u;
#pragma unroll
        for (int b = 0; b < 2; ++b)
            v_unit[b] = (uint32_t)((half * kPartDim + value_unit(32 * b + column)) * 16 - b * 512);
        {
            // key 8 * quarter + first + j of the tile: u = quarter / 2, half (first + j) / 4, place
            // 4 * (quarter % 2) + (first + j) % 4 of the unit
            const int first = lane / kVLanes * kPieces, dim = lane % kVLanes * 4;
            v_place = (uint32_t)((((quarter >> 1) * 2 + (first >> 2)) * kPartDim + value_unit(dim)) * 16 +
                                 (quarter & 1) * 8 + (first & 3) * 2);
        }
        // this lane's dims of its query row: 16 step + 8 half + j of the part
        fetch_keys();
        {
            const float *row = p.q + token * p.q_stride + head * kDim + part * kPartDim + 8 * half;
            float most = 0.f;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const floatx4 a = *reinterpret_cast<const floatx4 *>(row + 16 * s);
                const floatx4 b = *reinterpret_cast<const floatx4 *>(row + 16 * s + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) most = fmaxf(most, fmaxf(fabsf(a[j]), fabsf(b[j])));
            }
            const uint32_t bits = __builtin_bit_cast(uint32_t, max_xor32(most)), e = group_exponent(bits);
            extreme |= bits >> 23 > kExponentMost;
            q_factor = up_factor(e) * (p.scale * YVEX_LOG2E);
            // (read a second time: the registers are short)
            __asm__ volatile("" : "+v"(row));
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const floatx4 a = *reinterpret_cast<const floatx4 *>(row + 16 * s);
                const floatx4 b = *reinterpret_cast<const floatx4 *>(row + 16 * s + 4);
                u32x4 hi, lo;
                uint32_t h[4], l[4];
                split_pair_by_lane(a[0], a[1], down_factor(e), h[0], l[0]);
                split_pair_by_lane(a[2], a[3], down_factor(e), h[1], l[1]);
                split_pair_by_lane(b[0], b[1], down_factor(e), h[2], l[2]);
                split_pair_by_lane(b[2], b[3], down_factor(e), h[3], l[3]);
                hi = (u32x4){h[0], h[1], h[2], h[3]};
                lo = (u32x4){l[0], l[1], l[2], l[3]};
                q_hi[s] = __builtin_bit_cast(halfx8, hi);
                q_lo[s] = __builtin_bit_cast(halfx8, lo);
            }
        }

        // K(0), K(1) and V(0) in place, K(2) (or V(0)) on its way, the scores of tile 0
        if (lane == 0 && wave == 0) lds.failed = 0u;
        split_keys(0);
        if constexpr (kParts == 1) {
            fetch_values();
            split_values(0);
        }
        fetch_keys();
        split_keys(1);
        if constexpr (kParts == 1) fetch_keys();
        else fetch_values();
        __syncthreads();
        floatx16 s_even, s_odd;
        floatx4 f_even, f_odd;
        f_even = *reinterpret_cast<const floatx4 *>(lds.key_factor[0][part]) * q_factor;
#pragma unroll
        for (int i = 0; i < 16; ++i) s_even[i] = 0.f;
#pragma unroll
        for (int m = 0; m < kSteps; ++m) {
            const halfx8 lo = key_operand(0, m, 1), hi = key_operand(0, m, 0);
            s_even = mfma_32x32x16_f16(lo, q_hi[m], s_even);
            s_even = mfma_32x32x16_f16(hi, q_lo[m], s_even);
            s_even = mfma_32x32x16_f16(hi, q_hi[m], s_even);
        }
        if constexpr (kParts == 2) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s_even[r] *= f_even[r / 4];
            hand_over(s_even);
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 4; ++g) take_over(s_even, g);
        }
        if (wave_tiles != 0u) {
            if (unmasked == 0u) mask(s_even, 0u);
            float peak = -INFINITY;
#pragma unroll
            for (int g = 0; g < 4; ++g) peak = peak_of(s_even, f_even, g, peak);
            settle(peak);
        }

        uint32_t t = 0u;
        for (; t + 1u < tiles; t += 2u) {
            trip<0>(t, wave_tiles, unmasked, s_even, s_odd, f_even, f_odd);
            trip<1>(t + 1u, wave_tiles, unmasked, s_odd, s_even, f_odd, f_even);
        }
        if (t < tiles) trip<0>(t, wave_tiles, unmasked, s_even, s_odd, f_even, f_odd);

        // the accumulators are relative to 2^(reference - 127), weights to 2^kWeightShift and values to 2^14
        const bool own = q0 + (uint64_t)column < p.query_tokens;
        sum = sum_xor32(sum);
        const float inverse = 1.0f / sum;
        bool good = sum > 0.f && isfinite(sum) && isfinite(top);
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                out[b][i] = __builtin_amdgcn_ldexpf(quotient(out[b][i], sum, inverse),
                                                    reference - (141 + kWeightShift));
                good &= isfinite(out[b][i]);
            }
        if (extreme || (own && !good)) lds.failed = 1u;
        __syncthreads();
        if (lds.failed != 0u) return false;
        if (!own) return true;
        float *row = p.out + (token * p.query_heads + head) * kDim + part * kPartDim;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<floatx4 *>(row + 32 * b + 8 * g + 4 * half) =
                    (floatx4){out[b][4 * g], out[b][4 * g + 1], out[b][4 * g + 2], out[b][4 * g + 3]};
        if (p.lse && half == 0 && part == 0) p.lse[token * p.query_heads + head] = top * YVEX_LN2 + logf(sum);
        return true;
    }
};

}  // namespace

#endif  // YVEX_ROCM_KERNELS_GQA_F32_HALVES_H
