// Key and value rows of EXACT_F32 attention split into halves, tile by tile (f16_split.h), for the walk of
// gqa_f32_halved.h.
#ifndef YVEX_ROCM_KERNELS_GQA_F32_HALVE_ROWS_H
#define YVEX_ROCM_KERNELS_GQA_F32_HALVE_ROWS_H

#include "../kernel_params.h"
#include "f16_split.h"
#include "mfma.h"

namespace {

// A tile in memory and in LDS: [K hi | K lo] and [V hi | V lo].
//   K: 16-byte units (octet of dims, key);  V: units (16 keys u, lane half, dim) of eight keys in the order of the
//   score registers: keys 16 u + 4 half + 0..3, then 16 u + 8 + 4 half + 0..3
template <int kDim>
struct HalvedTile {
    static constexpr int kKeys = 32;
    static constexpr float kKeyFactor = 128.f;  // of every key value (gqa_f32_halved.h)
    static constexpr int kPlane = kKeys * kDim * 2, kTensor = 2 * kPlane, kBytes = 2 * kTensor;

    // Where the unit of `dim` lies among those of its keys: lanes that write units four dims apart,
    // and lanes that read neighbouring ones, meet every bank once.
    __device__ static __forceinline__ int value_unit(int dim) { return dim ^ ((dim >> 4) & 3); }
};

// Splits the rows of one tile of one kv head: a workgroup of four waves, eight rows of K and eight of V each.
// Beside the tile it leaves the exponent of each eight values (past kExponentMost where one lies past the range).
// Bound by memory: 14.6 MB of rows in and as much out, 1777 tokens of 8 kv heads of 128.
template <int kDim>
struct HalveRows {
    typedef HalvedTile<kDim> Tile;
    static constexpr int kPieces = kDim / 32, kOctets = kDim / 64, kVLanes = kDim / 4;

    static __device__ __forceinline__ floatx4 load(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset)
    {
        return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)offset, 0, 0));
    }

    // The rows of a tensor from the first key of the tile on; rows past the last read as zero.
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const float *rows, uint64_t stride,
                                                                     uint64_t kv_tokens, uint64_t first,
                                                                     uint32_t kv_head)
    {
        const uint64_t bytes = ((kv_tokens - 1 - first) * stride + kDim) * 4;
        return __builtin_amdgcn_make_buffer_rsrc((void *)(rows + first * stride + (uint64_t)kv_head * kDim), 0,
                                                 (int)(uint32_t)min(bytes, (uint64_t)0xffffffffu), 0x00027000);
    }

    static __device__ __forceinline__ uint32_t wave_max(uint32_t v)
    {
        v = dpp_max<0x112>(dpp_max<0x111>(v));  // row_shr 1, 2, 4, 8: the last lane of a row has its largest
        v = dpp_max<0x118>(dpp_max<0x114>(v));
        v = dpp_max<0x143>(dpp_max<0x142>(v));  // row_bcast 15, 31
        return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
    }

    static __device__ __forceinline__ uint32_t bits_of(float v)
    {
        return __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
    }

    static __device__ __forceinline__ void halves(float x, float factor, _Float16 &hi, _Float16 &lo)
    {
        hi = (_Float16)(x * factor);
        lo = (_Float16)fmaf(x, factor, -(float)hi);
    }

    static __device__ void run(const yvex_rocm_gqa_f32_halved_params &p, unsigned char *lds)
    {
        const int lane = threadIdx.x & 63, quarter = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const uint32_t tile = blockIdx.x, kv_head = blockIdx.y;
        const uint64_t first = (uint64_t)tile * Tile::kKeys;
        const uint32_t k_row = (uint32_t)p.walk.k_stride * 4u, v_row = (uint32_t)p.walk.v_stride * 4u;
        const __amdgpu_buffer_rsrc_t keys = rows_of((const float *)p.walk.k, p.walk.k_stride, p.walk.kv_tokens,
                                                    first, kv_head);
        const __amdgpu_buffer_rsrc_t values = rows_of((const float *)p.walk.v, p.walk.v_stride, p.walk.kv_tokens,
                                                      first, kv_head);
        // lane (octet of dims, key) of K, lane (quad of dims, kPieces consecutive keys) of V
        floatx4 k[kPieces], v[kPieces];
        const uint32_t k_offset = (uint32_t)(8 * quarter + (lane & 7)) * k_row + (uint32_t)(lane >> 3) * 32u;
        const uint32_t v_offset = (uint32_t)(8 * quarter + lane / kVLanes * kPieces) * v_row +
                                  (uint32_t)(lane % kVLanes) * 16u;
#pragma unroll
        for (int j = 0; j < kPieces; ++j) k[j] = load(keys, k_offset + 256 * (j / 2) + 16 * (j % 2));
#pragma unroll
        for (int j = 0; j < kPieces; ++j) v[j] = load(values, v_offset + (uint32_t)j * v_row);
        uint32_t v_most = 0u;
#pragma unroll
        for (int j = 0; j < kPieces; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) v_most = max(v_most, bits_of(v[j][i]));
        v_most = wave_max(v_most);
        const uint32_t v_exponent = group_exponent(v_most);
        if (lane == 0) {
            uint32_t *words = p.factors + ((uint64_t)kv_head * p.kv_tiles + tile) * 8u;
            words[4 + quarter] = v_most >> 23 > kExponentMost ? kExponentMost + 1u : v_exponent;
        }
        const float v_factor = down_factor(v_exponent);
        unsigned char *k_unit = lds + ((lane >> 3) * 32 + 8 * quarter + (lane & 7)) * 16;
#pragma unroll
        for (int r = 0; r < kOctets; ++r) {
            halfx8 hi, lo;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                _Float16 h, l;
                halves(k[2 * r + j / 4][j % 4], Tile::kKeyFactor, h, l);
                hi[j] = h;
                lo[j] = l;
            }
            *reinterpret_cast<halfx8 *>(k_unit + r * 4096) = hi;
            *reinterpret_cast<halfx8 *>(k_unit + r * 4096 + Tile::kPlane) = lo;
        }
        // key 8 * quarter + from + j of the tile: u = quarter / 2, half (from + j) / 4, place
        // 4 * (quarter % 2) + (from + j) % 4 of the unit; as many keys of a unit as a lane has at a time
        const int from = lane / kVLanes * kPieces, dim = lane % kVLanes * 4;
        constexpr int kRun = kPieces < 4 ? kPieces : 4;
#pragma unroll
        for (int j0 = 0; j0 < kPieces; j0 += kRun)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = ((quarter >> 1) * 2 + ((from + j0) >> 2)) * kDim + Tile::value_unit(dim + i);
                unsigned char *unit = lds + Tile::kTensor + at * 16 + (quarter & 1) * 8 + ((from + j0) & 3) * 2;
#pragma unroll
                for (int j = 0; j < kRun; j += 2) {
                    _Float16 h[2], l[2];
                    halves(v[j0 + j][i], v_factor, h[0], l[0]);
                    halves(v[j0 + j + 1][i], v_factor, h[1], l[1]);
                    *reinterpret_cast<halfx2 *>(unit + 2 * j) = (halfx2){h[0], h[1]};
                    *reinterpret_cast<halfx2 *>(unit + 2 * j + Tile::kPlane) = (halfx2){l[0], l[1]};
                }
            }
        __syncthreads();
        unsigned char *out = p.tiles + ((uint64_t)kv_head * p.kv_tiles + tile) * Tile::kBytes;
#pragma unroll
        for (int i = 0; i < Tile::kBytes / 4096; ++i) {
            const int at = (i * 256 + (int)threadIdx.x) * 16;
            *reinterpret_cast<u32x4 *>(out + at) = *reinterpret_cast<const u32x4 *>(lds + at);
        }
    }
};

}  // namespace

#endif  // YVEX_ROCM_KERNELS_GQA_F32_HALVE_ROWS_H
