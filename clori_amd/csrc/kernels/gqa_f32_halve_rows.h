// Key and value rows of EXACT_F32 attention split into 16-bit parts, tile by tile, for the walk of
// gqa_f32_halved.h.
#ifndef YVEX_ROCM_KERNELS_GQA_F32_HALVE_ROWS_H
#define YVEX_ROCM_KERNELS_GQA_F32_HALVE_ROWS_H

#include "../kernel_params.h"
#include "f16_split.h"
#include "mfma.h"

namespace {

// A tile in memory and in LDS: [K hi | K lo], f16, and [V 1 | V 2 | V 3], bf16.
//   K: 16-byte units (octet of dims, key);  V: units (16 keys u, lane half, dim) of eight keys in the order of the
//   score registers: keys 16 u + 4 half + 0..3, then 16 u + 8 + 4 half + 0..3
template <int kDim>
struct HalvedTile {
    static constexpr int kKeys = 32;
    static constexpr float kKeyFactor = 128.f;  // of every key value (gqa_f32_halved.h)
    static constexpr int kPlane = kKeys * kDim * 2;
    static constexpr int kKeyBytes = 2 * kPlane, kValueBytes = 3 * kPlane, kBytes = kKeyBytes + kValueBytes;

    // Where the unit of `dim` lies among those of its keys: lanes that write units four dims apart,
    // and lanes that read neighbouring ones, meet every bank once.
    __device__ static __forceinline__ int value_unit(int dim) { return dim ^ ((dim >> 4) & 3); }
};

// Splits the rows of one tile of one kv head: a workgroup of four waves, eight rows of K and eight of V each.
// Bound by memory: 14.6 MB of rows in and 18.4 out in 9.5 us, 1777 tokens of 8 kv heads of 128.
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

    static __device__ __forceinline__ void halves(float x, float factor, _Float16 &hi, _Float16 &lo)
    {
        hi = (_Float16)(x * factor);
        lo = (_Float16)fmaf(x, factor, -(float)hi);
    }

    // A value as the sum of three bf16 values, each the nearest of what is left: all 24 bits, and F32's range of
    // exponents.  The last bits of a value below 2^-102 would lie below bf16's normal numbers: it is a NaN
    // here, and so is every row that meets it.  Two values at a time.
    static __device__ __forceinline__ void thirds(float a, float b, uint32_t (&part)[3])
    {
        float left[2] = {a, b};
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (left[i] != 0.f && fabsf(left[i]) < 0x1p-102f) left[i] = __builtin_nanf("");
#pragma unroll
        for (int n = 0; n < 3; ++n) {
            part[n] = pack_bf16x2(left[0], left[1]);
            left[0] -= __builtin_bit_cast(float, part[n] << 16);
            left[1] -= __builtin_bit_cast(float, part[n] & 0xffff0000u);
        }
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
                unsigned char *unit = lds + Tile::kKeyBytes + at * 16 + (quarter & 1) * 8 + ((from + j0) & 3) * 2;
#pragma unroll
                for (int j = 0; j < kRun; j += 2) {
                    uint32_t part[3];
                    thirds(v[j0 + j][i], v[j0 + j + 1][i], part);
#pragma unroll
                    for (int n = 0; n < 3; ++n)
                        *reinterpret_cast<uint32_t *>(unit + 2 * j + n * Tile::kPlane) = part[n];
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
