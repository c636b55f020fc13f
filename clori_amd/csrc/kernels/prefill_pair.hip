// Grouped-query attention prefill at head dimension 256 for gfx950 (wave64): bf16 in and out,
// fp32 scores, online softmax and accumulation, the contract of prefill.hip.
//
// At 256 lanes a wave that holds 32 rows alone (128 accumulator, 64 query, 64 score registers)
// has its SIMD to itself, spills, and fetches one 1 KB operand from LDS per MFMA: four waves ask
// for 128 B/clk, all LDS has.  Here a workgroup of four waves owns 128 rows as two pairs; a pair
// shares 64 rows, and the two waves split the work of a 64-key step in both products:
//     S^T[key][row]: wave h computes keys 32h .. 32h+31 for all 64 rows  (16 k-steps x 2 row blocks)
//     O^T[dim][row]: wave h accumulates dims 128h .. 128h+127            (4 key slices x 4 x 2)
// Every operand fetched from LDS feeds two MFMAs (two blocks of 32 rows): 109 B/clk with the
// tile writes, the exchange of the probabilities (4 KB per wave and step) included.
//
// One step (64 MFMAs per wave) is two phases, and the softmax of a tile runs across the boundary:
//     S phase  S^T of tile t+1; behind its MFMAs the exponentials of tile t for the second row
//              block, then the tile's probabilities into the exchange area; the loads of V(t+1)
//     O phase  O^T update with tile t (own keys first, then the partner's); behind its MFMAs the
//              maximum of tile t+1 and the exponentials of its first row block; loads of K(t+3)
// Both barriers of a step sit a few MFMAs before the end of a phase, when every operand of the
// phase has been fetched, so that the first operands of the next phase are on their way under the
// last MFMAs.  "mid": the probabilities are exchanged, V(t) is in LDS, K(t+1) may be overwritten.
// "top": K(t+2) is in LDS, V(t) and the exchange area may be overwritten.  The loads of a tile have
// one and a half steps to arrive, at most two tiles are younger than the one waited for: vmcnt(16).
//
// The reference that the scores of a row are taken relative to is the row's maximum over the first
// tile of the walk, and it stays: fp32 sums and bf16 probabilities keep their relative precision
// whatever their magnitude, so nothing is lost as long as nothing overflows (a later score would
// have to be about 2^100 times the first tile's largest in weight).  The walk therefore carries no
// maximum, no decision and no rescaling.  Where a complete row sum or an accumulator is not finite in
// the end, the workgroup walks again with a loop that rescales in every tile (walk_rescaling); what is
// still not finite then is the inputs' fault.
//
// 2000 tokens of 24/4 heads behind 13333 (704 GFLOP): 873 us with one wave per 32 rows (a maximum, a
// decision and 33 spilled registers in every step), 634 us here.  The main loop holds no spilled
// register (256 + 256 registers: O^T and three quarters of the queries in accumulation registers) and
// meets no bank conflict; its MFMAs are busy 59 % of the waves' cycles, 46 % of the device's (256 units
// work on 496 workgroups), and the launch of 708 GFLOP with its masked keys takes 618 us: 1.15 PFLOP/s,
// where a large library GEMM reaches 1.28.
//
// A workgroup spends some 20000 cycles before its first and after its last step, most of them on
// instructions that it meets once (47 KB of code): whole walks of a few steps keep the kernel of
// prefill.hip (the line and both sides are in host/rocm_prefill.c).
#include "mfma.h"
#include "prefill_rows.h"

#include "../kernel_params.h"

namespace {

constexpr int kDim = 256;
constexpr int kKeyTile = 64;
constexpr int kRowBytes = kDim * 2;
constexpr int kTileBytes = kKeyTile * kRowBytes;   // 32 KB per K or V tile
constexpr int kRowsPerBlock = YVEX_ROCM_PREFILL_ROWS;
constexpr int kSteps = kDim / 16;                  // k-steps of S^T
constexpr int kDimBlocks = 4;                      // 32-dim blocks of the wave's half of O^T
constexpr int kLoads = 8;                          // 1 KB loads per wave and tile
constexpr int kDepth = 4;                          // operand fetches ahead of their MFMAs
constexpr int kVectorQueries = 4;                  // k-steps whose queries sit in vector registers
constexpr int kVArea = 2 * kTileBytes, kPArea = 4 * kTileBytes, kStatArea = kPArea + 4 * 4096;
constexpr int kLdsBytes = kStatArea + 4 * 64 * 4;
constexpr int kWaitTwoTiles = 0x0f70 | (1 << 14);  // vmcnt(16), lgkmcnt and expcnt untouched
constexpr int kWaitTwoTilesAndLds = 0x0070 | (1 << 14);  // vmcnt(16) and lgkmcnt(0)

typedef __attribute__((address_space(3))) short4v lds_short4;

__device__ inline void flag(int32_t *status, int code) { atomicCAS(status, 0, code); }

// chunk c of row r sits at chunk position c ^ swizzle(r) (prefill.hip: rows of 512 bytes)
__device__ constexpr int swizzle(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

struct PrefillPair {
    const yvex_rocm_prefill_params &p;
    unsigned char *const lds;
    const int lane, wave, n, g, half, pair;
    uint32_t row_head, kv_head, row0;  // row0: first packed row of the pair
    int32_t first_key, key_count;      // keys are numbered from the first one of this workgroup's run
    int32_t visible[2];                // last key the lane's row of either block sees
    i32x4 k_rsrc, v_rsrc;
    uint32_t k_row_bytes, v_row_bytes, lds_base, k_lane, v_lane, chunk_lane;
    uint32_t k_addr[8], v_addr[2][kDimBlocks][2];  // v_addr[0]: own keys, [1]: the partner's
    uint32_t p_own, p_other, stat_own, stat_other;
    bf16x8 q[2][kSteps];
    floatx16 o[2][kDimBlocks];
    // of the lane's row of either block: the reference (log2 units), its negative, the row sum
    float ref[2], neg_ref[2], l_run[2];
    uint32_t pk[2][8], pk_first[8];  // bf16 pairs [row block][slice * 4 + pair]; first block of the next tile
    u32x4 frag[kDepth];

    __device__ PrefillPair(const yvex_rocm_prefill_params &params, unsigned char *shared)
        : p(params), lds(shared), lane(threadIdx.x & 63),
          wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), n(threadIdx.x & 31),
          g((threadIdx.x & 63) >> 5), half(wave & 1), pair(wave >> 1)
    {
    }

    // 1 KB load j of this wave (rows 16 * wave + 2j and the next one) of a K or V tile.  A tile that
    // is not wanted is "loaded" from past the descriptor's range, so that the number of loads in
    // flight does not depend on the step.
    __device__ inline void stage(i32x4 rsrc, uint32_t lane_row, uint32_t row_bytes, uint32_t area, uint32_t tile,
                                 bool wanted, int j) const
    {
        lds_dma_b128(lds_base + area + wave * (16 * kRowBytes) + j * 1024, rsrc,
                     lane_row + (chunk_lane ^ (uint32_t)(swizzle(2 * j) << 4)),
                     (uint32_t)__builtin_amdgcn_readfirstlane(
                         (int)(wanted ? (tile * kKeyTile + 2 * j) * row_bytes : 0xfffffff0u)));
    }
    __device__ inline void stage_k(uint32_t tile, bool wanted, int buf, int j) const
    {
        stage(k_rsrc, k_lane, k_row_bytes, buf * kTileBytes, tile, wanted, j);
    }
    __device__ inline void stage_v(uint32_t tile, bool wanted, int buf, int j) const
    {
        stage(v_rsrc, v_lane, v_row_bytes, kVArea + buf * kTileBytes, tile, wanted, j);
    }

    // K operand of k-step kk: row 32 * half + n, dims 16kk + 8g .. +7
    __device__ inline u32x4 fetch_k(int buf, int kk) const
    {
        return *reinterpret_cast<const u32x4 *>(lds + k_addr[kk & 7] + (buf * kTileBytes + (kk >> 3) * 256));
    }
    // V^T operand `index` of the O phase (slice index / 4: two of the wave's own keys, then two of
    // the partner's; dim block index % 4)
    __device__ inline u32x4 fetch_v(int buf, int index) const
    {
        const int slice = index >> 2, db = index & 3;
        const int base = kVArea + buf * kTileBytes + (slice & 1) * 16 * kRowBytes;
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_short4 *)(lds + v_addr[slice >> 1][db][0] + base));
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_short4 *)(lds + v_addr[slice >> 1][db][1] + base));
        return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }

    // The two MFMAs of k-step kk.  The scores live in vector registers (the accumulation registers
    // hold O^T and most of the queries), so these are written as assembly; what reads them waits
    // for them by hand.
    __device__ inline void score(floatx16 (&s)[2], u32x4 k, int kk) const
    {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            if (kk == 0)
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[rb]) : "v"(k), "v"(q[rb][kk]));
            else if (kk < kVectorQueries)
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[rb]) : "v"(k), "v"(q[rb][kk]));
            else
                asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[rb]) : "v"(k), "a"(q[rb][kk]));
        }
    }

    // The two MFMAs of V^T operand j.
    __device__ inline void update(u32x4 v, const u32x4 (&theirs)[2][2], int j)
    {
        const int slice = j >> 2, u = slice & 1;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const u32x4 own = {pk[rb][u * 4], pk[rb][u * 4 + 1], pk[rb][u * 4 + 2], pk[rb][u * 4 + 3]};
            o[rb][j & 3] = mfma_32x32x16(as_bf16x8(v), as_bf16x8(slice < 2 ? own : theirs[rb][u]), o[rb][j & 3]);
        }
    }

    // element e of row block rb of the tile in hand: probability, row sum, packed pair
    __device__ inline void probability(floatx16 (&s)[2], uint32_t *pairs, int rb, int e)
    {
        const float pe = fast_exp2(__builtin_fmaf(s[rb][e], p.scale_log2, neg_ref[rb]));
        s[rb][e] = pe;
        l_run[rb] += pe;
        if (e & 1) pairs[e >> 1] = pack_bf16x2(s[rb][e - 1], pe);
    }

    // Masks the keys of tile `tile` (the wave's half of it) that a row does not see.
    __device__ inline void mask_tile(floatx16 (&s)[2], uint32_t tile) const
    {
        const int32_t key0 = (int32_t)(tile * kKeyTile) + half * 32 + g * 4;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (key0 + (i >> 2) * 8 + (i & 3) > visible[rb]) s[rb][i] = -INFINITY;
    }

    __device__ static inline float peak_of(const floatx16 &s)
    {
        float m = fmaxf(s[0], s[1]);
#pragma unroll
        for (int i = 2; i < 16; i += 2) m = fmaxf(m, fmaxf(s[i], s[i + 1]));
        return m;
    }

    // The rows' maxima over both waves' keys of a tile, in log2 units.
    __device__ inline void pair_peak(const floatx16 (&s)[2], float (&top)[2]) const
    {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            top[rb] = max_xor32(peak_of(s[rb])) * p.scale_log2;
            *reinterpret_cast<float *>(lds + stat_own + rb * 128) = top[rb];
        }
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
            top[rb] = fmaxf(top[rb], *reinterpret_cast<const float *>(lds + stat_other + rb * 128));
    }

    // Reads the partner's probabilities of the tile in hand.
    __device__ inline void take_partner(u32x4 (&theirs)[2][2]) const
    {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                theirs[rb][u] = *reinterpret_cast<const u32x4 *>(lds + p_other + (rb * 2 + u) * 1024);
    }
    __device__ inline void leave_pairs(int rb, int u) const
    {
        const u32x4 w = {pk[rb][u * 4], pk[rb][u * 4 + 1], pk[rb][u * 4 + 2], pk[rb][u * 4 + 3]};
        *reinterpret_cast<u32x4 *>(lds + p_own + (rb * 2 + u) * 1024) = w;
    }

    __device__ inline void open()
    {
        k_row_bytes = (uint32_t)p.k_stride * 2u;
        v_row_bytes = (uint32_t)p.v_stride * 2u;
        k_rsrc = raw_buffer(p.k + (uint64_t)(uint32_t)first_key * p.k_stride + (uint64_t)kv_head * kDim,
                            (uint32_t)key_count * k_row_bytes - kv_head * kRowBytes);
        v_rsrc = raw_buffer(p.v + (uint64_t)(uint32_t)first_key * p.v_stride + (uint64_t)kv_head * kDim,
                            (uint32_t)key_count * v_row_bytes - kv_head * kRowBytes);
        lds_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_address_of(lds));
        // lane L of load j fills chunk position L % 32 of row 16 * wave + 2j + L / 32; the swizzle of
        // that row is the one of L / 32 with the one of 2j exchanged in (swizzle permutes bits)
        const uint32_t lane_row = 16u * (uint32_t)wave + ((uint32_t)lane >> 5);
        k_lane = lane_row * k_row_bytes;
        v_lane = lane_row * v_row_bytes;
        chunk_lane = (((uint32_t)lane & 31u) ^ (uint32_t)swizzle(lane >> 5)) << 4;
#pragma unroll
        for (int k8 = 0; k8 < 8; ++k8)
            k_addr[k8] = (uint32_t)((half * 32 + n) * kRowBytes + (((2 * k8 + g) ^ swizzle(n)) << 4));
        // as in prefill.hip: 16-lane group b = lane / 16 covers dims 16 * (b & 1) and key half g, lane
        // a = lane % 16 addresses key row 8h + 4g + a / 4 and dims 4 * (a % 4)
        const int a = lane & 15, b1 = (lane >> 4) & 1;
#pragma unroll
        for (int whose = 0; whose < 2; ++whose)
#pragma unroll
            for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = 8 * h + 4 * g + (a >> 2);
                    const int chunk = (db * 4 + 2 * b1 + ((a >> 1) & 1)) ^ swizzle(r);
                    v_addr[whose][db][h] = (uint32_t)(((half ^ whose) * 32 + r) * kRowBytes + half * 256 +
                                                      (chunk << 4) + 8 * (a & 1));
                }
        p_own = (uint32_t)(kPArea + wave * 4096 + lane * 16);
        p_other = (uint32_t)(kPArea + (wave ^ 1) * 4096 + lane * 16);
        stat_own = (uint32_t)(kStatArea + wave * 256 + n * 4);
        stat_other = (uint32_t)(kStatArea + (wave ^ 1) * 256 + n * 4);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const uint32_t row = min(row0 + rb * 32 + n, p.rows - 1u), token = token_of(p, row);
            const uint32_t head = row_head * p.pack + (row - token * p.pack);
            const uint16_t *src = p.q + (uint64_t)token * p.q_stride + (uint64_t)head * kDim + g * 8;
#pragma unroll
            for (int kk = 0; kk < kSteps; ++kk) q[rb][kk] = as_bf16x8(load_b128(src + kk * 16));
            visible[rb] = (p.causal ? min((int32_t)(p.query_start + token), (int32_t)p.kv_tokens - 1)
                                    : (int32_t)p.kv_tokens - 1) - first_key;
        }
        clear();
    }
    __device__ inline void clear()
    {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            l_run[rb] = 0.f;
#pragma unroll
            for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[rb][db][i] = 0.f;
        }
    }

    // One step; kOdd: the step's number is odd (which buffers), kLast: no further tile.
    template <bool kOdd, bool kLast>
    __device__ __forceinline__ void step(uint32_t t, uint32_t tiles, floatx16 (&s)[2], floatx16 (&s_next)[2],
                                         int32_t first_visible)
    {
        constexpr int here = kOdd ? 1 : 0, next = here ^ 1;
        const bool want_v = t + 1u < tiles, want_k = t + 3u < tiles;
        u32x4 theirs[2][2];
        // ---- S phase: S^T of tile t+1, the exponentials of tile t for the second row block ----
#pragma unroll
        for (int j = 0; j < 8; ++j) pk[0][j] = pk_first[j];
#pragma unroll
        for (int kk = 0; kk < kSteps; ++kk) {
            if (!kLast) score(s_next, frag[kk % kDepth], kk);
            if (kk == 12) {
                // mid: every operand of this phase has been fetched, the probabilities are in LDS
                __builtin_amdgcn_s_waitcnt(kLast ? 0x0070 : kWaitTwoTilesAndLds);
                __syncthreads();
            }
            if (kk + kDepth >= kSteps) frag[kk % kDepth] = fetch_v(here, kk + kDepth - kSteps);
            else if (!kLast) frag[kk % kDepth] = fetch_k(next, kk + kDepth);
            if (kk == 12) take_partner(theirs);
            if (!kLast && kk < kLoads) stage_v(t + 1u, want_v, next, kk);
            if (kk < 2) leave_pairs(0, kk);
#pragma unroll
            for (int e = (kk * 8 + 4) / 5; e < (kk * 8 + 12) / 5 && e < 16; ++e) probability(s, pk[1], 1, e);
            if (kk == 5) leave_pairs(1, 0);
            if (kk == 10) leave_pairs(1, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- O phase: O^T update with tile t, the exponentials of tile t+1 for the first row block ----
#pragma unroll
        for (int j = 0; j < 4 * kDimBlocks; ++j) {
            update(frag[j % kDepth], theirs, j);
            if (!kLast && j == 12) {
                // top: every operand of this phase has been fetched
                __builtin_amdgcn_s_waitcnt(kWaitTwoTilesAndLds);
                __syncthreads();
            }
            if (j + kDepth < 4 * kDimBlocks) frag[j % kDepth] = fetch_v(here, j + kDepth);
            else if (!kLast) frag[j % kDepth] = fetch_k(here, j + kDepth - 4 * kDimBlocks);
            if (!kLast) {
                if (j < kLoads / 2) {
                    stage_k(t + 3u, want_k, next, 2 * j);
                    stage_k(t + 3u, want_k, next, 2 * j + 1);
                }
                // four MFMAs are behind the last one that wrote the scores: they can be read
                if (j == 1) {
                    asm volatile("" : "+v"(s_next[0]), "+v"(s_next[1]));
                    if ((int32_t)((t + 1u) * kKeyTile + kKeyTile - 1u) > first_visible ||
                        (int32_t)((t + 2u) * kKeyTile) > key_count)
                        mask_tile(s_next, t + 1u);
                }
#pragma unroll
                for (int e = ((j - 2) * 4 + 2) / 3; j >= 2 && e < ((j - 1) * 4 + 2) / 3 && e < 16; ++e)
                    probability(s_next, pk_first, 0, e);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    __device__ inline void run()
    {
        uint32_t item = blockIdx.x, split = 0u;
        const bool partial = item >= p.whole_items;
        if (partial) {
            split = (item - p.whole_items) / p.tail_items;
            item = p.whole_items + (item - p.whole_items) % p.tail_items;
        }
        const uint32_t level = item / p.row_heads, q_tile = p.query_tiles - 1u - level;
        row_head = item - level * p.row_heads;
        kv_head = kv_head_of(p, row_head);
        row0 = q_tile * kRowsPerBlock + pair * 64u;
        // keys visible to the last row of the workgroup bound the walk
        const uint32_t last_row = min(p.rows, (q_tile + 1u) * kRowsPerBlock) - 1u;
        const uint32_t kv_end = p.causal ? min(p.kv_tokens, p.query_start + token_of(p, last_row) + 1u) : p.kv_tokens;
        uint32_t tiles = (kv_end + kKeyTile - 1) / kKeyTile;
        const uint32_t slot = (item - p.whole_items) * p.splits + split;
        first_key = 0;
        if (partial) {
            const uint32_t per_split = (tiles + p.splits - 1u) / p.splits;
            const uint32_t begin = min(tiles, split * per_split);
            tiles = min(per_split, tiles - begin);
            first_key = tiles != 0u ? (int32_t)(begin * kKeyTile) : 0;
        }
        key_count = (int32_t)p.kv_tokens - first_key;
        if (tiles == 0u) {  // a run without steps (the whole workgroup alike)
            if (half == 0 && g == 0)
                for (int rb = 0; rb < 2; ++rb)
                    if (row0 + rb * 32 + n < p.rows) leave_statistics(slot, rb, 0.f, -INFINITY);
            return;
        }
        // last key the first row of the workgroup sees: tiles up to it need no mask
        const int32_t first_visible =
            p.causal ? (int32_t)(p.query_start + token_of(p, min(q_tile * kRowsPerBlock, p.rows - 1u))) - first_key
                     : key_count - 1;
        open();

        // ---- prologue: K(0), K(1), V(0) and K(2) on their way, S^T of tile 0 ----
#pragma unroll
        for (int j = 0; j < kLoads; ++j) stage_k(0u, true, 0, j);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) stage_k(1u, tiles > 1u, 1, j);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) stage_v(0u, true, 0, j);
        __builtin_amdgcn_s_waitcnt(kWaitTwoTiles);
        __syncthreads();
        floatx16 s_even[2], s_odd[2];
#pragma unroll
        for (int i = 0; i < kDepth; ++i) frag[i] = fetch_k(0, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < kSteps; ++kk) {
            score(s_even, frag[kk % kDepth], kk);
            if (kk + kDepth < kSteps) frag[kk % kDepth] = fetch_k(0, kk + kDepth);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();  // every wave is done with K(0)
#pragma unroll
        for (int j = 0; j < kLoads; ++j) stage_k(2u, tiles > 2u, 0, j);
        // wait states between an 8-pass MFMA and the first vector read of its result
        asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(s_even[0]), "+v"(s_even[1]));
        if ((int32_t)(kKeyTile - 1) > first_visible || (int32_t)kKeyTile > key_count) mask_tile(s_even, 0u);
        pair_peak(s_even, ref);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) neg_ref[rb] = ref[rb] == -INFINITY ? 0.f : -ref[rb];
#pragma unroll
        for (int e = 0; e < 16; ++e) probability(s_even, pk_first, 0, e);
        __builtin_amdgcn_s_waitcnt(kWaitTwoTilesAndLds);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kDepth; ++i) frag[i] = fetch_k(1, i);

        // ---- main loop: two steps per turn, the score registers change roles ----
        uint32_t t = 0u;
        for (; t + 2u < tiles; t += 2u) {
            step<false, false>(t, tiles, s_even, s_odd, first_visible);
            step<true, false>(t + 1u, tiles, s_odd, s_even, first_visible);
        }
        if (t + 1u < tiles) {
            step<false, false>(t, tiles, s_even, s_odd, first_visible);
            step<true, true>(t + 1u, tiles, s_odd, s_even, first_visible);
        } else {
            step<false, true>(t, tiles, s_even, s_odd, first_visible);
        }

        // ---- the pair's row sums, then partials or rows ----
        float l[2];
        pair_sum(l);
        if (any_row_overflowed(l)) {
            walk_rescaling(tiles);
            pair_sum(l);
        }
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            if (row0 + rb * 32 + n >= p.rows) continue;
            if (partial) leave_partial(slot, rb, l[rb]);
            else publish(rb, l[rb]);
        }
    }

    // The row sums of the pair, keys 0 .. 31 of the tiles first in both waves.
    __device__ inline void pair_sum(float (&l)[2]) const
    {
        float mine[2];
        __syncthreads();  // the area has been read
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            mine[rb] = sum_xor32(l_run[rb]);
            *reinterpret_cast<float *>(lds + stat_own + rb * 128) = mine[rb];
        }
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const float theirs = *reinterpret_cast<const float *>(lds + stat_other + rb * 128);
            l[rb] = half == 0 ? mine[rb] + theirs : theirs + mine[rb];
        }
    }

    // Whether a row of the workgroup is not finite (the same answer in every wave).  `l`: the complete
    // row sums; each is the sum of four parts (two lane halves, two waves) that may be finite when it is not.
    __device__ inline bool any_row_overflowed(const float (&l)[2]) const
    {
        bool bad = !(isfinite(l[0]) && isfinite(l[1]));
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) bad |= !isfinite(o[rb][db][i]);
        const bool wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0ull;
        __syncthreads();  // the area has been read
        if (lane == 0) *reinterpret_cast<uint32_t *>(lds + kStatArea + wave * 4) = wave_bad ? 1u : 0u;
        __syncthreads();
        const u32x4 w = *reinterpret_cast<const u32x4 *>(lds + kStatArea);
        return __builtin_amdgcn_readfirstlane((int)(w.x | w.y | w.z | w.w)) != 0;
    }

    // The same walk tile by tile, everything in its place: references raised and the accumulators
    // rescaled in every tile.  Only for rows the main loop has overflowed on.
    __device__ __forceinline__ void walk_rescaling(uint32_t tiles)
    {
        clear();
        ref[0] = ref[1] = -INFINITY;
        for (uint32_t t = 0u; t < tiles; ++t) {
            __syncthreads();  // every wave is done with the tiles and the areas
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                stage_k(t, true, 0, j);
                stage_v(t, true, 0, j);
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);
            __syncthreads();
            floatx16 s[2];
#pragma unroll
            for (int kk = 0; kk < kSteps; ++kk) score(s, fetch_k(0, kk), kk);
            asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(s[0]), "+v"(s[1]));
            mask_tile(s, t);
            float top[2];
            pair_peak(s, top);
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
                const float m_new = fmaxf(ref[rb], top[rb]);
                const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(ref[rb] - m_new);
                l_run[rb] *= alpha;
#pragma unroll
                for (int db = 0; db < kDimBlocks; ++db) o[rb][db] *= alpha;
                ref[rb] = m_new;
                neg_ref[rb] = m_new == -INFINITY ? 0.f : -m_new;
#pragma unroll
                for (int e = 0; e < 16; ++e) probability(s, pk[rb], rb, e);
                leave_pairs(rb, 0);
                leave_pairs(rb, 1);
            }
            __syncthreads();
            u32x4 theirs[2][2];
            take_partner(theirs);
#pragma unroll
            for (int j = 0; j < 4 * kDimBlocks; ++j) {
                const u32x4 v = fetch_v(0, j);
                update(v, theirs, j);
            }
        }
    }

    // Normalises and publishes the wave's half of a row, and its LSE.
    __device__ inline void publish(int rb, float l) const
    {
        const uint32_t row = row0 + rb * 32 + n, token = token_of(p, row);
        const uint32_t head = row_head * p.pack + (row - token * p.pack);
        const float inv = 1.0f / l;
        const uint64_t at = ((uint64_t)token * p.query_heads + head) * kDim + half * 128 + g * 4;
        bool bad = !isfinite(l);  // (an infinite sum would publish zeros)
#pragma unroll
        for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp) {
                const float a0 = o[rb][db][grp * 4 + 0] * inv, a1 = o[rb][db][grp * 4 + 1] * inv;
                const float a2 = o[rb][db][grp * 4 + 2] * inv, a3 = o[rb][db][grp * 4 + 3] * inv;
                bad |= !(isfinite(a0) && isfinite(a1) && isfinite(a2) && isfinite(a3));
                u32x2 w;
                w.x = pack_bf16x2(a0, a1);
                w.y = pack_bf16x2(a2, a3);
                if (p.gate) {
                    w = gate_four(w, p.gate + at + db * 32 + grp * 8);
                    bad |= pair_not_finite(w.x) || pair_not_finite(w.y);
                }
                *reinterpret_cast<u32x2 *>(p.out + at + db * 32 + grp * 8) = w;
            }
        if (bad) flag(p.status, YVEX_ROCM_DEVICE_NUMERIC);
        if (p.lse && g == 0 && half == 0)
            p.lse[(uint64_t)token * p.query_heads + head] = (ref[rb] + fast_log2(l)) * YVEX_LN2;
    }

    // What this run of keys contributes to a row.
    __device__ inline void leave_statistics(uint32_t slot, int rb, float l, float m) const
    {
        float *ml = p.part_ml + ((uint64_t)slot * kRowsPerBlock + pair * 64 + rb * 32 + n) * 2u;
        ml[0] = m;
        ml[1] = l;
    }
    __device__ inline void leave_partial(uint32_t slot, int rb, float l) const
    {
        // the sum is brought into [1, 2) (the largest into [2, 4)) by a whole power of two, so that the
        // merge's weights are relative to the row's own magnitude; fast_exp2 has no subnormal results:
        // 2^-126 is the least factor
        const bool none = !(l > 0.f);
        const float shift = none || !isfinite(l) ? 0.f : fminf(__builtin_floorf(fast_log2(l)), 126.f);
        const float factor = fast_exp2(-shift);
        if (g == 0 && half == 0) leave_statistics(slot, rb, l * factor, none && l == 0.f ? -INFINITY : ref[rb] + shift);
        const uint64_t at = (uint64_t)slot * kRowsPerBlock + pair * 64 + rb * 32 + n;
        float *acc = p.part_acc + at * kDim + half * 128 + g * 4;
#pragma unroll
        for (int db = 0; db < kDimBlocks; ++db)
#pragma unroll
            for (int grp = 0; grp < 4; ++grp)
                *reinterpret_cast<floatx4 *>(acc + db * 32 + grp * 8) =
                    (floatx4){o[rb][db][grp * 4] * factor, o[rb][db][grp * 4 + 1] * factor,
                              o[rb][db][grp * 4 + 2] * factor, o[rb][db][grp * 4 + 3] * factor};
    }
};

}  // namespace

// grid = whole_items + tail_items * splits (as in prefill.hip), block 256; merged by
// yvex_rocm_prefill_merge_256.
extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
yvex_rocm_prefill_bf16_256(const yvex_rocm_prefill_params p)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLdsBytes];
    PrefillPair(p, lds).run();
}
