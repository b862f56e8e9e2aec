// Block-wide copies of dimension tables from memory into LDS, and how a probe's
// blocks share its vectors.  Internal to libfls.so.
//
// Every block of a star probe copies 80-110 KB before its first row, so the
// copy's latency is the kernel's: a loop of one word (or byte) per work-item
// waits for a round trip per 4 KB (or 1 KB), while four 16-byte loads in
// flight per work-item take two round trips in all.  At 1M rows, where little
// else is left: Q3.1 24.2 -> 17.0 us, Q4.1 23.4 -> 20.3, Q2.1 17.3 -> 16.0 (a
// zeroing launch less among them in the first two).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fls_columns.hpp"

namespace fls {

typedef uint32_t u32x4_w __attribute__((ext_vector_type(4), aligned(4)));  // needs a word's alignment only

// put(i, w): word i of n, every work-item of the block together.
template <typename Put>
__device__ __forceinline__ void stage_each_word(const uint32_t* __restrict src, uint32_t n, Put put) {
    constexpr uint32_t kAhead = 4;
    const uint32_t n4 = n / 4u, t = threadIdx.x, step = blockDim.x;
    for (uint32_t i0 = t; i0 < n4; i0 += kAhead * step) {
        u32x4_w v[kAhead];
#pragma unroll
        for (uint32_t k = 0; k < kAhead; ++k)
            v[k] = *(const __attribute__((address_space(1))) u32x4_w*)(src + 4u * min(i0 + k * step, n4 - 1u));
#pragma unroll
        for (uint32_t k = 0; k < kAhead; ++k) {
            const uint32_t i = i0 + k * step;
            if (i < n4) {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) put(4u * i + j, v[k][j]);
            }
        }
    }
    if (4u * n4 + t < n) put(4u * n4 + t, src[4u * n4 + t]);
}

// n words to LDS.
__device__ __forceinline__ void stage_words(uint32_t* __restrict dst, const uint32_t* __restrict src, uint32_t n) {
    stage_each_word(src, n, [dst](uint32_t i, uint32_t w) { dst[i] = w; });
}

// n bytes to LDS, add to each (mod 256); src on a word boundary.
__device__ __forceinline__ void stage_bytes(uint8_t* __restrict dst, const uint8_t* __restrict src, uint32_t n,
                                            uint32_t add = 0) {
    if ((reinterpret_cast<uintptr_t>(src) & 3u) == 0) {
        const uint32_t a = add * 0x01010101u;
        stage_each_word(reinterpret_cast<const uint32_t*>(src), n / 4u, [dst, a](uint32_t i, uint32_t w) {
            w = ((w & 0x7f7f7f7fu) + (a & 0x7f7f7f7fu)) ^ ((w ^ a) & 0x80808080u);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) dst[4u * i + j] = (uint8_t)(w >> (8u * j));
        });
        const uint32_t i = (n & ~3u) + threadIdx.x;
        if (i < n) dst[i] = (uint8_t)(src[i] + add);
    } else {
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) dst[i] = (uint8_t)(src[i] + add);
    }
}

// A persistent probe's work is vector pairs (a half-wave each), shared out by
// the wave: with a whole block's 32 vectors as the step, 59,986,214 rows are
// 7.15 steps of 256 blocks, and the last one kept few of them busy while the
// rest waited.  Shared by the wave that step is the first two or three waves of
// every block: 60M rows Q3.1 105.5 -> 99.5 us, Q4.1 149.7 -> 141, Q2.1 82 ->
// 80.5; 120M 191.4 -> 184, 278 -> 269, 145.7 -> 142.

// Fixed widths: wave w of block b takes pairs w * blocks + b and every
// (waves x blocks)th after it, so the blocks read one region at a time.
__device__ __forceinline__ uint64_t first_pair() {
    return (uint64_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * gridDim.x + blockIdx.x;
}
__device__ __forceinline__ uint64_t pair_step() { return (uint64_t)gridDim.x * (blockDim.x >> 6); }

// Any encoding: block b has a contiguous share of the n pairs, wave w the w-th
// of it and every (waves)th after, so a block's metadata words share lines
// (taken as above they do not: 10M mixed rows Q4.1 78 -> 86 us, this way 62; 60M
// 263 -> 263 and 233; Q3.1 176 -> 166 and 162).
struct PairRange {
    uint64_t first, end, step;
};
__device__ __forceinline__ PairRange block_pairs(uint64_t n) {
    const uint64_t share = (n + gridDim.x - 1u) / gridDim.x, at = share * blockIdx.x;
    return PairRange{at + (uint64_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)),
                     at + share < n ? at + share : n, blockDim.x >> 6};
}

// Pairs a block should have before another one is launched.  Fewer than its
// waves, because a small table otherwise leaves most CUs idle.  Fixed widths,
// blocks of 16, 8 and 4 pairs: 1M rows Q4.1 19.3, 15.2 and 15.1 us, Q3.1 17.2,
// 15.2 and 15.3; 3M rows Q4.1 21.8, 19.1 and 21.0 (each block stages its
// tables).  Any encoding, where a vector takes longer: 1M rows Q4.1 54.7, 45.3
// and 44.5, 100,003 rows (a slow RLE vector among them) 57.3, 52.9 and 49.8.
constexpr uint64_t kFixedPairs = 8;
constexpr uint64_t kAnyPairs = 4;

// Blocks of such a probe: n_pairs in blocks of per_block, at most the resident ones.
inline int pair_grid(const void* kernel, int block, size_t lds, uint64_t n_pairs, uint64_t per_block, uint32_t* grid) {
    uint64_t most = 0;
    if (const int st = resident_blocks(kernel, block, lds, &most)) return st;
    const uint64_t want = n_pairs / per_block + (n_pairs % per_block != 0);
    *grid = (uint32_t)(want < 1 ? 1 : want < most ? want : most);
    return FLS_OK;
}

}  // namespace fls
