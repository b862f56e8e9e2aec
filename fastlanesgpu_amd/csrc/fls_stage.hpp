// Block-wide copies of dimension tables from memory into LDS.  Internal to
// libfls.so.
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

}  // namespace fls
