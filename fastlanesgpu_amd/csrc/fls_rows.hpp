// Row-order (coalesced) view of a 1024-value vector, shared by the GPU
// encoders.  Internal to libfls.so.
//
// A half-wave holds a vector with lane l reading rows 32j + l (j = 0..31),
// i.e. element l of every 32-row chain j: each load instruction reads two
// whole 128-byte lines.  FastLanes delta's chains are 32 consecutive rows,
// chain c owned in the packed format by the lane l with chain_slot(l) = c, its
// element j in register row rsum_row(j) (rsum.cuh:8-106).  Chain deltas and
// run starts are therefore neighbour-lane comparisons, and only the payload
// itself has to move to its owning lane, through a padded LDS tile.  (A lane
// reading its own chain straight from memory touches 64 lines per
// instruction.  Over 59,986,214 values, that way and this way: delta plan 104
// and 39 us, delta pack 105 and 39, RLE plan 121 and 35, RLE pack 128 and 52,
// transposed bit-pack at 24 bits 1,137 and 62, at 6 bits 1,013 and 47; a copy
// of the same bytes takes 36 to 64.)
#pragma once

#include "fls/device/unpack.hpp"
#include "fls_runtime.hpp"

namespace fls {

__device__ __forceinline__ uint32_t wid(uint32_t x) { return x ? 32u - __clz(x) : 0u; }

// Half-wave (32-lane) reductions.  Within a 16-lane row DPP moves data at
// VALU speed (quad_perm swaps at distance 1 and 2, then row_ror:4 and
// row_ror:8 -- after the quad steps each lane holds its quad, and each
// rotation doubles the span, so every row lane ends with the row total, for
// sums too); one lane exchange then joins the two rows of the half-wave.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kRowRor4 = 0x124, kRowRor8 = 0x128;
constexpr int kWaveShr1 = 0x138;  // lane i <- lane i-1

template <typename Op>
__device__ __forceinline__ uint32_t half_reduce(uint32_t x, Op op) {
    x = op(x, dpp<kQuadXor1>(x));
    x = op(x, dpp<kQuadXor2>(x));
    x = op(x, dpp<kRowRor4>(x));
    x = op(x, dpp<kRowRor8>(x));
    return op(x, (uint32_t)__shfl_xor(x, 16, 64));
}
__device__ __forceinline__ uint32_t h_or(uint32_t x) {
    return half_reduce(x, [](uint32_t a, uint32_t b) { return a | b; });
}
__device__ __forceinline__ uint32_t h_min(uint32_t x) {
    return half_reduce(x, [](uint32_t a, uint32_t b) { return min(a, b); });
}
__device__ __forceinline__ uint32_t h_max(uint32_t x) {
    return half_reduce(x, [](uint32_t a, uint32_t b) { return max(a, b); });
}
__device__ __forceinline__ uint32_t h_sum(uint32_t x) {
    return half_reduce(x, [](uint32_t a, uint32_t b) { return a + b; });
}

// The chain that lane l packs.
__device__ __forceinline__ uint32_t chain_slot(uint32_t l) { return 2u * (l & 15u) + (l >> 4); }

// Value of original row k of the column, padding past n with the last value.
__device__ __forceinline__ uint32_t padded(const uint32_t* __restrict in, uint64_t n, uint64_t k) {
    return in[k < n ? k : n - 1];
}

// Coalesced load of vector v: x[j] = row 32j + l (rows past n repeat row n-1).
__device__ __forceinline__ void load_rows(const uint32_t* __restrict in, uint64_t n, uint64_t v, uint32_t (&x)[32]) {
    const uint64_t base = v * 1024u + dev::lane32();
    if (v * 1024u + 1024u <= n) {
#pragma unroll
        for (int j = 0; j < 32; ++j) x[j] = __builtin_nontemporal_load(in + base + 32u * j);
    } else {
#pragma unroll
        for (int j = 0; j < 32; ++j) x[j] = padded(in, n, base + 32u * j);
    }
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Transpose tile: row j of chain c at 33c + j, conflict-free both ways.
constexpr int kTile = 32 * 33;

// Rows in the coalesced layout into the tile (one half-wave; wave_sync before
// reading it back).
__device__ __forceinline__ void rows_to_tile(const uint32_t (&x)[32], uint32_t* __restrict tile) {
    const uint32_t l = dev::lane32();
#pragma unroll
    for (int j = 0; j < 32; ++j) tile[33 * j + l] = x[j];  // element l of chain j
}

}  // namespace fls
