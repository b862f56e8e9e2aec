// FastLanes RLE decode of one vector straight to memory, in original row order
// or in stored (transposed) order.  Internal to libfls.so.
//
// The run index of a row is its chain's first index plus the run starts among
// the chain's elements up to the row: with a chain's 32 start bits in one word
// (bit rsum_row(e) = element e starts a run) that is one AND and one bit count
// with a mask, so every work-item computes the four consecutive outputs of its
// own 16-byte store and nothing has to be transposed through LDS.  Only the
// run values, the start words and the first indices are staged.
#pragma once

#include "fls_columns.hpp"

namespace fls {

// Runs staged at a time: 2,304 bytes of LDS per vector (with 1,024 runs, four
// blocks of 8 vectors per CU instead of eight).  A vector with more runs goes
// through the stage in two passes, each storing the outputs whose run it holds.
constexpr uint32_t kRunStage = 512;

struct alignas(16) RleLds {
    uint32_t starts[32];  // start word and first run index: by chain (row order)
    uint32_t first[32];   // or by lane (stored order)
    uint32_t runs[kRunStage];
};

// Rows of a chain's elements 0..e: element k sits in row
// rsum_row(k) = 4 (k % 8) + {0, 2, 1, 3}[k / 8].
__device__ __forceinline__ uint32_t chain_rows_upto(uint32_t e) {
    const uint32_t k = e >> 3, s = e & 7u;
    const uint32_t full = (k > 0 ? 0x11111111u : 0u) | (k > 1 ? 0x44444444u : 0u) | (k > 2 ? 0x22222222u : 0u);
    return full | ((0x11111111u & (0xffffffffu >> (28u - 4u * s))) << ((0x3120u >> (4u * k)) & 3u));
}

// Where a vector's RLE parts lie.
struct RleVector {
    uint32_t ibw;          // width of the index deltas
    uint32_t first;        // this lane's first run index
    const uint32_t* idx;   // index words
    const uint32_t* vals;  // run values, LSB-first at vbw bits
    uint32_t n_runs, vbw, vbase;
};

// Index deltas wider than a bit: no encoder here writes them, but the format
// takes them.  One lane walks its chain.
template <bool ROWS>
__device__ __forceinline__ void rle_emit_wide(const RleVector& r, uint32_t last, uint32_t rows,
                                              uint32_t* __restrict dst) {
    const uint32_t l = dev::lane32();
    const uint32_t mask = r.ibw >= 32u ? 0xffffffffu : ((1u << r.ibw) - 1u);
    uint32_t acc = r.first;
#pragma unroll 1
    for (uint32_t e = 0; e < 32u; ++e) {
        const uint32_t row = (uint32_t)dev::rsum_row((int)e), bit = row * r.ibw, k = bit >> 5, s = bit & 31u;
        const uint32_t lo = ldg(r.idx + 32u * k + l), hi = ldg(r.idx + 32u * (s + r.ibw > 32u ? k + 1u : k) + l);
        acc += __builtin_amdgcn_alignbit(hi, lo, s) & mask;
        const uint32_t x = r.vbase + linear_extract(r.vals, min(acc, last), r.vbw);
        const uint32_t at = ROWS ? 32u * (2u * (l & 15u) + (l >> 4)) + e : 32u * row + l;
        if (at < rows) dst[at] = x;
    }
}

// Decode the half-wave's vector to dst: rows 0..rows-1 in original order
// (ROWS), or all 1,024 stored positions (rows = 1024).  VEC: dst is 16-byte
// aligned; otherwise stores go through the caches, because they end in the middle
// of a line (120M rows of mean run 8: 199 us non-temporal, 144 this way).  LONG:
// the form for waves with a vector of more runs than the stage holds.  `lds` is
// this half-wave's; every exchange stays inside it.
template <bool ROWS, bool VEC, bool LONG = false>
__device__ __forceinline__ void rle_emit(const RleVector& r, RleLds& lds, uint32_t rows, uint32_t* __restrict dst) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t l = dev::lane32();
    const uint32_t nr = r.n_runs < 1024u ? r.n_runs : 1024u, last = nr ? nr - 1u : 0u;
    if (r.ibw > 1u) return rle_emit_wide<ROWS>(r, last, rows, dst);
    if constexpr (!LONG) {
        // Two passes over the stage store only what each holds, so a word per
        // work-item at consecutive places: the words of a 16-byte store taken
        // one at a time touched four lines each (60M rows of 1,024 runs a
        // vector: row order 134 us, stored order 202; this way 94 and 143).  The
        // wave's two vectors go the same way, or both ways' code runs in turn
        // (vectors of about 512 runs 69 and 72 us apart, 64 and 70 together).
        if (__any(last >= kRunStage)) return rle_emit<ROWS, false, true>(r, lds, rows, dst);
    }
    // through the cache: RLE vectors end anywhere in a line, which the next one
    // shares (with non-temporal loads here a line was read twice: 62.2 us
    // against 49.2 for 67M rows)
    const uint32_t starts = r.ibw ? ldg(r.idx + l) : 0u;
    const uint32_t vmask = r.vbw >= 32u ? 0xffffffffu : ((1u << r.vbw) - 1u);
    auto stage = [&](uint32_t from, uint32_t to) {  // runs [from, to) into the stage
        for (uint32_t k0 = from; k0 < to; k0 += 128u) {
            uint32_t lo[4] = {}, hi[4] = {}, sh[4] = {};
            if (r.vbw) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {  // four runs' words in flight
                    const uint32_t k = k0 + 32u * i + l, bit = (k < to ? k : from) * r.vbw, w = bit >> 5;
                    sh[i] = bit & 31u;
                    lo[i] = ldg(r.vals + w);
                    hi[i] = ldg(r.vals + (sh[i] + r.vbw > 32u ? w + 1u : w));
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t k = k0 + 32u * i + l;
                if (k < to) lds.runs[k - from] = r.vbase + (__builtin_amdgcn_alignbit(hi[i], lo[i], sh[i]) & vmask);
            }
        }
    };
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const uint32_t slot = ROWS ? 2u * (l & 15u) + (l >> 4) : l;
    stage(0u, min(last + 1u, kRunStage));
    lds.starts[slot] = starts;
    lds.first[slot] = r.first;
    fence();
    // run index of output t of this work-item.  VEC: t = 4j + i is place
    // 4l + 128j + i; else place 32t + l.
    uint32_t m[4], s4[4], f4[4];
    const uint32_t g = l >> 3, e0 = 4u * (l & 7u);
    if constexpr (ROWS && VEC) {  // place: chain g + 4j, element e0 + i
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] = chain_rows_upto(e0 + i);
    } else if constexpr (ROWS) {  // chain t, element l
        m[0] = chain_rows_upto(l);
    } else if constexpr (VEC) {  // lane e0 + i, row g + 4j: element j + 8 {0, 2, 1, 3}[g]
        m[0] = g == 0 ? 0u : g == 1 ? 0x55555555u : g == 2 ? 0x11111111u : 0x77777777u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s4[i] = lds.starts[e0 + i];
            f4[i] = lds.first[e0 + i];
        }
    }
    auto index = [&](int t) -> uint32_t {
        const int j = t >> 2, i = t & 3;
        uint32_t s, f, k;
        if constexpr (ROWS && VEC) {
            s = lds.starts[g + 4u * j];
            f = lds.first[g + 4u * j];
            k = m[i];
        } else if constexpr (ROWS) {
            s = lds.starts[t];
            f = lds.first[t];
            k = m[0];
        } else if constexpr (VEC) {
            s = s4[i];
            f = f4[i];
            k = m[0] | ((0x11111111u & (0xffffffffu >> (28 - 4 * j))) << g);
        } else {  // the lane's own row t: element t/4 + 8 {0, 2, 1, 3}[t % 4]
            s = starts;
            f = r.first;
            k = (i == 0 ? 0u : i == 1 ? 0x55555555u : i == 2 ? 0x11111111u : 0x77777777u) |
                ((0x11111111u & (0xffffffffu >> (28 - 4 * j))) << i);
        }
        return min(f + __builtin_popcount(s & k), last);
    };
    uint32_t from = 0;  // first run in the stage
    for (;;) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint32_t k[4], x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                k[i] = index(4 * j + i) - from;
                x[i] = lds.runs[min(k[i], kRunStage - 1u)];
            }
            const uint32_t p = VEC ? 4u * l + 128u * (uint32_t)j : 128u * (uint32_t)j + l;
            constexpr uint32_t step = VEC ? 1u : 32u;  // place of output 4j + i: p + step * i
            if ((!LONG || last < kRunStage) && p + 3u * step < rows) {
                if constexpr (VEC) {
                    __builtin_nontemporal_store(u32x4{x[0], x[1], x[2], x[3]}, reinterpret_cast<u32x4*>(dst + p));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if constexpr (LONG) __builtin_nontemporal_store(x[i], dst + p + step * i);
                        else dst[p + step * i] = x[i];
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (k[i] < kRunStage && p + step * i < rows) dst[p + step * i] = x[i];
            }
            __builtin_amdgcn_sched_barrier(0);  // few outputs in flight: their registers cost more waves than they hide
        }
        from += kRunStage;
        if (!LONG || from > last) break;
        fence();
        stage(from, min(last + 1u, from + kRunStage));
        fence();
    }
    fence();  // the stage may be written again
}

}  // namespace fls
