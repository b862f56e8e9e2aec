// One-launch scan of the encoders' per-vector word counts into offsets.
// Internal to libfls.so.
#pragma once

#include "fls/device/wave.hpp"
#include "fls_encode.hpp"

namespace fls {

// offsets[i] = sum_{k<i} words[i]; vmeta[i] = offsets[i] << 8 | bw[i];
// *total = sum of all, in one launch.  A block takes a ticket, scans its 1,024
// entries and publishes their sum, then adds up the sums of the blocks before
// it (a work-item per block, so one round trip up to 1,024 blocks).  A block
// waits only on blocks that drew their ticket before it, and every block
// publishes before it waits, so each wait ends.  The planner that fills words
// prepares the state (scan_clear); blocks that draw no valid ticket from it
// (scan_ticket) leave everything as it is.  Bound by those round trips: 6 us for 58,581
// vectors against 15 us (and two more launch gaps) as a reduction, a
// one-block scan of the sums and an apply pass.  (With 4,096 entries per block,
// too few to keep the loads moving, 7 us; mixed columns, which resolve their
// plan in it, 6.6 against 9.6 for 117,188 vectors.)
constexpr int kScanBlock = (int)kScanChunk;  // a work-item per entry
constexpr int kScanWaves = kScanBlock / 64;
constexpr unsigned long long kScanReady = 1ull << 63;  // a published sum

// Exclusive scan of one 32-bit value per work-item over the block: a DPP
// prefix sum per wave, then the 16 wave totals read by every work-item (a
// block's values here are vector word counts, at most 2^21 in total).
// sh: kScanWaves words of LDS.
__device__ __forceinline__ uint32_t block_exclusive_scan32(uint32_t x, uint32_t* sh, uint32_t& total) {
    const uint32_t incl = dev::wave_inclusive_sum(x);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 63u) sh[w] = incl;
    __syncthreads();
    uint32_t before = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kScanWaves; ++k) {
        const uint32_t t = sh[k];
        before += k < w ? t : 0u;
        tot += t;
    }
    total = tot;
    return before + incl - x;
}

// The widths' flag bits (kScanFlag) are counted here too, one atomic per
// block: an atomic on the counter per flagged vector costs 5.6 ns each, all on
// one address (117,188 of them: 655 us of a planning pass that takes 76).
// load(i, w, bw): vector i's word count and width word, read before vmeta[i] is
// written.
template <typename Load>
__device__ __forceinline__ void scan_vectors(Load load, uint64_t n, unsigned long long* __restrict state,
                                             fls_vmeta* vmeta, uint64_t* __restrict total_out,
                                             uint32_t* __restrict flagged) {
    __shared__ uint32_t sh[kScanWaves], s_flags[kScanWaves], s_ticket;
    __shared__ uint64_t sh64[kScanWaves];
    const uint32_t t = threadIdx.x;
    if (t == 0) s_ticket = scan_ticket(atomicAdd(state, 1ull), n, gridDim.x);
    __syncthreads();
    const uint32_t b = s_ticket;
    if (b == kNoTicket) return;  // the whole block
    unsigned long long* sums = state + 1;
    const uint64_t i = (uint64_t)b * kScanChunk + t;
    uint32_t w = 0, bw = 0;
    if (i < n) load(i, w, bw);
    uint32_t total;
    const uint32_t ex = block_exclusive_scan32(w, sh, total);
    if (t == 0) atomicExch(&sums[b], kScanReady | total);
    asm volatile("" : : : "memory");  // published before the waits below
    uint64_t before = 0;
    for (uint32_t q = t; q < b; q += kScanBlock) {
        unsigned long long x;
        do x = __hip_atomic_load(&sums[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while (!(x & kScanReady));
        before += x & ~kScanReady;
    }
    before = dev::wave_sum(before);
    const uint32_t flags = dev::wave_sum(bw >> 31);
    if (dev::is_wave_leader()) {
        sh64[t >> 6] = before;
        s_flags[t >> 6] = flags;
    }
    __syncthreads();
    uint64_t off = 0;
    uint32_t n_flags = 0;
#pragma unroll
    for (int k = 0; k < kScanWaves; ++k) {
        off += sh64[k];
        n_flags += s_flags[k];
    }
    if (t == 0) {
        if (b == gridDim.x - 1u) *total_out = off + total;
        if (flagged && n_flags) atomicAdd(flagged, n_flags);
    }
    if (i < n) vmeta[i] = FLS_VMETA(off + ex, bw & 0xffu);
}

}  // namespace fls
