// Internal helpers shared by the GPU encoders.  Internal to libfls.so.
#pragma once

#include "fls_runtime.hpp"
#include "fls_scan_ticket.hpp"

namespace fls {

// 32-bit words of scratch the plan/scan passes need for n_vec vectors.
uint64_t scratch_words(uint64_t n_vec);

// Vectors per block of the offset scan.
constexpr uint32_t kScanChunk = 1024;

// State of the offset scan (a ticket word, then a published sum per block): n
// words that the planner prepares with scan_clear before the scan is launched,
// and that one scan uses up.
struct ScanState {
    unsigned long long* p;
    uint32_t n;
    unsigned long long ticket;  // scan_ticket_word of the vectors
};

// Called by every work-item of a planner whose grid has at least a work-item
// per 8 vectors and 256 in all.
__device__ __forceinline__ void scan_clear(const ScanState& st) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < st.n) st.p[i] = i ? 0ull : st.ticket;
}

// The caller's scratch, cut up: per vector its width word and word count,
// then the scan's state.
struct EncodeScratch {
    uint32_t* bws;
    uint32_t* words;
    ScanState state;
};
EncodeScratch encode_scratch(void* d_scratch, uint64_t n_vec);

// A planner's mark on a vector's width word: the scan counts the marked vectors.
constexpr uint32_t kScanFlag = 1u << 31;

// vmeta[i] = (exclusive prefix of words) << 8 | (bws[i] & 255); *d_total =
// sum(words); *d_flagged (optional) += vectors whose bws has kScanFlag.
int scan_offsets(const EncodeScratch& e, uint64_t n_vec, fls_vmeta* vmeta, uint64_t* d_total, hipStream_t s,
                 uint32_t* d_flagged = nullptr);

}  // namespace fls
