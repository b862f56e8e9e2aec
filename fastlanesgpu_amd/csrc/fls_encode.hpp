// Internal helpers shared by the GPU encoders.  Internal to libfls.so.
#pragma once

#include "fls_runtime.hpp"

namespace fls {

// 32-bit words of scratch the plan/scan passes need for n_vec vectors.
uint64_t scratch_words(uint64_t n_vec);

// A planner's mark on a vector's width word: the scan counts the marked vectors.
constexpr uint32_t kScanFlag = 1u << 31;

// vmeta[i] = (exclusive prefix of words) << 8 | (bws[i] & 255); *d_total =
// sum(words); *d_flagged (optional) += vectors whose bws has kScanFlag.
int scan_offsets(const uint32_t* words, const uint32_t* bws, uint64_t n_vec, uint64_t* block_sums, fls_vmeta* vmeta,
                 uint64_t* d_total, hipStream_t s, uint32_t* d_flagged = nullptr);

}  // namespace fls
