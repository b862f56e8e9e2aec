// Tickets of the offset scan's blocks.  The scan's state is caller's memory that
// an earlier launch has prepared, so what it holds is checked before a block
// indexes by it: a scan over memory that no planner has prepared for this many
// vectors, or that an earlier scan has used up, is refused block by block,
// before any store and any wait.
// Plain C++ (constexpr functions are callable from HIP device code), so the host
// tests run the rule on stale and arbitrary state.
#pragma once

#include <stdint.h>

namespace fls {

// Upper half of the ticket word of a state prepared for n_vec vectors: never 0,
// and another one for another number.
constexpr uint32_t scan_tag(uint64_t n_vec) { return (uint32_t)((n_vec * 0x9E3779B97F4A7C15ull) >> 32) | 1u; }

// The ticket word a planner leaves: the tag, no ticket drawn.
constexpr unsigned long long scan_ticket_word(uint64_t n_vec) { return (unsigned long long)scan_tag(n_vec) << 32; }

constexpr uint32_t kNoTicket = 0xffffffffu;

// The block number that the ticket word, as a block drew it, stands for in a
// scan of `blocks` blocks over n_vec vectors, or kNoTicket.
constexpr uint32_t scan_ticket(unsigned long long drawn, uint64_t n_vec, uint32_t blocks) {
    return (uint32_t)(drawn >> 32) == scan_tag(n_vec) && (uint32_t)drawn < blocks ? (uint32_t)drawn : kNoTicket;
}

}  // namespace fls
