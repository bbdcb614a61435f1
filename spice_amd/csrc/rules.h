#pragma once
// Sizes of a network's buffers and windows that follow from its numbers alone (no HIP in here).
#include "dview.h"

#include <algorithm>
#include <cstdint>

namespace spice::hipx
{
constexpr int WINDOW_MAX = 15; // longest window (steps)

// The longest window of at most n steps: never a multiple of CLOCK_SLOTS, so that the clock a
// window writes is not the slot its workgroups read.
inline int window_steps( std::int64_t n )
{
	int const w = int( std::min<std::int64_t>( n, WINDOW_MAX ) );
	return w % CLOCK_SLOTS == 0 ? w - 1 : w;
}

// Entries of the spike ring of a net whose windows have at most wcap steps. The window from step T
// on clears the counters of the steps T + W .. T + W + wcap - 1, so none of these may be the entry of
// a step whose counter the same launch reads: T - delay is the oldest that it delivers, and T - n - 1
// (n <= wcap <= delay steps in the window before) the oldest that the spike log asks for. Four at
// least, so that with a delay of one step the entry of a step is its clock slot, known without
// reading the clock.
inline int ring_entries( int delay, int wcap ) { return std::max( 4, delay + 2 * wcap + 1 ); }
} // namespace spice::hipx
