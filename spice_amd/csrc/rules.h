#pragma once
// Sizes of a network's buffers and windows that follow from its numbers alone (no HIP in here).
#include "dview.h"

#include <spice/util/host_defines.h>

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

// One staged row segment of a chunk of spikes (window.h). Rows may name a target many times, so a
// segment may be longer than its tile is wide.
struct alignas( 16 ) win_seg
{
	std::int64_t place; // first target id in the row store (0 for an empty segment), step of the window << 48
	std::int32_t src;
	std::int32_t len;

	HYBRID static win_seg of( std::int64_t at, std::int32_t len, std::int32_t src, std::int32_t step = 0 )
	{
		return { ( len > 0 ? at : 0 ) | std::int64_t( step ) << 48, src, len };
	}
	HYBRID std::int64_t at() const { return place & ( ( std::int64_t( 1 ) << 48 ) - 1 ); }
	HYBRID std::int32_t step() const { return std::int32_t( place >> 48 ); }
};
} // namespace spice::hipx
