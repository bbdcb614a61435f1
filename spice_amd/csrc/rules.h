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

constexpr int TILE_MAX = 1024;  // targets per tile (LDS accumulators)
constexpr int TILE_WIDE = 8192; // and of the wide tiles that static models may have step by step
constexpr int SEG_TILES = 3;    // log2 of the tiles of a row that lie side by side in the segment table (kernels.h, seg_at)

// Entries of the segment table for n rows and ntiles tiles.
inline std::uint64_t seg_entries( std::int64_t n, std::int64_t ntiles ) { return std::uint64_t( n ) * std::uint64_t( ( ( ntiles - 1 ) >> SEG_TILES ) + 1 ) << SEG_TILES; }

// Optional memory (bytes; faster forms of what a network can do without them): at most a fifth of
// the free memory less what the network still has to allocate. Small amounts are not asked about.
constexpr std::uint64_t OPTIONAL_SMALL = std::uint64_t( 64 ) << 20;
inline bool optional_fits( std::uint64_t bytes, std::uint64_t free, std::uint64_t reserve ) { return free > reserve && bytes <= ( free - reserve ) / 5; }
// The largest table of 8-byte entries of a served or batched net (whose memory is estimated before
// it is built; larger ones have 4-byte offsets).
constexpr std::uint64_t TABLE_BATCHED = std::uint64_t( 1 ) << 30;
// The most that the table of such a net of n neurons in ntiles tiles or fewer takes.
inline std::uint64_t batched_table_bytes( std::int64_t n, std::int64_t ntiles )
{
	std::uint64_t const bytes = 8 * seg_entries( n, ntiles );
	return bytes <= TABLE_BATCHED ? bytes : std::max( TABLE_BATCHED, 4 * std::uint64_t( n ) * std::uint64_t( ntiles + 1 ) );
}

// Width of `tiles` tiles over n neurons, in 64s.
inline std::int64_t tile_width( std::int64_t n, std::int64_t tiles ) { return ( ( n + tiles - 1 ) / tiles + 63 ) / 64 * 64; }

// Targets per delivery tile of a new network of n neurons, `targets` of which have inputs
// (csr_dev::targets). Two-kernel plastic steps: about two tiles per CU, of 256 at least.
inline int lazy_tile_w( std::int64_t n, int cus ) { return int( std::clamp<std::int64_t>( tile_width( n, 2 * cus ), 256, TILE_MAX ) ); }
// Windows (ahead: of several steps): one tile per CU, as
// every tile stages all of the window's arrivals and a wider one does it less often (synth 1e9:
// 29 us per step with 251 tiles of 3,200, 50 with 391 of 2,048), but none wider than its kernel
// takes; windows of several steps, whose accumulators take LDS per step, two per CU beyond that.
// The tiles without inputs cost little, except in
// windows of static models, whose workgroups of 1,024 threads (default_launch) have a CU each
// (Brunel, 100,000 and 40,000 neurons of which half have inputs, us per step: 3.4 and 1.9 with a
// tile per CU of all, 4.7 and 2.2 with one per CU of those). Where few neurons have inputs, the tiles
// are still those of all neurons, and the segment table has an entry for each of them and row: two per
// CU at most, or four with plasticity, whose tiles are the better the narrower, where the table takes
// at most 1 GB then (us per step, with up to two and up to four: brunel_3pop_stdp, 100,000 neurons of
// which 20,000 have inputs, 2.7 and 2.4; synth, 10,000 of 100,000 and of 300,000, 9.5 and 10.3, 12.1
// and 19.0).
constexpr std::uint64_t TABLE_SMALL = std::uint64_t( 1 ) << 30;
inline int window_tile_w( std::int64_t n, std::int64_t targets, bool plastic, bool ahead, int cus )
{
	std::int64_t const tiled = targets <= 0 || ( ahead && !plastic ) ? n : targets;
	std::int64_t const most = ahead || plastic ? TILE_MAX : 4 * 1024;
	std::int64_t w = tile_width( tiled, ahead && tile_width( tiled, cus ) > most ? 2 * cus : cus );
	if( 2 * targets < n )
	{
		if( plastic ) w = std::max( w, tile_width( n, 4 * cus ) );
		if( !plastic || 8 * seg_entries( n, ( n + w - 1 ) / w ) > TABLE_SMALL ) w = std::max( w, tile_width( n, 2 * cus ) );
	}
	return int( std::clamp<std::int64_t>( w, 64, most ) );
}

// One staged row segment of a chunk of spikes (window.h). Rows may name a target many times, so a
// segment may be longer than its tile is wide. step: of the window, in the bits that the source (of a
// plastic network: 24 bits) or the place leaves.
struct alignas( 16 ) win_seg
{
	std::int64_t at; // first target id in the row store (0 for an empty segment)
	std::int32_t src;
	std::int32_t len;

	template <bool plastic>
	HYBRID static win_seg of( std::int64_t at, std::int32_t len, std::int32_t src, std::int32_t step )
	{
		if( len <= 0 ) at = 0;
		return plastic ? win_seg{ at, src | step << 24, len } : win_seg{ at | std::int64_t( step ) << 48, src, len };
	}
	// Gives the step, and leaves place and source alone.
	template <bool plastic>
	HYBRID std::int32_t take_step()
	{
		std::int32_t const step = plastic ? src >> 24 : std::int32_t( at >> 48 );
		if( plastic )
			src &= ( 1 << 24 ) - 1;
		else
			at &= ( std::int64_t( 1 ) << 48 ) - 1;
		return step;
	}
};
} // namespace spice::hipx
