#pragma once
// The window kernel: one launch simulates a window of W <= delay steps of a network.
//
// A spike emitted at step T reaches its targets at T + D, so the arrivals of the steps
// [T0, T0 + W), W <= D, are all known when the window starts, and a workgroup that owns a tile of
// target neurons needs nothing from the others inside the window: it delivers the arrivals of all
// W steps to its tile (LDS accumulators per step), then advances its neurons W steps with their
// state in registers, then appends the tile's spikes of every step to the ring. One launch, one
// chain of dependent loads (counts, ids, tile offsets, targets) and one read and write of the
// neuron state per W steps instead of per step, and W times the loads in flight per workgroup.
// With W = 1 (delay 1, or a receive() that reads its target) the workgroup delivers and then
// updates one step.
//
// What bounds it: small windows the chain of dependent loads and the launch (Vogels 1e8, one step:
// 3.5 us in the kernel, 3 us around it), larger ones the lines that a CU can have in flight (Vogels
// 1e9, delay 8: 27 of 36 us per window in the walk, 4,100 segments of 18 targets per tile), the largest the
// memory (Brunel 1e10). A row's segment inside a tile is walked by a group of 2^lg lanes (lg from the
// mean segment length), several segments per group in flight: no per-event search. What is read
// of a segment, see below.
//
// Accumulators: models with input classes (model.h) count the inputs of each class, others add
// the inputs up, in 64 bits (doubles, or fixed point). No 32-bit float atomics: ds_add_f32 takes
// 193 cycles per wave instruction on gfx950 (three per lane, whatever the addresses), ds_add_f64
// 21 and ds_add_u32 7 at random addresses, and was what a Vogels-Abbott delivery waited for.
#include "kernels.h"

#include <algorithm>

namespace spice::hipx
{
constexpr std::size_t LDS_PER_CU = 160 << 10;
constexpr std::size_t LDS_DYNAMIC = LDS_PER_CU - 4096; // beside what the window kernels declare themselves

// Lets `kernel` be launched with `bytes` of dynamic LDS. The limit belongs to the kernel, whichever
// networks run it, so it is set to the same for all of them.
inline void allow_lds( void const * kernel, std::size_t bytes )
{
	if( bytes > ( 64 << 10 ) ) SPICE_HIP( hipFuncSetAttribute( kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int( std::max( bytes, LDS_DYNAMIC ) ) ) );
}

constexpr int WIN_VEC = 4;   // consecutive targets a lane reads at once (the row store is padded by as many)
constexpr int WIN_TABLE = 64; // partial sums kept per input class

// What an input of attribute type T is accumulated in.
template <typename T, bool FIXED>
using win_acc = std::conditional_t<std::is_floating_point_v<T>, std::conditional_t<FIXED, long long, double>, T>;

// Models whose steps run as windows: static ones, and plastic ones whose passes apply every event.
template <typename Model>
inline constexpr bool windowed_v = !is_plastic_v<Model> || windowed_plastic_v<Model>;

// Longest window (steps, before the clock's restriction): 1 unless the delivery may run before its
// targets' update. Plastic models: an input is read beside the passes of the window before, and
// before this window's, so no event of its synapse may fall into the 2 W - 1 steps before it
// unless the input is dropped: a post event's target is refractory for R steps, and a pre event's
// source does not spike twice within R.
template <typename Model>
constexpr int longest_window_v = !overlap_capable_v<Model> ? 1
                                 : is_plastic_v<Model>     ? ( refractory_steps_v<typename Model::synapse> + 1 ) / 2
                                                           : WINDOW_MAX;

// WIN_VEC consecutive target ids, from any entry of the row store.
struct targets
{
	std::int32_t id[WIN_VEC];
};
__device__ inline targets load_targets( std::int32_t const * p )
{
	targets t;
	__builtin_memcpy( &t, p, sizeof( t ) ); // one 16-byte load (4-byte alignment suffices)
	return t;
}

// Orders a wave's LDS writes before its own later LDS reads (and reads before writes): the LDS
// serves a wave's instructions in order, so only the compiler has to keep them.
__device__ inline void wave_lds_fence()
{
	__builtin_amdgcn_fence( __ATOMIC_ACQ_REL, "wavefront" );
	__builtin_amdgcn_wave_barrier();
}

// ---- what a delivery reads of a row's segment in a tile --------------------------------------
// the row store; its halves, 4 or 8 per lane; segment records (the last two: models with input classes);
// the row store by offsets in place of the segment table, or by either
enum { IDS32, IDS16, IDS16X8, RECORDS, IDS32_OFFSETS, IDS32_ANY };
constexpr int SKIP_AT = 28; // IDS16X8: a staged segment's first place in its piece lies above its length (of 24 bits, as the segment table has)

// The low halves of the target ids, which tell a target within a tile (of at most 65,536); n of them
// are read at once: 4 from any place, 8 from a multiple of 8 (the store is padded by 8).
template <int n>
struct halves
{
	std::uint16_t id[n];
};
template <int n>
__device__ inline halves<n> load_halves( std::uint16_t const * p )
{
	halves<n> h;
	__builtin_memcpy( &h, n == 8 ? __builtin_assume_aligned( p, 16 ) : p, sizeof( h ) );
	return h;
}
// y / d for y < 2^25, d <= 2^7 and magic = 2^32 / d, rounded up (d = 1: magic 0).
HYBRID inline std::int32_t tile_quotient( std::uint32_t y, std::uint32_t magic )
{
	return magic ? std::int32_t( ( std::uint64_t( y ) * magic ) >> 32 ) : std::int32_t( y );
}
static inline __global__ __launch_bounds__( 256 ) void k_halves( std::int32_t const * col, std::int64_t n, std::uint16_t * out )
{
	for( std::int64_t i = ( std::int64_t( blockIdx.x ) * 256 + threadIdx.x ) * 8; i < n; i += std::int64_t( gridDim.x ) * 256 * 8 )
	{
		// (the row store is padded by one piece of 4)
		targets const c[2] = { load_targets( col + i ), load_targets( col + std::min( i + 4, n ) ) };
		halves<8> h;
#pragma unroll
		for( int x = 0; x < 8; x++ ) h.id[x] = std::uint16_t( c[x / 4].id[x % 4] );
		__builtin_memcpy( out + i, &h, sizeof( h ) );
	}
}

// The segment table and the halves in one pass over the row store (Brunel 1e10: k_segments 12.2 ms and
// k_halves 12.3 on their own), one wave per row, 8 ids per lane; where each tile's segment starts is
// kept in LDS, ntiles + 1 words per wave. magic: 2^32 / (tile_w / 64), rounded up.
constexpr int PASS_TILES = 1023;
static inline __global__ __launch_bounds__( 256 ) void k_segments_halves( dview v, std::int64_t nnz, std::uint32_t magic, std::uint16_t * out )
{
	extern __shared__ std::uint32_t pass_lds[];
	std::int64_t const r = uniform64( ( std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x ) >> 6 );
	if( r >= v.N ) return;
	std::uint32_t * const starts = pass_lds + ( threadIdx.x >> 6 ) * ( v.ntiles + 1 );
	int const lane = lane_id();
	std::int64_t const lo = v.row_ptr[r];
	std::int32_t const len = std::int32_t( v.row_ptr[r + 1] - lo );
	// (exact: id / 64 is below 2^25 and tile_w / 64 at most 2^7)
	auto tile_of = [&]( std::int32_t id ) { return tile_quotient( std::uint32_t( id ) >> 6, magic ); };
	std::int32_t before = -1; // the tile of the id before the pass's
	for( std::int32_t e0 = 0; e0 < len; e0 += 64 * 8 )
	{
		std::int32_t const e = e0 + 8 * lane, mine = len - e < 8 ? ( len - e < 0 ? 0 : len - e ) : 8;
		// (pieces that start past the last edge hold nothing; the row store is padded by one piece)
		targets const c[2] = { load_targets( v.col + std::min( lo + e, nnz ) ), load_targets( v.col + std::min( lo + e + 4, nnz ) ) };
		halves<8> h;
		std::int32_t q[8];
#pragma unroll
		for( int x = 0; x < 8; x++ )
		{
			h.id[x] = std::uint16_t( c[x / 4].id[x % 4] );
			q[x] = x < mine ? tile_of( c[x / 4].id[x % 4] ) : v.ntiles;
		}
		if( mine == 8 )
			__builtin_memcpy( out + lo + e, &h, sizeof( h ) );
		else
			for( int x = 0; x < 7; x++ )
				if( x < mine ) out[lo + e + x] = h.id[x];
		std::int32_t p = std::int32_t( shfl_u32( std::uint32_t( q[7] ), lane - 1 ) );
		if( lane == 0 ) p = before;
#pragma unroll
		for( int x = 0; x < 8; x++ )
		{
			if( x < mine )
				for( std::int32_t t = p + 1; t <= q[x]; t++ ) starts[t] = std::uint32_t( e + x );
			p = q[x];
		}
		before = std::int32_t( __builtin_amdgcn_readlane( q[7], 63 ) );
	}
	std::int32_t const last = len > 0 ? tile_of( v.col[lo + len - 1] ) : -1;
	for( std::int32_t t = last + 1 + lane; t <= v.ntiles; t += 64 ) starts[t] = std::uint32_t( len );
	wave_lds_fence();
	for( std::int32_t t = lane; t < v.ntiles; t += 64 )
		v.segs[seg_at( v, r, t )] = std::uint64_t( lo + starts[t] ) | std::uint64_t( starts[t + 1] - starts[t] ) << 40;
}

// ---- segment records -------------------------------------------------------------------------
// For models with input classes a delivery needs of a row's segment in a tile only the targets, and
// those fit 16 bits inside a tile. Where segments are short and the network runs step by step, each
// (row, tile) gets a record of 2^lg bytes, 16 to 64: the segment's length, then its targets less
// the tile's start. A segment then costs one aligned read instead of its bounds and, after them, an
// unaligned piece of the row store; the chain of dependent accesses that bounds such a step loses
// two links, as the arrivals' ids are read beside their count. A segment that does not fit has
// REC_LONG for its length, then (at bytes 4 and 8) its true length and its place in col.
// us per step, without and with: synth 1e9 (5 targets per segment) 30.1, 21.7; Vogels 1e8 7.8, 6.5.
// Windows of several steps gain less (Vogels 1e9, delay 8: 7.55, 7.0) than the records cost where
// a network is built (5 ms), so they have none. Spike lists per tile instead of one per step, which
// need no atomic, were slower to read (8.5 and 28.3).
constexpr std::uint16_t REC_LONG = 0xffff;
HYBRID constexpr int rec_capacity( int lg ) { return ( 1 << lg ) / 2 - 1; }
// (A row's record of a tile lies where the segment table has their entry, see seg_at: synth 1e9, 3.3 GB
// of records, 21.7 us per step with 8 tiles side by side, 21.9 with 4, 23.3 with 32, 24.0 row by row.)
struct alignas( 16 ) rec_part // 16 bytes of a record
{
	std::uint16_t t[8];
};

// The number of the x-th of the BS >> gl groups of lanes that deliver records to a tile: the tiles
// that share lines begin at different arrivals, so that not all of them wait for the same line's
// first read (synth 1e9, 24.0 us per step, 25.0 without).
template <int BS>
__device__ inline int rec_group( int x, int gl, std::int32_t tile )
{
	int const ng = BS >> gl;
	return ( x + ( ( tile & ( ( 1 << SEG_TILES ) - 1 ) ) * ng >> SEG_TILES ) ) & ( ng - 1 );
}

// Builds the records, one wave per row, a lane per tile; *longs counts the segments that do not fit.
static inline __global__ __launch_bounds__( 256 ) void k_records( dview v, unsigned char * recs, int lg, unsigned long long * longs )
{
	std::int64_t const r = uniform64( ( std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x ) >> 6 );
	if( r >= v.N ) return;
	std::int64_t const nnz = v.row_ptr[v.N];
	int const cap = rec_capacity( lg );
	for( int t = lane_id(); t < v.ntiles; t += 64 )
	{
		segment const s = segment_of( v, r, t );
		std::int64_t const a = s.at;
		std::int32_t const len = s.len, t0 = t * v.tile_w;
		rec_part * const out = reinterpret_cast<rec_part *>( recs + ( seg_at( v, r, t ) << lg ) );
		if( len > cap )
		{
			rec_part p{};
			p.t[0] = REC_LONG;
			__builtin_memcpy( &p.t[2], &len, 4 );
			__builtin_memcpy( &p.t[4], &a, 8 );
			out[0] = p;
			atomicAdd( longs, 1ull );
			continue;
		}
		std::int32_t before = len; // what the part's first 16 bits hold: the length, then the target before the part's
		for( int i = 0; i < 1 << ( lg - 4 ); i++ )
		{
			// entries 8 i - 1 .. 8 i + 6 of the segment; a piece that starts past the last edge holds
			// none of them (the row store is padded by one piece)
			targets const c[2] = { load_targets( v.col + std::min( a + 8 * i, nnz ) ), load_targets( v.col + std::min( a + 8 * i + 4, nnz ) ) };
			rec_part p;
			p.t[0] = std::uint16_t( before );
#pragma unroll
			for( int x = 0; x < 7; x++ ) p.t[x + 1] = std::uint16_t( c[x / 4].id[x % 4] - t0 ); // (past the segment's end: never read as a target)
			before = c[1].id[3] - t0;
			out[i] = p;
			if( 8 * i + 7 >= len ) break;
		}
	}
}

template <typename Model, bool FIXED>
struct window_lds
{
	using N = typename Model::neuron;
	static constexpr int classes = input_classes_v<Model>;
	// accumulators per neuron and step: a count per class, or a sum per received attribute
	static constexpr int nacc = classes > 0 ? classes : ( __builtin_popcount( receive_mask_v<N> ) > 0 ? __builtin_popcount( receive_mask_v<N> ) : 1 );
	using word = std::conditional_t<( classes > 0 ), std::uint32_t, unsigned long long>;
	// byte offsets of the dynamic LDS: staged segments, accumulators [W][nacc][tile_w], spike
	// masks [W][tile_w / 64], and the masks' exclusive prefix counts
	HYBRID static std::size_t acc_at( int bs ) { return sizeof( win_seg ) * std::size_t( bs ); }
	HYBRID static std::size_t mask_at( int bs, int tw, int w ) { return acc_at( bs ) + sizeof( word ) * std::size_t( nacc ) * std::size_t( tw ) * std::size_t( w ); }
	// rows of masks: the window's steps, then (plastic models) the arriving rows and the spiking targets
	HYBRID static int rows( int w ) { return w + ( is_plastic_v<Model> ? 2 : 0 ); }
	HYBRID static std::size_t pre_at( int bs, int tw, int w ) { return mask_at( bs, tw, w ) + 8 * std::size_t( tw / 64 ) * std::size_t( rows( w ) ); }
	HYBRID static std::size_t bytes( int bs, int tw, int w ) { return pre_at( bs, tw, w ) + 4 * std::size_t( tw / 64 ) * std::size_t( rows( w ) ); }
};

// Receive target inside a window (models without input classes): backend.atomic_add goes to the
// LDS accumulators of the event's step, reads of the target (W = 1 only) to its state.
template <typename Neuron, bool FIXED>
struct win_iter
{
	dview const * v;
	std::int32_t j, t0, stride;
	unsigned long long * acc; // [nacc][stride] of the event's step
	template <int I>
	__device__ auto get() const
	{
		using T = typename Neuron::template type<I>;
		constexpr std::uint32_t mask = receive_mask_v<Neuron>;
		constexpr int a = __builtin_popcount( mask & ( ( 1u << I ) - 1u ) );
		using A = win_acc<T, FIXED>;
		return tile_proxy<T, I, A, ( ( mask >> I ) & 1u ) != 0>{ v, j, reinterpret_cast<A *>( acc + a * stride ), t0, 0u };
	}
	__device__ uint_ id() const { return uint_( j ); }
};

// The sum of n inputs of class c, as adding them one after the other to zero gives it: for fp32
// from a table of the first sums.
template <typename Model, bool FIXED, typename T>
__device__ inline auto class_sum( std::uint32_t n, T value, float const * table, int shift )
{
	if constexpr( !std::is_floating_point_v<T> )
		return T( T( n ) * value );
	else if constexpr( FIXED )
		return (long long)( (unsigned long long)( n ) * (unsigned long long)( (long long)__builtin_rint( double( value ) * double( 1ull << shift ) ) ) );
	else
	{
		T x = table[n < WIN_TABLE ? n : WIN_TABLE - 1];
		for( std::uint32_t k = WIN_TABLE - 1; k < n; k++ ) x += value;
		return x;
	}
}

// The state of WIN_VEC consecutive synapses.
template <typename S>
struct synapses
{
	typename S::tuple_t s[WIN_VEC];
	__device__ void load( void * const * arr, std::int64_t i )
	{
		util::for_n<S::size>( [&]( auto I ) {
			using T = typename S::template type<I>;
			T t[WIN_VEC] = {};
			if constexpr( !is_factored_attr<S>( int( I ) ) ) __builtin_memcpy( t, static_cast<T const *>( arr[I] ) + i, sizeof( t ) );
#pragma unroll
			for( int x = 0; x < WIN_VEC; x++ ) std::get<I>( s[x] ) = t[x];
		} );
	}
};

__device__ inline std::uint32_t wave_inclusive_scan32( std::uint32_t x )
{
	int const l = lane_id();
#pragma unroll
	for( int d = 1; d < 64; d <<= 1 )
	{
		std::uint32_t const y = shfl_u32( x, l - d );
		if( l >= d ) x += y;
	}
	return x;
}

// Ring entry of the view's step. A ring of CLOCK_SLOTS entries (delay 1) has it at the clock's
// place, known before the clock is read.
__device__ inline std::int32_t window_entry( dview const & v ) { return v.rsize == CLOCK_SLOTS ? std::int32_t( v.ctl - v.ctl0 ) : v.ctl->rslot; }

// The window [T0, T0 + W) of the tile at place `pos` of v.tile_ids.
template <typename Model, bool FIXED, int BS, int FORM = IDS32>
__device__ inline void window_tile( dview const & v, std::int32_t pos, int W )
{
	constexpr bool REC = FORM == RECORDS;
	constexpr bool READS32 = FORM == IDS32 || FORM == IDS32_OFFSETS || FORM == IDS32_ANY;
	constexpr int KIND = FORM == IDS32_OFFSETS ? OFFSETS : FORM == IDS32_ANY ? ANY : TABLE;
	using N = typename Model::neuron;
	using S = typename Model::synapse;
	using L = window_lds<Model, FIXED>;
	using word = typename L::word;
	constexpr bool plastic = is_plastic_v<Model>;
	constexpr int nacc = L::nacc;
	constexpr std::uint32_t rmask = receive_mask_v<N>;

	extern __shared__ __align__( 16 ) unsigned char dyn[];
	__shared__ std::uint32_t base[WINDOW_MAX + 2];
	__shared__ std::uint32_t ev_total, spk_total;
	// fp32 input classes: the sum of the first k inputs of class c
	constexpr bool tables = L::classes > 0 && !FIXED;
	__shared__ float table[tables ? L::classes * WIN_TABLE : 1];

	int const tid = threadIdx.x, lane = lane_id();
	std::int32_t const tws = v.tile_w; // stride of the LDS arrays
	win_seg * const seg = reinterpret_cast<win_seg *>( dyn );
	word * const acc = reinterpret_cast<word *>( dyn + L::acc_at( BS ) );
	std::uint64_t * const masks = reinterpret_cast<std::uint64_t *>( dyn + L::mask_at( BS, tws, W ) );
	std::uint32_t * const wpre = reinterpret_cast<std::uint32_t *>( dyn + L::pre_at( BS, tws, W ) );

	std::int32_t const R = v.rsize;
	ctl_t const clk = *v.ctl;
	std::int64_t const T0 = clk.step;
	std::int32_t const slot0 = window_entry( v );
	int const lg = v.wlanes;
	auto entry = [&]( std::int32_t k ) { // ring entry of T0 + k, -D <= k < 2 * WINDOW_MAX
		std::int32_t const r = slot0 + k;
		return r < 0 ? r + R : r >= R ? r - R : r;
	};
	std::int32_t const tile = v.tile_ids[pos];
	bool const active = pos < v.nact; // some row has a target in the tile
	std::int32_t const t0 = tile * tws;
	std::int32_t const tw = ( v.N - t0 ) < tws ? ( v.N - t0 ) : tws;
	snn_info const info = info_of( v );

	// arrivals of the window's steps: lane q holds the count of step q, then the inclusive prefix.
	// Entries of steps before 0 are empty (counts start at zero).
	std::uint32_t incl = 0;
	// records: the first ids beside the count that tells which of them are this step's
	constexpr int REC_U = 4; // arrivals per group of lanes in flight
	std::int32_t early_id[REC_U] = {};
	if( active && lane < W ) incl = v.counts[entry( lane - v.D ) * COUNT_STRIDE];
	if constexpr( REC )
		if( active )
		{
			int const gl = v.rec_lg - 4;
#pragma unroll
			for( int u = 0; u < REC_U; u++ )
			{
				std::int32_t const k = u * ( BS >> gl ) + rec_group<BS>( tid >> gl, gl, tile );
				early_id[u] = v.ring[std::int64_t( entry( -v.D ) ) * v.N + ( k < v.N ? k : 0 )];
			}
		}
	// and the state of this thread's first neuron, used after the delivery
	typename N::tuple_t early{};
	bool const has_early = REC && tid < tw;
	if( has_early ) load_tuple<N>( early, v.na, t0 + tid );
	for( int x = tid; x < int( sizeof( word ) * nacc * std::size_t( tws ) * std::size_t( W ) / 16 ); x += BS )
		reinterpret_cast<uint4 *>( acc )[x] = uint4{ 0, 0, 0, 0 };
	if( tid == 0 ) ev_total = spk_total = 0;
	if constexpr( tables )
	{
		if( tid < L::classes )
		{
			float const x = float( N::input_value( tid, info ) );
			float t = 0.0f;
			for( int k = 0; k < WIN_TABLE; k++ )
			{
				table[tid * WIN_TABLE + k] = t;
				t += x;
			}
		}
	}
	if( W > 1 )
	{
#pragma unroll
		for( int d = 1; d < 16; d <<= 1 )
		{
			std::uint32_t const y = shfl_u32( incl, lane - d );
			if( lane >= d ) incl += y;
		}
	}
	std::int32_t total = __builtin_amdgcn_readlane( std::int32_t( incl ), W - 1 );

	// arrival k of the window: its source and step
	auto fetch_id = [&]( std::int32_t k, std::int32_t & q ) {
		std::int32_t const kk = k < total ? k : total - 1;
		q = 0;
		for( int m = 0; m < W - 1; m++ ) q += kk >= __builtin_amdgcn_readlane( std::int32_t( incl ), m ) ? 1 : 0;
		std::int32_t const below = std::int32_t( shfl_u32( incl, q - 1 ) ); // (every lane takes part)
		return v.ring[std::int64_t( entry( q - v.D ) ) * v.N + ( kk - ( q > 0 ? below : 0 ) )];
	};

	std::uint32_t ev = 0;
	if constexpr( REC )
		{
			// Delivery from records: a group of 2^(rec_lg - 4) lanes per arrival, 16 bytes each, U
			// arrivals per group in flight; nothing is staged.
			constexpr int U = REC_U;
			int const gl = v.rec_lg - 4, ng = BS >> gl, g = rec_group<BS>( tid >> gl, gl, tile ), l = tid & ( ( 1 << gl ) - 1 );
			auto const * recs = reinterpret_cast<rec_part const *>( v.recs );
			for( std::int32_t c = 0; c < total; c += U * ng )
			{
				rec_part r[U];
				std::int32_t at[U]; // where the counters of the arrival's class and step start
				bool ok[U];
				std::int32_t src[U];
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					std::int32_t const k = c + u * ng + g;
					ok[u] = k < total;
					std::int32_t const id = c == 0 ? early_id[u] : v.ring[std::int64_t( entry( -v.D ) ) * v.N + ( ok[u] ? k : 0 )];
					src[u] = ok[u] ? id : 0;
				}
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					r[u] = rec_part{};
					if( c + u * ng < total ) r[u] = recs[( seg_at( v, src[u], tile ) << gl ) + l];
					at[u] = N::input_class( src[u], info ) * tws;
				}
				if( c == 0 ) __syncthreads(); // the accumulators are clear
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					if( c + u * ng >= total ) continue;
					std::uint32_t head = r[u].t[0];
					if( gl ) head = shfl_u32( head, lane & ~( ( 1 << gl ) - 1 ) );
					int const len = ok[u] && head != REC_LONG ? int( head ) : 0;
					if( l == 0 ) ev += std::uint32_t( len );
					int const e0 = 8 * l - 1;
#pragma unroll
					for( int x = 0; x < 8; x++ )
						if( ( x > 0 || l > 0 ) && e0 + x < len ) atomicAdd( acc + ( at[u] + r[u].t[x] ), 1u );
					if( ok[u] && head == REC_LONG )
					{
						rec_part const whole = recs[seg_at( v, src[u], tile ) << gl];
						std::int32_t n;
						std::int64_t off;
						__builtin_memcpy( &n, &whole.t[2], 4 );
						__builtin_memcpy( &off, &whole.t[4], 8 );
						if( l == 0 ) ev += std::uint32_t( n );
						for( std::int32_t e = l; e < n; e += 1 << gl ) atomicAdd( acc + ( at[u] + v.col[off + e] - t0 ), 1u );
					}
				}
			}
			if( total == 0 ) __syncthreads(); // the accumulators are clear
			total = 0;                        // nothing is left for the walk below
		}

	// Delivery, wave by wave: a wave stages up to 64 of the window's arrivals at a time (one segment
	// each) in its own part of the LDS and walks them; the next ones' ids and segment bounds are
	// read beside the walk. No wave waits for another before the update.
	if constexpr( !REC ) __syncthreads(); // the accumulators are clear
	constexpr int NW = BS / 64;
	int const wave = tid >> 6;
	// arrivals per wave and round: few ones are spread over all waves
	std::int32_t const per = total >= 64 * NW ? 64 : ( total + NW - 1 ) / NW;
	std::int32_t k0 = wave * per;
	std::int32_t const mylane = lane < per ? lane : per - 1; // (the lanes past a round's arrivals repeat its last)
	if( k0 < total )
	{
		win_seg * const mine = seg + wave * 64;
		std::int32_t src, q = 0, src_n = 0, q_n = 0;
		packed_segment ps;
		auto fetch_seg = [&]() { ps = load_segment<KIND>( v, src, tile ); };
		src = fetch_id( k0 + mylane, q );
		fetch_seg();
		if( k0 + NW * per < total ) src_n = fetch_id( k0 + NW * per + mylane, q_n );

		int const G = 1 << lg, g = lane >> lg, l = lane & ( G - 1 ), ng = 64 >> lg;
		for( ; k0 < total; k0 += NW * per )
		{
			std::int32_t const cnt = ( total - k0 ) < per ? ( total - k0 ) : per;
			segment const sg = unpack_segment<KIND>( v, ps );
			std::int64_t const a = sg.at;
			std::int32_t const len = lane < cnt ? sg.len : 0;
			if constexpr( L::classes > 0 )
			{
				// in the place of the source: where the class's counters of the step start (for target 0).
				// IDS16X8: from the piece that the segment begins in, its place there above the length
				std::int32_t const at = ( q * nacc + N::input_class( src, info ) ) * tws - ( READS32 ? t0 : 0 );
				std::int32_t const skip = FORM == IDS16X8 && len > 0 ? std::int32_t( a ) & 7 : 0;
				mine[lane] = win_seg{ len > 0 ? a & ~std::int64_t( FORM == IDS16X8 ? 7 : 0 ) : 0, at, ( len + skip ) | skip << SKIP_AT };
			}
			else
				mine[lane] = win_seg::of<plastic>( a, len, src, q );
			ev += std::uint32_t( len );
			wave_lds_fence();
			if( k0 + NW * per < total )
			{
				src = src_n;
				q = q_n;
				fetch_seg();
				if( k0 + 2 * NW * per < total ) src_n = fetch_id( k0 + 2 * NW * per + mylane, q_n );
			}
			constexpr int V = FORM == IDS16X8 ? 8 : WIN_VEC; // entries per lane
			constexpr int U = plastic ? 2 : 4; // segments per group in flight (with weights, 4 measured 3 % slower)
			for( std::int32_t c = 0; c < cnt; c += U * ng )
			{
				win_seg r[U];
				std::int32_t len[U], step[U], most = 0;
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					std::int32_t const k = c + u * ng + g;
					r[u] = mine[k & 63]; // (records from cnt on are empty)
					len[u] = k < 64 ? ( FORM == IDS16X8 ? r[u].len & ( ( 1 << SKIP_AT ) - 1 ) : r[u].len ) : 0;
					step[u] = FORM == IDS16X8 ? r[u].len >> SKIP_AT : 0; // (its skip)
					if constexpr( L::classes == 0 ) step[u] = r[u].template take_step<plastic>();
					most = len[u] > most ? len[u] : most;
				}
				for( std::int32_t e = l * V;; e += G * V )
				{
					// (past a segment's end its first entries are read, at valid addresses, and ignored)
					if constexpr( L::classes > 0 && ( FORM == IDS16 || FORM == IDS16X8 ) )
					{
						halves<V> j[U];
#pragma unroll
						for( int u = 0; u < U; u++ ) j[u] = load_halves<V>( v.col16 + r[u].at + ( e < len[u] ? e : 0 ) );
#pragma unroll
						for( int u = 0; u < U; u++ )
#pragma unroll
							for( int x = 0; x < V; x++ )
								if( e + x < len[u] && ( V == WIN_VEC || e + x >= step[u] ) ) atomicAdd( acc + ( r[u].src + ( ( j[u].id[x] - t0 ) & 0xffff ) ), 1u );
						if( e - l * V + G * V >= most ) break;
						continue;
					}
					targets j[U];
#pragma unroll
					for( int u = 0; u < U; u++ )
						if constexpr( FORM == IDS16 )
						{
							halves<V> const low = load_halves<V>( v.col16 + r[u].at + ( e < len[u] ? e : 0 ) );
#pragma unroll
							for( int x = 0; x < V; x++ ) j[u].id[x] = t0 + ( ( low.id[x] - t0 ) & 0xffff );
						}
						else
							j[u] = load_targets( v.col + r[u].at + ( e < len[u] ? e : 0 ) );
					synapses<S> sy[U];
					if constexpr( plastic )
					{
#pragma unroll
						for( int u = 0; u < U; u++ ) sy[u].load( v.sa, r[u].at + ( e < len[u] ? e : 0 ) );
					}
#pragma unroll
					for( int u = 0; u < U; u++ )
#pragma unroll
						for( int x = 0; x < WIN_VEC; x++ )
						{
							if( e + x >= len[u] ) continue;
							if constexpr( L::classes > 0 )
								atomicAdd( acc + ( r[u].src + j[u].id[x] ), 1u );
							else
							{
								int const s = step[u];
								tile_backend<FIXED> bak{ make_backend<FIXED>( v, std::uint32_t( r[u].src ), std::uint32_t( j[u].id[x] ), std::uint32_t( T0 + s ), util::TAG_RECEIVE ) };
								win_iter<N, FIXED> dst{ &v, j[u].id[x], t0, tws, acc + s * ( nacc * tws ) };
								if constexpr( plastic )
									deliver_event<N>( r[u].src, dst, reg_iter<typename S::tuple_t>{ sy[u].s[x], std::uint32_t( r[u].at + e + x ) }, info, bak );
								else
									deliver_event<N>( r[u].src, dst, no_syn_iter{}, info, bak );
							}
						}
					if( e - l * WIN_VEC + G * WIN_VEC >= most ) break;
				}
			}
			wave_lds_fence(); // the next round overwrites the records
		}
	}
	__syncthreads(); // the sums are complete

	// the tile's neurons, W steps each
	int const nw = tws >> 6;
	for( int x = tid; x < tws; x += BS )
	{
		std::uint32_t spikes = 0; // bit q: spiked at T0 + q
		if( x < tw )
		{
			std::int64_t const i = t0 + x;
			typename N::tuple_t s = early;
			if( !has_early || x != tid ) load_tuple<N>( s, v.na, i );
			// plastic models: the arrivals of this neuron's own spikes (of the steps from T0 - D), its
			// traces, and the history words that the window's steps go to
			std::uint32_t arrivals = 0;
			float xt = 0.0f, yt = 0.0f, x0 = 0.0f;
			unsigned long long h0 = 0, h1 = 0;
			std::int64_t const hw0 = ( T0 & ( HISTORY - 1 ) ) >> 6, hw1 = ( ( T0 + W - 1 ) & ( HISTORY - 1 ) ) >> 6;
			bool has_out = false, has_in = false;
			if constexpr( plastic )
			{
				int const b = int( ( T0 - v.D ) & ( HISTORY - 1 ) ), sh = b & 63;
				unsigned long long a = v.hring[std::int64_t( b >> 6 ) * v.N + i] >> sh;
				if( sh + W > 64 ) a |= v.hring[std::int64_t( ( ( b >> 6 ) + 1 ) & ( HWORDS - 1 ) ) * v.N + i] << ( 64 - sh );
				arrivals = std::uint32_t( a ) & ( ( 1u << W ) - 1u );
				h0 = v.hring[hw0 * v.N + i];
				if( hw1 != hw0 ) h1 = v.hring[hw1 * v.N + i];
				xt = v.xtr[( clk.wseq & 3 ) * std::int64_t( v.N ) + i];
				yt = v.ytr[( clk.wseq & 3 ) * std::int64_t( v.N ) + i];
				x0 = xt;
				has_out = v.hasp[i];
				has_in = v.tp_ptr[i + 1] > v.tp_ptr[i];
			}
			float sum = clk.sum, c = clk.c;
			for( int q = 0; q < W; q++ )
			{
				// the step's compensated dt, then the next step's clock: exactly kahan_sum::add
				float const dt = v.DT - c;
				float const t = sum + dt;
				c = ( t - sum ) - dt;
				sum = t;
				std::int64_t const T = T0 + q;
				// the step's inputs; a split receive()'s gate is tested on the state that the
				// delivery's receive() would have read
				bool open = true;
				if constexpr( gated_receive_v<N> ) open = N::accepts( reg_iter<typename N::tuple_t>{ s, std::uint32_t( i ) } );
				util::for_n<N::size>( [&]( auto I ) {
					if constexpr( ( ( rmask >> I ) & 1u ) != 0 )
					{
						using A = typename N::template type<I>;
						using AC = std::conditional_t<std::is_floating_point_v<A>, std::conditional_t<FIXED, long long, A>, A>;
						AC in = AC( 0 );
						if constexpr( L::classes > 0 )
							util::for_n<L::classes>( [&]( auto C ) {
								if constexpr( N::input_attr[C] == int( I ) )
									in = AC( in + class_sum<Model, FIXED>( acc[( q * nacc + C ) * tws + x], A( N::input_value( C, info ) ),
									                                       table + ( tables ? C * WIN_TABLE : 0 ), v.shift ) );
							} );
						else
						{
							constexpr int a = __builtin_popcount( rmask & ( ( 1u << I ) - 1u ) );
							in = AC( reinterpret_cast<win_acc<A, FIXED> const *>( acc + ( q * nacc + a ) * tws )[x] );
						}
						if constexpr( std::is_floating_point_v<A> && FIXED )
						{
							if( open ) std::get<I>( s ) = std::get<I>( s ) + float( in ) * __builtin_ldexpf( 1.0f, -v.shift );
						}
						else
						{
							if( open ) std::get<I>( s ) = A( std::get<I>( s ) + in );
						}
					}
				} );
				auto bak = make_backend<FIXED>(
				    v, std::uint32_t( i ), std::uint32_t( T ), std::uint32_t( std::uint64_t( T ) >> 32 ), util::TAG_NEURON_UPDATE );
				bool const spiked = N::update( reg_iter<typename N::tuple_t>{ s, std::uint32_t( i ) }, dt, info, bak );
				if( spiked ) spikes |= 1u << q;
				if constexpr( plastic )
				{
					float const d = S::trace_decay( dt );
					xt = fmaf( xt, d, ( arrivals >> q ) & 1u ? 1.0f : 0.0f );
					yt = fmaf( yt, d, spiked ? 1.0f : 0.0f );
				}
			}
			store_tuple<N>( s, v.na, i );
			if constexpr( plastic )
			{
				// the steps' history bits (over those of the steps HISTORY before)
				unsigned long long const all = ( 1ull << W ) - 1ull;
				int const sh = int( T0 & 63 );
				unsigned long long const n0 = ( h0 & ~( all << sh ) ) | ( (unsigned long long)( spikes ) << sh );
				if( n0 != h0 ) v.hring[hw0 * v.N + i] = n0;
				if( hw1 != hw0 )
				{
					unsigned long long const n1 = ( h1 & ~( all >> ( 64 - sh ) ) ) | ( (unsigned long long)( spikes ) >> ( 64 - sh ) );
					if( n1 != h1 ) v.hring[hw1 * v.N + i] = n1;
				}
				std::int64_t const nx = ( ( clk.wseq + 1 ) & 3 ) * std::int64_t( v.N ) + i, par = ( clk.wseq & 1 ) * std::int64_t( v.N ) + i;
				v.xtr[nx] = xt;
				v.ytr[nx] = yt;
				v.fl8[par] = std::uint8_t( arrivals ? __builtin_ctz( arrivals ) + 1 : 0 );
				std::uint32_t const x0b = __builtin_bit_cast( std::uint32_t, x0 );
				v.xpost[par] = arrivals ? X_ARRIVED : x0b == X_ARRIVED ? 0x7fc00000u : x0b;
				v.sp8[par] = std::uint8_t( spikes ? __builtin_ctz( spikes ) + 1 : 0 );
				if( has_out && arrivals ) spikes |= 1u << W;
				if( has_in && ( spikes & std::uint32_t( all ) ) ) spikes |= 2u << W;
			}
		}
		for( int q = 0; q < L::rows( W ); q++ )
		{
			std::uint64_t const m = ballot( ( spikes >> q ) & 1u );
			if( lane == 0 ) masks[q * nw + ( x >> 6 )] = m;
		}
	}
	{
		std::uint32_t const t = wave_inclusive_scan32( ev );
		if( lane == 63 && t ) atomicAdd( &ev_total, t );
	}
	__syncthreads();

	// a wave per step: the masks' prefix counts, and one atomic reserves the tile's ring places
	for( int q = tid >> 6; q < L::rows( W ); q += BS / 64 )
	{
		std::uint32_t const n = lane < nw ? std::uint32_t( __popcll( masks[q * nw + lane] ) ) : 0u;
		std::uint32_t const in = wave_inclusive_scan32( n );
		if( lane < nw ) wpre[q * nw + lane] = in - n;
		if( lane == 63 && in )
		{
			std::uint32_t * count = &v.counts[entry( q < W ? q : 0 ) * COUNT_STRIDE];
			if constexpr( plastic )
				if( q >= W ) count = ( q == W ? v.fl_count : v.po_count ) + ( clk.wseq & 3 );
			base[q] = atomicAdd( count, in );
			if( q < W ) atomicAdd( &spk_total, in );
		}
	}
	if( tile == 0 )
	{
		// the counters of the steps after the window (no workgroup of this launch reads those
		// entries: ring_entries), and the clock of the step after it
		if( tid < v.wcap ) v.counts[entry( W + tid ) * COUNT_STRIDE] = 0;
		if( tid == 0 )
		{
			float sum = clk.sum, c = clk.c;
			for( int q = 0; q < W; q++ )
			{
				float const y = v.DT - c;
				float const t = sum + y;
				c = ( t - sum ) - y;
				sum = t;
			}
			ctl_t * const next = v.ctl0 + ( ( v.ctl - v.ctl0 + W ) & ( CLOCK_SLOTS - 1 ) );
			next->c = c;
			next->sum = sum;
			next->step = T0 + W;
			next->rslot = entry( W );
			if constexpr( plastic )
			{
				next->wseq = clk.wseq + 1;
				next->wprev = W;
				next->psum = clk.sum;
				next->pc = clk.c;
				// the next window's list counters (last read by the passes of window wseq - 3)
				v.fl_count[( clk.wseq + 1 ) & 3] = 0;
				v.po_count[( clk.wseq + 1 ) & 3] = 0;
			}
		}
	}
	__syncthreads();
	for( int x = tid; x < tws; x += BS )
		for( int q = 0; q < L::rows( W ); q++ )
		{
			std::uint64_t const m = masks[q * nw + ( x >> 6 )];
			if( !( ( m >> lane ) & 1ull ) ) continue;
			std::int32_t * list = v.ring + std::int64_t( entry( q < W ? q : 0 ) ) * v.N;
			if constexpr( plastic )
				if( q >= W ) list = ( q == W ? v.fl_id : v.po_id ) + ( clk.wseq & 1 ) * std::int64_t( v.N );
			list[base[q] + wpre[q * nw + ( x >> 6 )] + std::uint32_t( lanes_below( m ) )] = t0 + x;
		}
	if( tid == 0 )
	{
		// this tile's statistics slot, no result awaited
		if( ev_total ) atomicAdd( &v.bstats[std::int64_t( pos ) * NSTAT + ST_EVENTS], static_cast<unsigned long long>( ev_total ) );
		if( spk_total ) atomicAdd( &v.bstats[std::int64_t( pos ) * NSTAT + ST_SPIKES], static_cast<unsigned long long>( spk_total ) );
	}
}

// Workgroups go to the XCDs round robin, each with an L2 of its own: workgroup b of n takes the
// place that gives each XCD one contiguous range of tiles, so a spike's tile offsets and the
// memory lines shared by neighbouring segments of its row are fetched into one L2.
constexpr int XCDS = 8;
__device__ inline std::int32_t xcd_place( std::int32_t b, std::int32_t n )
{
	std::int32_t const x = b % XCDS, per = n / XCDS, more = n % XCDS;
	return x * per + ( x < more ? x : more ) + b / XCDS;
}

// Plasticity of the window before the view's step: a pre pass over the plastic slots of the rows
// whose spike arrived in it, and a post pass over the incoming plastic synapses (by-target index) of
// the neurons that spiked in it, leaving out sources that arrived in it (the pre pass has those).
// Refractory endpoints have at most one arrival and one spike each in a window, so a synapse has at
// most a pre event (at step a) and a post event (at step b), applied in step order in one
// read-modify-write; the traces at a and b are the per-step recurrence continued from the window's
// start. One index space of work items, (row, part) then (target, part), taken round robin by the
// waves of workgroups blk, blk + nblk, ...; statistics go to slots slot0 + blk. Bound by the rate
// of random memory lines, 43 to 53 G of 64 bytes a second on the whole card: the post pass's weights.
template <typename Model, bool FIXED>
__device__ inline void window_passes( dview const & v, std::int64_t blk, std::int64_t nblk, std::int64_t slot0 )
{
	using S = typename Model::synapse;
	constexpr int U = 4; // synapses per lane in flight
	ctl_t const clk = *v.ctl;
	int const W = clk.wprev;
	std::int64_t const Tp = clk.step - W; // the window's first step
	if( W == 0 || *v.caught == clk.step - 1 ) return;
	std::int32_t const k = clk.wseq - 1; // its number
	std::int64_t const par = ( k & 1 ) * std::int64_t( v.N ), tr = ( k & 3 ) * std::int64_t( v.N );
	std::int64_t const npre = std::int64_t( v.fl_count[k & 3] ) * v.fparts;
	std::int64_t const nitems = npre + std::int64_t( v.po_count[k & 3] ) * v.pparts;
	snn_info const info = info_of( v );
	int const lane = lane_id();
	// lane q: the dt of the window's step q and the traces' decay in it
	float decay = 0.0f, dts = 0.0f;
	{
		float sum = clk.psum, c = clk.pc;
		for( int q = 0; q < W; q++ )
		{
			float const dt = v.DT - c;
			float const t = sum + dt;
			c = ( t - sum ) - dt;
			sum = t;
			if( lane == q )
			{
				dts = dt;
				decay = S::trace_decay( dt );
			}
		}
	}
	auto decay_of = [&]( int q ) { return __builtin_bit_cast( float, __builtin_amdgcn_readlane( __builtin_bit_cast( std::int32_t, decay ), q ) ); };
	auto backend = [&]( std::int64_t e, int q ) {
		return make_backend<FIXED>( v, std::uint32_t( e ), std::uint32_t( std::uint64_t( e ) >> 32 ), std::uint32_t( Tp + q ), util::TAG_SYNAPSE_UPDATE );
	};
	std::int64_t const wave0 = uniform64( ( blk * blockDim.x + threadIdx.x ) >> 6 );
	std::int64_t const nwaves = nblk * ( blockDim.x >> 6 );
	unsigned long long touched = 0, written = 0, words = 0, rows = 0;
	auto dt_of = [&]( int q ) { return __builtin_bit_cast( float, shfl_u32( __builtin_bit_cast( std::uint32_t, dts ), q < 0 ? 0 : q ) ); };
	// one event (of step q, whose dt is given where the rule takes it); counts it, and whether it
	// changed the synapse
	auto event = [&]( typename S::tuple_t & sy, std::int64_t e, int q, float dt, bool pre, bool post, float x, float y ) {
		typename S::tuple_t const before = sy;
		auto bak = backend( e, q );
		if constexpr( factored_v<Model> )
		{
			std::get<S::pre_trace>( sy ) = x;
			std::get<S::post_trace>( sy ) = y;
			S::on_event( reg_iter<typename S::tuple_t>{ sy, std::uint32_t( e ) }, pre, post, dt, info, bak );
		}
		else
			S::on_event( reg_iter<typename S::tuple_t>{ sy, std::uint32_t( e ) }, pre, post, x, y, info, bak );
		touched++;
		written += same_bits<S>( before, sy ) ? 0 : 1;
	};
	for( std::int64_t it = wave0; it < nitems; it += nwaves )
	{
		if( it < npre )
		{
			std::int64_t const f = it / v.fparts;
			std::int64_t const p = it - f * v.fparts;
			std::int32_t const s = uniform( v.fl_id[par + f] );
			int const a = uniform( v.fl8[par + s] ) - 1;
			std::int64_t const r0 = v.row_ptr[s];
			std::int64_t const lo = r0 + v.pl_lo[s], hi = r0 + v.pl_hi[s];
			std::int64_t const chunk = ( ( hi - lo + v.fparts - 1 ) / v.fparts + 63 ) & ~std::int64_t( 63 );
			std::int64_t const beg = lo + p * chunk;
			std::int64_t const end = beg + chunk < hi ? beg + chunk : hi;
			// lane q: the row's pre trace after step q
			float xs = 0.0f;
			{
				float x = v.xtr[tr + s];
				for( int q = 0; q < W; q++ )
				{
					x = fmaf( x, decay_of( q ), q == a ? 1.0f : 0.0f );
					if( lane == q ) xs = x;
				}
			}
			for( std::int64_t first = beg; first < end; first += 64 * U )
			{
				std::int32_t j[U];
				bool ok[U];
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					std::int64_t const e = first + lane + 64 * u;
					ok[u] = e < end;
					j[u] = v.col[ok[u] ? e : beg];
				}
				typename S::tuple_t sy[U];
				int b[U];
				float y[U];
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					std::int64_t const e = first + lane + 64 * u;
					ok[u] = ok[u] && S::plastic( s, j[u], info );
					if constexpr( !has_inert_v<S> ) load_synapse<S>( sy[u], v.sa, ok[u] ? e : beg );
					b[u] = int( v.sp8[par + j[u]] ) - 1;
					y[u] = v.ytr[tr + j[u]];
				}
				// the targets' post traces after step a, the row's pre trace after their steps b
				for( int q = 0; q <= a; q++ )
				{
					float const dq = decay_of( q );
#pragma unroll
					for( int u = 0; u < U; u++ ) y[u] = fmaf( y[u], dq, q == b[u] ? 1.0f : 0.0f );
				}
				float xb[U], db[U];
				float const da = dt_of( a );
#pragma unroll
				for( int u = 0; u < U; u++ ) db[u] = factored_v<Model> ? dt_of( b[u] ) : 0.0f;
#pragma unroll
				for( int u = 0; u < U; u++ ) xb[u] = __builtin_bit_cast( float, shfl_u32( __builtin_bit_cast( std::uint32_t, xs ), b[u] < 0 ? 0 : b[u] ) );
				if constexpr( has_inert_v<S> )
				{
					// events that cannot change the synapse do not read it
#pragma unroll
					for( int u = 0; u < U; u++ )
					{
						if( !ok[u] ) continue;
						bool const post = b[u] >= 0;
						if( b[u] == a ? S::inert( true, true, xb[u], y[u], da ) : S::inert( true, false, 0.0f, y[u], da ) && ( !post || S::inert( false, true, xb[u], 0.0f, db[u] ) ) )
						{
							ok[u] = false;
							touched += post && b[u] != a ? 2 : 1;
						}
					}
#pragma unroll
					for( int u = 0; u < U; u++ )
						if( ok[u] ) load_synapse<S>( sy[u], v.sa, first + lane + 64 * u );
				}
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					if( !ok[u] ) continue;
					std::int64_t const e = first + lane + 64 * u;
					typename S::tuple_t const before = sy[u];
					bool const post = b[u] >= 0;
					if( post && b[u] < a ) event( sy[u], e, b[u], db[u], false, true, xb[u], 0.0f );
					event( sy[u], e, a, da, true, b[u] == a, b[u] == a ? xb[u] : 0.0f, y[u] );
					if( post && b[u] > a ) event( sy[u], e, b[u], db[u], false, true, xb[u], 0.0f );
					store_synapse<S>( before, sy[u], v.sa, e );
				}
			}
			if( lane == 0 )
			{
				if( end > beg ) words += std::uint64_t( end - beg ); // target ids
				if( p == 0 ) rows++;
			}
		}
		else
		{
			std::int64_t const g = it - npre;
			std::int64_t const f = g / v.pparts;
			std::int64_t const p = g - f * v.pparts;
			std::int32_t const d = uniform( v.po_id[par + f] );
			int const b = uniform( v.sp8[par + d] ) - 1;
			float const dt_b = dt_of( b );
			std::int64_t const lo = v.tp_ptr[d], hi = v.tp_ptr[d + 1];
			std::int64_t const chunk = ( ( hi - lo + v.pparts - 1 ) / v.pparts + 63 ) & ~std::int64_t( 63 );
			std::int64_t const beg = lo + p * chunk;
			std::int64_t const end = beg + chunk < hi ? beg + chunk : hi;
			for( std::int64_t first = beg; first < end; first += 64 * U )
			{
				tp_entry te[U];
				bool ok[U];
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					std::int64_t const x = first + lane + 64 * u;
					ok[u] = x < end;
					te[u] = v.tp_ent[ok[u] ? x : beg];
				}
				// the source's trace at the window's start, or that its spike arrived in the window
				std::int64_t e[U];
				float xv[U];
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					e[u] = tp_place( te[u] );
					std::uint32_t const x = v.xpost[par + tp_src( te[u] )];
					ok[u] = ok[u] && x != X_ARRIVED;
					xv[u] = __builtin_bit_cast( float, x );
				}
				typename S::tuple_t sy[U];
				if constexpr( !has_inert_v<S> )
				{
					// (few sources arrived: their weights are read for nothing)
#pragma unroll
					for( int u = 0; u < U; u++ ) load_synapse<S>( sy[u], v.sa, e[u] );
				}
				for( int q = 0; q <= b; q++ )
				{
					float const dq = decay_of( q );
#pragma unroll
					for( int u = 0; u < U; u++ ) xv[u] = fmaf( xv[u], dq, 0.0f ); // (no arrival in the window)
				}
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					if constexpr( has_inert_v<S> )
						if( ok[u] && S::inert( false, true, xv[u], 0.0f, dt_b ) ) // the event cannot change the synapse
						{
							ok[u] = false;
							touched++;
						}
					if constexpr( has_inert_v<S> )
						if( ok[u] ) load_synapse<S>( sy[u], v.sa, e[u] );
				}
#pragma unroll
				for( int u = 0; u < U; u++ )
				{
					if( !ok[u] ) continue;
					typename S::tuple_t const before = sy[u];
					event( sy[u], e[u], b, dt_b, false, true, xv[u], 0.0f );
					store_synapse<S>( before, sy[u], v.sa, e[u] );
				}
			}
			if( lane == 0 )
			{
				if( end > beg ) words += 2 * std::uint64_t( end - beg ); // (source, offset) entries
				if( p == 0 ) rows++;
			}
		}
	}
	block_add_stats<4>( v, slot0 + blk, { touched, written, words, rows }, { ST_FLUSH_SYN, ST_FLUSH_WRITTEN, ST_FLUSH_SLOTS, ST_FLUSH_ROWS } );
}

// The passes on their own (a synchronization before a state export applies those of the last
// window, which the next window's kernel would otherwise run beside it).
template <typename Model, bool FIXED>
__global__ __launch_bounds__( 256 ) void k_window_passes( dview v )
{
	window_passes<Model, FIXED>( v, blockIdx.x, gridDim.x, v.ntiles );
}

// One workgroup per tile, those with incoming synapses first; then (plastic models) the
// workgroups of the passes of the window before.
// FORM: what the delivery reads (instances of their own: with the delivery from records in all of
// them its registers cost 2 % -- Brunel 1e6 0.88 us per step, 0.90 with it inside). Records: one step.
template <typename Model, bool FIXED, int BS, int FORM = IDS32>
__global__ __launch_bounds__( BS ) void k_window( dview v, std::int32_t W )
{
	std::int32_t const b = blockIdx.x;
	if( b < v.ntiles )
		window_tile<Model, FIXED, BS, FORM>( v, b < v.nact ? xcd_place( b, v.nact ) : b, FORM == RECORDS ? 1 : W );
	else if constexpr( is_plastic_v<Model> )
		window_passes<Model, FIXED>( v, b - v.ntiles, std::int32_t( gridDim.x ) - v.ntiles, v.ntiles );
}

// ---- factored traces as synapse attributes (exports, imports, the per-synapse contract) -----
// out[e] = factored trace attribute `attr` of synapse e: the trace of its source or target where the
// synapse is plastic, init()'s value elsewhere. x, y: the traces now. One wave per row.
template <typename Model>
__global__ __launch_bounds__( 256 ) void k_expand_trace( dview v, float const * x, float const * y, int attr, float * out )
{
	using S = typename Model::synapse;
	std::int64_t const r = uniform64( ( std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x ) >> 6 );
	if( r >= v.N ) return;
	snn_info const info = info_of( v );
	for( std::int64_t e = v.row_ptr[r] + lane_id(); e < v.row_ptr[r + 1]; e += 64 )
	{
		std::int32_t const j = v.col[e];
		out[e] = !S::plastic( std::int32_t( r ), j, info ) ? S::trace_init : attr == S::pre_trace ? x[r] : y[j];
	}
}

// Gathers a factored trace from an imported attribute, in[e]: t[source or target] = the value of some
// plastic synapse of it.
template <typename Model>
__global__ __launch_bounds__( 256 ) void k_gather_trace( dview v, int attr, float const * in, float * t )
{
	using S = typename Model::synapse;
	std::int64_t const r = uniform64( ( std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x ) >> 6 );
	if( r >= v.N || !v.hasp[r] ) return;
	snn_info const info = info_of( v );
	for( std::int64_t e = v.row_ptr[r] + lane_id(); e < v.row_ptr[r + 1]; e += 64 )
	{
		std::int32_t const j = v.col[e];
		if( S::plastic( std::int32_t( r ), j, info ) ) t[attr == S::pre_trace ? r : j] = in[e];
	}
}

// *bad = 1 unless imported attribute `attr` keeps the factored form: a trace the same for all
// plastic synapses of a neuron (t, from k_gather_trace) and init()'s value elsewhere; any other
// attribute unchanged by an event-free step.
template <typename Model>
__global__ __launch_bounds__( 256 ) void k_check_factored( dview v, int attr, void const * in, float const * t, std::int32_t * bad )
{
	using S = typename Model::synapse;
	std::int64_t const r = uniform64( ( std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x ) >> 6 );
	if( r >= v.N ) return;
	snn_info const info = info_of( v );
	for( std::int64_t e = v.row_ptr[r] + lane_id(); e < v.row_ptr[r + 1]; e += 64 )
	{
		std::int32_t const j = v.col[e];
		bool const plastic = S::plastic( std::int32_t( r ), j, info );
		if( is_factored_attr<S>( attr ) )
		{
			float const want = !plastic ? S::trace_init : t[attr == S::pre_trace ? r : std::int64_t( j )];
			if( __builtin_bit_cast( std::uint32_t, want ) != static_cast<std::uint32_t const *>( in )[e] ) *bad = 1;
		}
		else if( plastic )
		{
			typename S::tuple_t sy{};
			util::for_n<S::size>( [&]( auto I ) {
				using T = typename S::template type<I>;
				if constexpr( !is_factored_attr<S>( int( I ) ) ) std::get<I>( sy ) = ld<T>( int( I ) == attr ? in : v.sa[I], e );
			} );
			typename S::tuple_t const before = sy;
			auto bak = make_backend<false>( v, std::uint32_t( e ), std::uint32_t( std::uint64_t( e ) >> 32 ), 0u, util::TAG_SYNAPSE_UPDATE );
			S::on_event( reg_iter<typename S::tuple_t>{ sy, std::uint32_t( e ) }, false, false, v.DT, info, bak );
			if( !same_bits<S>( before, sy ) ) *bad = 1;
		}
	}
}

static inline __global__ __launch_bounds__( 256 ) void k_fill( float * p, std::int64_t n, float x )
{
	std::int64_t const i = std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
	if( i < n ) p[i] = x;
}

// ---- by-target index of the plastic synapses (eager plasticity) ----------------------------
// One workgroup per target tile walks every row's segment inside the tile, in row order (64 rows
// per wave and round), and keeps a counter per target in LDS: COUNT stores them, the fill appends
// (offset in the row, source) to the target's list at its counter. Lists come out ordered by source
// up to the rows in flight at once, which is what the post pass wants (neighbouring entries
// gather neighbouring traces and row starts), without a sort, a second buffer or global atomics;
// a tile's open list lines stay in its XCD's L2. At 1e9 synapses (4.1e8 plastic) a row-major count
// and fill with global atomics and a segmented radix sort took 42 ms.
constexpr int TP_BLOCK = 1024;
template <typename Model, bool COUNT>
__global__ __launch_bounds__( TP_BLOCK ) void k_tp_tile( dview v, std::uint32_t * cnt, tp_entry * ent )
{
	using S = typename Model::synapse;
	constexpr int U = 4;
	struct alignas( 16 ) rec
	{
		std::int64_t off; // first target id in the row store
		std::int32_t row;
		std::int32_t len;
	};
	__shared__ rec segs[TP_BLOCK];
	__shared__ std::uint32_t cur[TILE_MAX];
	__shared__ std::int64_t first[COUNT ? 1 : TILE_MAX];
	int const tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
	std::int32_t const tile = v.tile_ids[xcd_place( blockIdx.x, v.nact )];
	std::int32_t const t0 = tile * v.tile_w;
	std::int32_t const tw = ( v.N - t0 ) < v.tile_w ? ( v.N - t0 ) : v.tile_w;
	for( int x = tid; x < tw; x += TP_BLOCK )
	{
		cur[x] = 0;
		if constexpr( !COUNT ) first[x] = v.tp_ptr[t0 + x];
	}
	__syncthreads();
	snn_info const info = info_of( v );
	int const G = 1 << v.wlanes, g = lane >> v.wlanes, l = lane & ( G - 1 ), ng = 64 >> v.wlanes;
	rec * const mine = segs + wave * 64;
	for( std::int32_t r0 = wave * 64; r0 < v.N; r0 += TP_BLOCK )
	{
		std::int32_t const r = r0 + lane;
		std::int64_t a = 0;
		std::int32_t len = 0;
		if( r < v.N && v.hasp[r] )
		{
			segment const s = segment_of( v, r, tile );
			a = s.at;
			len = s.len;
		}
		mine[lane] = rec{ len > 0 ? a : 0, r, len };
		wave_lds_fence();
		for( int c = 0; c < 64; c += U * ng )
		{
			rec q[U];
			std::int32_t n[U], most = 0;
#pragma unroll
			for( int u = 0; u < U; u++ )
			{
				int const k = c + u * ng + g;
				q[u] = mine[k & 63];
				n[u] = k < 64 ? q[u].len : 0;
				most = n[u] > most ? n[u] : most;
			}
			for( std::int32_t e = l * WIN_VEC; e - l * WIN_VEC < most; e += G * WIN_VEC )
			{
				targets j[U];
#pragma unroll
				for( int u = 0; u < U; u++ ) j[u] = load_targets( v.col + q[u].off + ( e < n[u] ? e : 0 ) );
#pragma unroll
				for( int u = 0; u < U; u++ )
#pragma unroll
					for( int x = 0; x < WIN_VEC; x++ )
					{
						if( e + x >= n[u] || !S::plastic( q[u].row, j[u].id[x], info ) ) continue;
						std::uint32_t const at = atomicAdd( &cur[j[u].id[x] - t0], 1u );
						if constexpr( !COUNT )
							ent[first[j[u].id[x] - t0] + at] = make_tp( q[u].row, q[u].off + e + x );
					}
			}
		}
		wave_lds_fence(); // the next round overwrites the records
	}
	if constexpr( COUNT )
	{
		__syncthreads();
		for( int x = tid; x < tw; x += TP_BLOCK ) cnt[t0 + x] = cur[x];
	}
}

// Appends the spikes of the n steps before the view's step to the net's spike log (one workgroup;
// the counts of a window's steps are final only when its kernel has ended, so the log is written
// by the next one, or by a kernel of its own after the last).
__device__ inline void log_steps( dview const & v, int n )
{
	if( !v.slog ) return;
	std::int64_t const k0 = v.ctl->step - n - v.slog->t0; // first of the steps' places in the log's window
	if( k0 < 0 || k0 + n > v.slog->nsteps ) return;
	std::int32_t const slot0 = window_entry( v );
	auto entry = [&]( std::int32_t k ) { return slot0 + k < 0 ? slot0 + k + v.rsize : slot0 + k; };
	std::uint64_t base = k0 == 0 ? 0ull : v.slog_off[k0 - 1] + v.counts[entry( -n - 1 ) * COUNT_STRIDE];
	std::uint64_t const cap = v.slog->cap;
	for( int q = 0; q < n; q++ )
	{
		std::uint32_t const cnt = v.counts[entry( q - n ) * COUNT_STRIDE];
		std::int32_t const * ids = v.ring + std::int64_t( entry( q - n ) ) * v.N;
		if( threadIdx.x == 0 ) v.slog_off[k0 + q] = base;
		for( std::uint32_t i = threadIdx.x; i < cnt; i += blockDim.x )
			if( base + i < cap ) v.slog_ids[base + i] = ids[i];
		base += cnt;
	}
}

// Batched windows: workgroup b < ntiles runs the tile at place tile_pos[b] of net tile_net[b], the
// next nplast run passes block pass_local[.] of the pass_count[.] blocks of net pass_net[.], the
// rest append net b - ntiles - nplast's spikes of the nlog steps before the window to its log.
template <typename Model, bool FIXED, int BS>
__global__ __launch_bounds__( BS ) void k_batch_window( dview const * views, std::int32_t const * tile_net, std::int32_t const * tile_pos,
                                                        std::int32_t ntiles, std::int32_t W, std::int32_t nlog, std::int32_t const * pass_net,
                                                        std::int32_t const * pass_local, std::int32_t const * pass_count, std::int32_t nplast )
{
	std::int32_t const b = blockIdx.x;
	if( b < ntiles )
	{
		window_tile<Model, FIXED, BS, IDS32_ANY>( views[tile_net[b]], tile_pos[b], W );
		return;
	}
	std::int32_t const p = b - ntiles;
	if constexpr( is_plastic_v<Model> )
		if( p < nplast )
		{
			dview const & v = views[pass_net[p]];
			window_passes<Model, FIXED>( v, pass_local[p], pass_count[p], v.ntiles );
			return;
		}
	log_steps( views[p - nplast], nlog );
}

static __global__ __launch_bounds__( 256 ) void k_batch_log( dview const * views, std::int32_t nlog ) { log_steps( views[blockIdx.x], nlog ); }
} // namespace spice::hipx
