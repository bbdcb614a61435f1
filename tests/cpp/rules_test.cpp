// Host-only checks of spice_amd/csrc/rules.h. Exits non-zero on the first failure.
#include "rules.h"

#include <cstdio>
#include <cstdlib>
#include <set>
#include <type_traits>

using namespace spice::hipx;

#define CHECK( c, ... )                                                           \
	do                                                                            \
	{                                                                             \
		if( !( c ) )                                                              \
		{                                                                         \
			std::printf( "FAIL %s:%d: %s -- ", __FILE__, __LINE__, #c );          \
			std::printf( __VA_ARGS__ );                                           \
			std::printf( "\n" );                                                  \
			std::exit( 1 );                                                       \
		}                                                                         \
	} while( 0 )

// No counter that a window, or the spike log beside it, reads is one that the window clears or adds
// to: all delays, longest windows, and lengths of the window and of the one before it.
static void ring()
{
	for( int delay = 1; delay <= 300; delay++ )
		for( int longest = 1; longest <= WINDOW_MAX; longest++ )
		{
			int const cap = delay >= 2 ? std::max( 1, window_steps( std::min( delay, longest ) ) ) : 1;
			int const R = ring_entries( delay, cap );
			auto entry = [&]( int k ) { // as in the kernels: one wrap either way
				CHECK( -R <= k && k < R, "delay %d cap %d entry %d", delay, cap, k );
				return ( k + R ) % R;
			};
			for( int W = 1; W <= cap; W++ )
				for( int n = 0; n <= cap; n++ )
				{
					std::set<int> read, cleared, added;
					for( int q = 0; q < W; q++ ) read.insert( entry( q - delay ) ); // arrivals
					if( n > 0 )
						for( int q = -n - 1; q < 0; q++ ) read.insert( entry( q ) ); // spike log
					for( int q = 0; q < W; q++ ) added.insert( entry( q ) );
					for( int q = 0; q < cap; q++ ) cleared.insert( entry( W + q ) );
					for( int e : read ) CHECK( !cleared.count( e ) && !added.count( e ), "delay %d cap %d W %d n %d entry %d", delay, cap, W, n, e );
					for( int e : added ) CHECK( !cleared.count( e ), "delay %d cap %d W %d entry %d", delay, cap, W, e );
				}
		}
}

// A staged segment gives back what it was made of, at any length that a row may have.
static void staged_segments()
{
	for( std::int64_t at : { std::int64_t( 0 ), std::int64_t( 7 ), std::int64_t( 65536 ), ( std::int64_t( 1 ) << 40 ) - 1 } )
		for( std::int32_t len : { 0, 1, 65528, 65535, 65536, 65537, 131072, 1 << 24, INT32_MAX - 7 } )
			for( int step = 0; step < WINDOW_MAX; step++ )
			{
				for( std::int32_t src : { 0, 12345, ( 1 << 24 ) - 1 } )
				{
					auto back = [&]( auto plastic ) {
						constexpr bool P = decltype( plastic )::value;
						win_seg s = win_seg::of<P>( at, len, src, step );
						CHECK( s.take_step<P>() == step && s.at == ( len > 0 ? at : 0 ) && s.len == len && s.src == src, "at %lld len %d step %d src %d", (long long)( at ), len, step, src );
					};
					back( std::true_type{} );
					back( std::false_type{} );
				}
			}
	static_assert( sizeof( win_seg ) == 16, "" );
}

// Tiles: however few neurons have inputs, at most two per CU, or four with plasticity (or as wide as its
// kernel takes), and a segment table of at most 1 GB, or that of tiles for two per CU; where half of the neurons have
// inputs or more, one per CU of those (windows of several steps: of all, or two).
static void tiles()
{
	int const cus = 256;
	for( double x = 1; x < 3e7; x = x * 1.07 + 1 )
		for( double share : { 0.0, 1e-5, 1e-3, 0.01, 0.1, 0.3, 0.4999, 0.5, 0.8, 1.0 } )
			for( int kind = 0; kind < 4; kind++ )
			{
				bool const plastic = kind & 1, ahead = kind & 2;
				std::int64_t const n = std::int64_t( x ), targets = share == 0.5 ? n - n / 2 : std::int64_t( share * double( n ) );
				int const w = window_tile_w( n, targets, plastic, ahead, cus ), most = plastic || ahead ? TILE_MAX : 4 * 1024;
				std::int64_t const tiles = ( n + w - 1 ) / w;
				CHECK( w >= 64 && w <= most && w % 64 == 0, "n %lld w %d", (long long)n, w );
				CHECK( tiles <= ( plastic ? 4 : 2 ) * cus || w == most, "n %lld targets %lld kind %d w %d", (long long)n, (long long)targets, kind, w );
				std::int64_t const two = std::min<std::int64_t>( tile_width( n, 2 * cus ), most );
				if( share < 0.5 ) CHECK( 8 * seg_entries( n, tiles ) <= std::max( TABLE_SMALL, 8 * seg_entries( n, ( n + two - 1 ) / two ) ), "n %lld targets %lld kind %d w %d", (long long)n, (long long)targets, kind, w );
				else
				{
					std::int64_t const of = ahead && !plastic ? n : targets, one = tile_width( of, cus );
					CHECK( w == std::clamp<std::int64_t>( ahead && one > most ? tile_width( of, 2 * cus ) : one, 64, most ), "n %lld targets %lld kind %d w %d", (long long)n, (long long)targets, kind, w );
				}
			}
}

// Optional memory leaves what the network still needs, however much of it was taken before, and a
// served net's table never takes more than its estimate, also once its tiles are wider.
static void memory()
{
	std::uint64_t const G = std::uint64_t( 1 ) << 30;
	for( std::uint64_t free : { 0 * G, 1 * G, 7 * G, 50 * G, 288 * G } )
		for( std::uint64_t reserve : { 0 * G, 1 * G, 6 * G, 49 * G, 200 * G } )
		{
			std::uint64_t left = free;
			for( int k = 0; k < 5; k++ )
				for( std::uint64_t bytes = OPTIONAL_SMALL + 1; bytes < 2 * left; bytes = bytes * 3 / 2 )
					if( optional_fits( bytes, left, reserve ) ) left -= bytes;
			CHECK( left == free || left >= reserve, "free %llu reserve %llu", (unsigned long long)free, (unsigned long long)reserve );
		}
	for( std::int64_t n : { 100, 40000, 900000, 8000000 } )
		for( std::int64_t tiles = 1; tiles < n / 64 + 2; tiles = tiles * 5 / 4 + 1 )
			for( std::int64_t fewer = tiles; fewer > 0; fewer = fewer * 9 / 10 )
			{
				std::uint64_t const bytes = 8 * seg_entries( n, fewer ), taken = bytes <= TABLE_BATCHED ? bytes : 4 * std::uint64_t( n ) * std::uint64_t( fewer + 1 );
				CHECK( taken <= batched_table_bytes( n, tiles ), "n %lld tiles %lld now %lld", (long long)n, (long long)tiles, (long long)fewer );
			}
}

int main()
{
	memory();
	tiles();
	ring();
	staged_segments();
	std::printf( "ALL OK\n" );
}
