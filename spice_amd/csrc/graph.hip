// Random-graph generation on gfx950 (subsystem a).
//
// Semantics: include/spice/util/graphgen.h (the reference's generator,
// spice/util/adj_list.cpp:49-91, re-keyed on Philox). Work split:
//   k_degrees : one thread per source row, sums the clipped per-connection degrees;
//   scan      : exclusive scan of row degrees -> int64 row offsets (CSR, > 2^32 edges OK);
//   k_targets : one or more wave64 per source row. For each covering connection every lane draws
//               4 consecutive exponentials per Philox block and keeps them; wave and row prefix
//               sums (exact, whole numbers) give the total and then the positions, 4 targets
//               stored per lane (a wave stores 1 KB contiguous per round).
// Everything is integer except the final double-precision scaling, so the result equals the
// sequential host build bit for bit.
#include "graph.h"

#include <algorithm>
#include <type_traits>

namespace spice::hipx
{
using util::gen::conn;

static __global__ __launch_bounds__( 256 ) void k_degrees(
    conn const * conns, int nconns, std::int64_t n, std::int64_t width, std::uint64_t seed, std::int32_t * deg )
{
	std::int64_t const r = std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
	if( r >= n ) return;
	std::int64_t total = 0;
	for( int c = 0; c < nconns; c++ )
	{
		conn const cn = conns[c];
		if( r < cn.src_first || r >= cn.src_last ) continue;
		std::int64_t d = util::gen::sample_degree( seed, std::uint32_t( r ), std::uint32_t( c ), cn );
		if( d > width - total ) d = width - total;
		total += d;
	}
	deg[r] = std::int32_t( total );
}

// ---- exponential draws and positions without divisions ----------------------------------------
// util::gen::exp_fix_one and ::position are whole numbers, floor() of a double-precision value. Both
// are formed here from a cheaper value that is within 2^-20 of it, and the original is evaluated
// only where that value lies within MARGIN of a whole number (one draw in 2^17), so the results are
// the same: exp_fix_one agrees for all 2^32 arguments.
constexpr double MARGIN = 1.0 / 262144.0;

// -ln by table: c ~ 1 / m for the 128 stretches of m in [1, 2), rounded to float (so that m * c - 1 is
// one fma), and 2^24 ln c.
constexpr int LOG_BITS = 7;
struct log_entry
{
	double c, lnc;
};
__device__ inline void fill_log_table( log_entry * t )
{
	for( int i = threadIdx.x; i < 1 << LOG_BITS; i += blockDim.x )
	{
		double const c = double( float( 1.0 / ( 1.0 + ( double( i ) + 0.5 ) / double( 1 << LOG_BITS ) ) ) );
		t[i] = log_entry{ c, 16777216.0 * util::det::log( c ) };
	}
}

// 2^24 (-ln( (x + 1) 2^-32 )): with (x + 1) = 2^e m and r = m c - 1, |r| < 2^-8,
// ln( 1 + r ) = r - r^2/2 + r^3/3 - r^4/4 + r^5/5 to 2^-50.
__device__ inline double exp_fast( std::uint32_t x, log_entry const * t )
{
	std::uint64_t const b = util::det::bits( double( x ) + 1.0 );
	std::uint32_t const hi = std::uint32_t( b >> 32 );
	log_entry const le = t[( hi >> ( 20 - LOG_BITS ) ) & ( ( 1 << LOG_BITS ) - 1 )];
	double const m = util::det::from_bits( ( std::uint64_t( ( hi & 0x000fffffu ) | 0x3ff00000u ) << 32 ) | std::uint32_t( b ) );
	double const r = __builtin_fma( m, le.c, -1.0 );
	double p = __builtin_fma( r, 0.2, -0.25 );
	p = __builtin_fma( p, r, 1.0 / 3.0 );
	p = __builtin_fma( p, r, -0.5 );
	p = __builtin_fma( p, r, 1.0 );
	constexpr double LN2 = 0.69314718055994530942 * 16777216.0;
	return __builtin_fma( -16777216.0 * r, p, __builtin_fma( double( 32 + 1023 - int( hi >> 20 ) ), LN2, le.lnc ) );
}

// Whether floor( y ) (y to 2^-20) may not be the original's.
__device__ inline bool near_whole( double y ) { return !( __builtin_fabs( __builtin_amdgcn_fract( y ) - 0.5 ) < 0.5 - MARGIN ); }

// Four draws of a Philox block, as util::gen::exp_fix4.
__device__ inline void exp_fix4_fast( util::philox_u4 const & x, log_entry const * t, std::uint32_t ( &f )[4] )
{
	std::uint32_t const in[4] = { x.x, x.y, x.z, x.w };
	bool unsure = false;
#pragma unroll
	for( int q = 0; q < 4; q++ )
	{
		double const y = exp_fast( in[q], t );
		f[q] = std::uint32_t( y > 0.0 ? y : 0.0 );
		unsure = unsure || near_whole( y );
	}
	if( unsure )
	{
#pragma unroll 1
		for( int q = 0; q < 4; q++ )
		{
			std::uint32_t const v = util::gen::exp_fix_one( q == 0 ? in[0] : q == 1 ? in[1] : q == 2 ? in[2] : in[3] );
			f[0] = q == 0 ? v : f[0];
			f[1] = q == 1 ? v : f[1];
			f[2] = q == 2 ? v : f[2];
			f[3] = q == 3 ? v : f[3];
		}
	}
}

// util::gen::position of four successive prefix sums t (whole numbers below 2^53) from draw k on;
// scale = R / ttotal.
__device__ inline void positions4( double const ( &t )[4], double scale, double ttotal, std::int32_t R, std::int32_t k, std::int32_t ( &p )[4] )
{
	bool unsure = false;
#pragma unroll
	for( int q = 0; q < 4; q++ )
	{
		double const y = t[q] * scale;
		p[q] = std::int32_t( y ) + k + q;
		unsure = unsure || near_whole( y );
	}
	if( unsure )
	{
#pragma unroll 1
		for( int q = 0; q < 4; q++ )
		{
			std::int32_t const v = util::gen::position( std::uint64_t( q == 0 ? t[0] : q == 1 ? t[1] : q == 2 ? t[2] : t[3] ), std::uint64_t( ttotal ), R, k + q );
			p[0] = q == 0 ? v : p[0];
			p[1] = q == 1 ? v : p[1];
			p[2] = q == 2 ? v : p[2];
			p[3] = q == 3 ? v : p[3];
		}
	}
}

// Inclusive prefix sum of doubles over a wave (whole numbers, exact): row shifts, then row
// broadcasts, in the vector ALU.
__device__ inline double wave_scan_f64( double x )
{
	auto step = [&]( auto ctrl, auto rows ) {
		std::uint64_t const b = util::det::bits( x );
		std::uint32_t const lo = std::uint32_t( __builtin_amdgcn_update_dpp( 0, int( std::uint32_t( b ) ), decltype( ctrl )::value, decltype( rows )::value, 0xf, false ) );
		std::uint32_t const hi = std::uint32_t( __builtin_amdgcn_update_dpp( 0, int( std::uint32_t( b >> 32 ) ), decltype( ctrl )::value, decltype( rows )::value, 0xf, false ) );
		x += util::det::from_bits( ( std::uint64_t( hi ) << 32 ) | lo );
	};
	using std::integral_constant;
	step( integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{} ); // row_shr 1, 2, 4, 8
	step( integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{} );
	step( integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{} );
	step( integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{} );
	step( integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{} ); // row_bcast 15, 31
	step( integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{} );
	return x;
}
__device__ inline double lane63( double x )
{
	std::uint64_t const b = util::det::bits( x );
	return util::det::from_bits( ( std::uint64_t( std::uint32_t( __builtin_amdgcn_readlane( int( std::uint32_t( b >> 32 ) ), 63 ) ) ) << 32 ) |
	                             std::uint32_t( __builtin_amdgcn_readlane( int( std::uint32_t( b ) ), 63 ) ) );
}

// A connection too long for the registers: two passes over the draws by one wave, 4 consecutive draws
// per lane (pass 1 the total, pass 2 the prefix sums and positions).
static __device__ void long_connection( conn const & cn, int c, std::int64_t r, std::int64_t d, std::int32_t R, std::uint64_t seed, std::int32_t * col )
{
	int const lane = lane_id();
	std::int64_t const nblk = ( d + 1 + 3 ) / 4;
	std::uint64_t part = 0;
	for( std::int64_t b = lane; b < nblk; b += 64 )
	{
		std::uint32_t f[4];
		util::gen::exp_fix4( seed, std::uint32_t( r ), std::uint32_t( c ), std::uint32_t( b ), f );
#pragma unroll
		for( int q = 0; q < 4; q++ )
			if( 4 * b + q <= d ) part += f[q];
	}
	std::uint64_t const ttotal = wave_sum( part );
	std::uint64_t carry = 0;
	for( std::int64_t b0 = 0; b0 < nblk; b0 += 64 )
	{
		std::int64_t const b = b0 + lane;
		std::uint32_t f[4] = { 0, 0, 0, 0 };
		if( b < nblk ) util::gen::exp_fix4( seed, std::uint32_t( r ), std::uint32_t( c ), std::uint32_t( b ), f );
		std::uint64_t s[4];
		s[0] = f[0];
		s[1] = s[0] + f[1];
		s[2] = s[1] + f[2];
		s[3] = s[2] + f[3];
		std::uint64_t const incl = wave_inclusive_scan( s[3] );
		std::uint64_t const excl = carry + incl - s[3];
#pragma unroll
		for( int q = 0; q < 4; q++ )
		{
			std::int64_t const k = 4 * b + q;
			if( k < d ) col[k] = cn.dst_first + util::gen::position( excl + s[q], ttotal, R, std::int32_t( k ) );
		}
		carry += shfl_u64( incl, 63 );
	}
}

// Targets of rows, NW waves per row. A connection's draws are split into one stretch per wave; up to
// 2,048 of them per wave (8 KB) are drawn once and kept in LDS for the total and then the positions, longer
// connections are drawn twice by the row's first wave. Bound by the vector ALU (Philox, the
// logarithm; busy 92 to 96 % of the time): 1e9 targets 2.3 ms, and 4.6 with every draw made twice and a division each in its
// logarithm and its position.
constexpr int LANE_BLOCKS = 8; // Philox blocks (of 4 draws) per lane
template <int NW>
static __global__ __launch_bounds__( NW == 16 ? 1024 : 256 ) void k_targets(
    conn const * conns, int nconns, std::int64_t n, std::int64_t width, std::uint64_t seed, std::int64_t const * row_ptr, std::int32_t * col )
{
	constexpr int bs = NW == 16 ? 1024 : 256;
	struct alignas( 16 ) block4
	{
		std::uint32_t f[4];
	};
	__shared__ log_entry table[1 << LOG_BITS];
	__shared__ block4 draws[bs * LANE_BLOCKS];
	__shared__ double tot[2][NW];
	fill_log_table( table );
	__syncthreads();
	int const lane = lane_id(), wave = threadIdx.x >> 6;
	int const w = NW == 1 ? 0 : wave; // wave of the row
	block4 * const mine = draws + wave * ( 64 * LANE_BLOCKS ) + lane;
	int turn = 0;
	constexpr std::int64_t per_block = bs / ( 64 * NW );
	for( std::int64_t r = uniform64( blockIdx.x * per_block + ( NW == 1 ? wave : 0 ) ); r < n; r += gridDim.x * per_block )
	{
		std::int64_t off = row_ptr[r];
		std::int64_t total = 0;
		for( int c0 = 0; c0 < nconns; c0 += 64 )
		{
			// lane c: the degree of connection c0 + c
			std::int32_t dg = 0;
			if( c0 + lane < nconns )
			{
				conn const cn = conns[c0 + lane];
				if( r >= cn.src_first && r < cn.src_last ) dg = util::gen::sample_degree( seed, std::uint32_t( r ), std::uint32_t( c0 + lane ), cn );
			}
			for( std::uint64_t todo = ballot( dg > 0 ); todo; todo &= todo - 1 )
			{
				int const l = __builtin_ctzll( todo ), c = c0 + l;
				std::int64_t d = __builtin_amdgcn_readlane( dg, l );
				if( d > width - total ) d = width - total;
				total += d;
				if( d == 0 ) continue;
				std::int32_t const first = conns[c].dst_first;
				std::int32_t const R = ( conns[c].dst_last - first ) - std::int32_t( d );
				std::int64_t const nblk = ( d + 1 + 3 ) / 4;
				if( nblk <= 64 * LANE_BLOCKS * NW )
				{
					// this wave's blocks
					std::int32_t const each = ( std::int32_t( nblk ) + NW - 1 ) / NW;
					std::int32_t const b0 = w * each, b1 = b0 + each < nblk ? b0 + each : std::int32_t( nblk );
					double part = 0.0;
#pragma unroll 1
					for( int k = 0; b0 + 64 * k < b1; k++ )
					{
						std::int32_t const b = b0 + 64 * k + lane;
						block4 x{ { 0, 0, 0, 0 } };
						if( b < b1 )
						{
							exp_fix4_fast( util::philox( seed, { std::uint32_t( b ), std::uint32_t( r ), std::uint32_t( c ), util::TAG_GRAPH_POS } ), table, x.f );
#pragma unroll
							for( int q = 1; q < 4; q++ )
								if( 4 * b + q > d ) x.f[q] = 0;
						}
						mine[64 * k] = x;
						part += double( x.f[0] + x.f[1] + x.f[2] + x.f[3] ); // (a draw is below 22.2 x 2^24)
					}
					// what the waves before this one drew, and the total T_d
					double carry = 0.0, ttotal = lane63( wave_scan_f64( part ) );
					if constexpr( NW > 1 )
					{
						if( lane == 0 ) tot[turn][w] = ttotal;
						__syncthreads();
						ttotal = 0.0;
						for( int x = 0; x < NW; x++ )
						{
							double const y = tot[turn][x];
							carry += x < w ? y : 0.0;
							ttotal += y;
						}
						turn ^= 1; // (the other half is written before any wave is past the next barrier)
					}
					double const scale = double( R ) / ttotal; // (ttotal 0: not a number, so never sure)
#pragma unroll 1
					for( int k = 0; b0 + 64 * k < b1; k++ )
					{
						std::int32_t const b = b0 + 64 * k + lane;
						block4 const x = mine[64 * k];
						std::uint32_t const s1 = x.f[0] + x.f[1], s2 = s1 + x.f[2], s3 = s2 + x.f[3];
						double const incl = wave_scan_f64( double( s3 ) );
						double const base = carry + ( incl - double( s3 ) );
						carry += lane63( incl );
						if( b >= b1 || 4 * b >= d ) continue;
						double const ts[4] = { base + double( x.f[0] ), base + double( s1 ), base + double( s2 ), base + double( s3 ) };
						std::int32_t p[4];
						positions4( ts, scale, ttotal, R, 4 * b, p );
#pragma unroll
						for( int q = 0; q < 4; q++ ) p[q] += first;
						std::int32_t * const o = col + off + 4 * b;
						if( 4 * b + 3 < d )
							__builtin_memcpy( o, p, sizeof( p ) );
						else
							for( int q = 0; q < 3; q++ )
								if( 4 * b + q < d ) o[q] = p[q];
					}
				}
				else if( w == 0 )
					long_connection( conns[c], c, r, d, R, seed, col + off );
				off += d;
			}
		}
	}
}

// k_targets for every row of a graph: as many waves per row as hold the longest likely connection
// (six standard deviations above the mean).
static void launch_targets( std::vector<conn> const & conns, conn const * dconns, std::int64_t n, std::int64_t width, std::uint64_t seed,
                            std::int64_t const * row_ptr, std::int32_t * col, hipStream_t s )
{
	double longest = 0.0;
	for( auto const & c : conns )
	{
		double const d = c.mean + 6.0 * c.sd;
		longest = d > longest ? d : longest;
	}
	constexpr std::int64_t blocks = 256 * 8 * 4; // (rows beyond are taken in turn)
	auto go = [&]( auto nw ) {
		constexpr int NW = decltype( nw )::value;
		constexpr int bs = NW == 16 ? 1024 : 256;
		std::int64_t const per = bs / ( 64 * NW );
		unsigned const grid = unsigned( std::min<std::int64_t>( ( n + per - 1 ) / per, blocks * 256 / bs ) );
		SPICE_LAUNCH( k_targets<NW><<<dim3( grid ), bs, 0, s>>>( dconns, int( conns.size() ), n, width, seed, row_ptr, col ) );
	};
	if( longest < 256.0 * LANE_BLOCKS - 4.0 ) // (a wave holds 256 x LANE_BLOCKS draws, the last one of a connection sets the scale)
		go( std::integral_constant<int, 1>{} );
	else if( longest < 1024.0 * LANE_BLOCKS - 4.0 )
		go( std::integral_constant<int, 4>{} );
	else
		go( std::integral_constant<int, 16>{} );
}

// ---- exclusive scan int32 -> int64 (3 phases) --------------------------------------------
constexpr int SCAN_BLOCK = 256, SCAN_ITEMS = 4, SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

// Block-level exclusive scan of a tile; writes tile-local prefixes and the tile total. Each
// thread reads its items before writing the same positions, so in == out is allowed.
template <typename In>
static __global__ __launch_bounds__( SCAN_BLOCK ) void k_scan_tiles( In const * in, std::int64_t * out, std::int64_t n, std::int64_t * tile_sums )
{
	__shared__ std::uint64_t wsum[SCAN_BLOCK / 64];
	std::int64_t const base = std::int64_t( blockIdx.x ) * SCAN_TILE + std::int64_t( threadIdx.x ) * SCAN_ITEMS;
	std::uint64_t v[SCAN_ITEMS];
	std::uint64_t t = 0;
#pragma unroll
	for( int q = 0; q < SCAN_ITEMS; q++ )
	{
		v[q] = ( base + q < n ) ? std::uint64_t( std::int64_t( in[base + q] ) ) : 0;
		t += v[q];
	}
	std::uint64_t const incl = wave_inclusive_scan( t );
	int const w = threadIdx.x >> 6;
	if( lane_id() == 63 ) wsum[w] = incl;
	__syncthreads();
	std::uint64_t wbase = 0;
	for( int i = 0; i < w; i++ ) wbase += wsum[i];
	std::uint64_t run = wbase + incl - t;
#pragma unroll
	for( int q = 0; q < SCAN_ITEMS; q++ )
	{
		if( base + q < n ) out[base + q] = std::int64_t( run );
		run += v[q];
	}
	if( threadIdx.x == SCAN_BLOCK - 1 ) tile_sums[blockIdx.x] = std::int64_t( run );
}

// Single block: exclusive scan of the tile totals (in place), total into out_total.
static __global__ __launch_bounds__( 1024 ) void k_scan_tile_sums( std::int64_t * tile_sums, std::int64_t ntiles, std::int64_t * out_total )
{
	__shared__ std::uint64_t wsum[16];
	__shared__ std::uint64_t carry_s;
	if( threadIdx.x == 0 ) carry_s = 0;
	__syncthreads();
	for( std::int64_t b0 = 0; b0 < ntiles; b0 += 1024 )
	{
		std::int64_t const i = b0 + threadIdx.x;
		std::uint64_t const x = i < ntiles ? std::uint64_t( tile_sums[i] ) : 0;
		std::uint64_t const incl = wave_inclusive_scan( x );
		int const w = threadIdx.x >> 6;
		if( lane_id() == 63 ) wsum[w] = incl;
		__syncthreads();
		std::uint64_t wbase = carry_s;
		for( int k = 0; k < w; k++ ) wbase += wsum[k];
		if( i < ntiles ) tile_sums[i] = std::int64_t( wbase + incl - x );
		__syncthreads();
		if( threadIdx.x == 1023 ) carry_s = wbase + incl;
		__syncthreads();
	}
	if( threadIdx.x == 0 ) *out_total = std::int64_t( carry_s );
}

static __global__ __launch_bounds__( 256 ) void k_scan_add( std::int64_t * out, std::int64_t n, std::int64_t const * tile_sums )
{
	std::int64_t const i = std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
	if( i < n ) out[i] += tile_sums[i / SCAN_TILE];
}

// Exclusive scan with the per-tile sums in `sums` (ceil(n / SCAN_TILE) entries, at least 1);
// out[n] = total. Enqueued on s.
template <typename In>
static void exclusive_scan_to_i64( In const * in, std::int64_t * out, std::int64_t n, std::int64_t * sums, hipStream_t s )
{
	std::int64_t const ntiles = ( n + SCAN_TILE - 1 ) / SCAN_TILE;
	if( n > 0 )
	{
		SPICE_LAUNCH( k_scan_tiles<In><<<dim3( unsigned( ntiles ) ), SCAN_BLOCK, 0, s>>>( in, out, n, sums ) );
	}
	SPICE_LAUNCH( k_scan_tile_sums<<<1, 1024, 0, s>>>( sums, ntiles, out + n ) );
	if( n > 0 )
	{
		SPICE_LAUNCH( k_scan_add<<<dim3( unsigned( ( n + 255 ) / 256 ) ), 256, 0, s>>>( out, n, sums ) );
	}
}

void exclusive_scan_i32_to_i64( std::int32_t const * in, std::int64_t * out, std::int64_t n, hipStream_t s )
{
	std::int64_t const ntiles = ( n + SCAN_TILE - 1 ) / SCAN_TILE;
	dbuf<std::int64_t> sums( ntiles > 0 ? ntiles : 1 );
	exclusive_scan_to_i64( in, out, n, sums.data(), s );
	SPICE_HIP( hipStreamSynchronize( s ) ); // `sums` is released on return
}

csr_dev generate_csr( std::vector<conn> const & conns, std::int64_t n, std::int64_t width, std::uint64_t seed, hipStream_t s )
{
	csr_dev g;
	g.n = n;
	g.width = width;
	g.targets = target_range( conns );
	g.row_ptr.resize( n + 1 );
	dbuf<conn> dconns( conns.size() > 0 ? conns.size() : 1 );
	if( !conns.empty() )
		SPICE_HIP( hipMemcpyAsync( dconns.data(), conns.data(), conns.size() * sizeof( conn ), hipMemcpyHostToDevice, s ) );
	dbuf<std::int32_t> deg( n > 0 ? n : 1 );
	if( n > 0 )
		SPICE_LAUNCH( k_degrees<<<dim3( unsigned( ( n + 255 ) / 256 ) ), 256, 0, s>>>(
		    dconns.data(), int( conns.size() ), n, width, seed, deg.data() ) );
	exclusive_scan_i32_to_i64( deg.data(), g.row_ptr.data(), n, s );
	SPICE_HIP( hipMemcpy( &g.nnz, g.row_ptr.data() + n, sizeof( std::int64_t ), hipMemcpyDeviceToHost ) );
	g.col.resize( g.nnz + COL_PAD );
	if( n > 0 && g.nnz > 0 )
	{
		launch_targets( conns, dconns.data(), n, width, seed, g.row_ptr.data(), g.col.data(), s );
	}
	SPICE_HIP( hipStreamSynchronize( s ) );
	return g;
}

// ---- graph into caller-owned device memory --------------------------------------------------
// Row lengths go straight into row_ptr[0 .. n) (int64) and are scanned in place, so the only
// scratch is the connection table and the scan's per-tile sums.
static __global__ __launch_bounds__( 256 ) void k_degrees_i64(
    conn const * conns, int nconns, std::int64_t n, std::int64_t width, std::uint64_t seed, std::int64_t * len )
{
	std::int64_t const r = std::int64_t( blockIdx.x ) * blockDim.x + threadIdx.x;
	if( r >= n ) return;
	std::int64_t total = 0;
	for( int c = 0; c < nconns; c++ )
	{
		conn const cn = conns[c];
		if( r < cn.src_first || r >= cn.src_last ) continue;
		std::int64_t d = util::gen::sample_degree( seed, std::uint32_t( r ), std::uint32_t( c ), cn );
		if( d > width - total ) d = width - total;
		total += d;
	}
	len[r] = total;
}

std::int64_t graph_scratch_tiles( std::int64_t n ) { return n > 0 ? ( n + SCAN_TILE - 1 ) / SCAN_TILE : 1; }

std::int64_t generate_into( std::vector<conn> const & conns, std::int64_t n, std::int64_t width, std::uint64_t seed, std::int64_t * row_ptr,
                            std::int32_t * col, std::uint64_t col_cap, conn * conn_scratch, std::int64_t * tile_scratch, hipStream_t s )
{
	// conn_scratch and tile_scratch need no clearing: the copy below and the scan write every
	// entry they later read
	if( !conns.empty() )
		SPICE_HIP( hipMemcpyAsync( conn_scratch, conns.data(), conns.size() * sizeof( conn ), hipMemcpyHostToDevice, s ) );
	if( n > 0 )
		SPICE_LAUNCH( k_degrees_i64<<<dim3( unsigned( ( n + 255 ) / 256 ) ), 256, 0, s>>>( conn_scratch, int( conns.size() ), n, width, seed, row_ptr ) );
	exclusive_scan_to_i64( row_ptr, row_ptr, n, tile_scratch, s );
	std::int64_t nnz = 0;
	SPICE_HIP( hipMemcpyAsync( &nnz, row_ptr + n, sizeof( nnz ), hipMemcpyDeviceToHost, s ) );
	SPICE_HIP( hipStreamSynchronize( s ) ); // conns (host) copied, nnz read
	if( col && std::uint64_t( nnz ) <= col_cap && n > 0 && nnz > 0 )
	{
		launch_targets( conns, conn_scratch, n, width, seed, row_ptr, col, s );
		SPICE_HIP( hipStreamSynchronize( s ) );
	}
	return nnz;
}

csr_dev upload_csr( std::int64_t const * row_ptr, std::int32_t const * col, std::int64_t n, std::int64_t width, hipStream_t s )
{
	csr_dev g;
	g.n = n;
	g.width = width;
	g.nnz = row_ptr[n];
	std::int64_t first = n, last = -1; // (rows are sorted by target)
	for( std::int64_t r = 0; r < n; r++ )
		if( row_ptr[r + 1] > row_ptr[r] )
		{
			first = col[row_ptr[r]] < first ? col[row_ptr[r]] : first;
			last = col[row_ptr[r + 1] - 1] > last ? col[row_ptr[r + 1] - 1] : last;
		}
	g.targets = last >= first ? last - first + 1 : 0;
	g.row_ptr.resize( n + 1 );
	g.col.resize( g.nnz + COL_PAD );
	SPICE_HIP( hipMemcpyAsync( g.row_ptr.data(), row_ptr, ( n + 1 ) * sizeof( std::int64_t ), hipMemcpyHostToDevice, s ) );
	if( g.nnz > 0 )
		SPICE_HIP( hipMemcpyAsync( g.col.data(), col, g.nnz * sizeof( std::int32_t ), hipMemcpyHostToDevice, s ) );
	SPICE_HIP( hipStreamSynchronize( s ) );
	return g;
}
} // namespace spice::hipx
