#pragma once
// Batched stepping of many independent networks of one model (parameter sweeps, served
// jobs). Every net keeps its own buffers, clock and statistics (it is an ordinary hip_net);
// the batch adds device tables that map the workgroups of ONE launch per window to (net, tile), for
// plastic models (net, workgroup of the passes), and spike logs -- or, for nets on two-kernel
// steps, of one launch per step phase; single steps replay captured HIP graphs of those launches
// (graphs.h). Per-net results are
// identical to stepping the nets one by one: the kernels run the same per-net bodies and all
// randomness is keyed on (net seed, neuron, step). Nets may sit at different steps (served
// jobs join a running mix): each net's clock slot is chosen from its own step parity.
#include "net.h"

#include <memory>
#include <vector>

namespace spice::hipx
{
struct batch_iface
{
	virtual ~batch_iface() = default;
	virtual void run( std::int64_t n ) = 0;
	virtual void synchronize() = 0;
	virtual int size() const = 0;
	virtual net_iface * net( int i ) = 0;
	// opens the spike-log window of every net (with a log) over the next nsteps steps
	virtual void begin_spike_log( std::int64_t nsteps ) = 0;
};

template <typename Model>
class hip_batch final : public batch_iface
{
	static constexpr bool plastic = is_plastic_v<Model>;
	static constexpr bool windowed = windowed_v<Model>; // steps run as windows
	// delivery workgroup size: most tiles of a sweep belong to small nets and carry few events,
	// so more, smaller workgroups shorten the launch's critical path
	static constexpr int recv_block = SPICE_BATCH_RECV_BLOCK;

public:
	// `nets` must outlive the batch unless they are also handed over in `owned`. The batch
	// destroys `stream` at the end if `own_stream`.
	hip_batch( std::vector<hip_net<Model> *> nets, std::vector<std::unique_ptr<hip_net<Model>>> && owned, hipStream_t stream, bool own_stream )
	    : _nets( std::move( nets ) )
	    , _owned( std::move( owned ) )
	    , _s( stream )
	    , _own_stream( own_stream )
	{
		if( _nets.empty() ) throw std::invalid_argument( "empty batch" );
		_fixed = _nets[0]->fixed();
		for( auto * n : _nets )
			if( n->fixed() != _fixed ) throw std::invalid_argument( "all nets of a batch use the same accumulation mode" );
		for( auto * n : _nets )
		{
			launch_cfg c = n->get_launch();
			int const tw = batch_tile_w( n->num_neurons(), c.tile_w, std::int64_t( _nets.size() ), n->params().delay );
			if( tw != c.tile_w )
			{
				c.tile_w = tw;
				n->set_launch( c );
			}
		}
		build();
	}

	// Device tables of the nets' workgroups and views. Windows, unless a net's plasticity went back
	// to the per-synapse contract (hip_net::make_lazy): then every net's does, and steps are two
	// kernels.
	void build()
	{
		_built = false; // (until all of it is done: an allocation may fail on the way)
		_windows = windowed;
		if constexpr( factored_v<Model> )
		{
			for( auto * n : _nets ) _windows = _windows && !n->lazy();
			if( !_windows )
				for( auto * n : _nets ) n->make_lazy();
		}
		std::vector<std::int32_t> tn, tl, bn, bl, fn, fl, fc;
		std::vector<dview> vs[CLOCK_SLOTS];
		for( std::size_t k = 0; k < _nets.size(); k++ )
		{
			hip_net<Model> & n = *_nets[k];
			// windows: one workgroup per tile; two-kernel steps: (tile, part) work items of the tiles
			// with incoming synapses
			for( int t = 0; t < ( _windows ? n.num_all_tiles() : n.num_tiles() * n.num_receive_parts() ); t++ )
			{
				tn.push_back( std::int32_t( k ) );
				tl.push_back( t );
			}
			if( !_windows )
				for( int b = 0; b < n.num_update_blocks(); b++ )
				{
					bn.push_back( std::int32_t( k ) );
					bl.push_back( b );
				}
			if constexpr( plastic )
			{
				int const nf = n.num_batch_flush_blocks();
				for( int b = 0; b < nf; b++ )
				{
					fn.push_back( std::int32_t( k ) );
					fl.push_back( b );
					fc.push_back( nf );
				}
			}
			// batch step t runs net step host_step + (t - _step): the clock slot of that
			for( int p = 0; p < CLOCK_SLOTS; p++ ) vs[( _step + p ) & ( CLOCK_SLOTS - 1 )].push_back( n.view( int( ( n.host_step() + p ) & ( CLOCK_SLOTS - 1 ) ) ) );
		}
		_ntiles = std::int32_t( tn.size() );
		_nblocks = std::int32_t( bn.size() );
		_nflush = std::int32_t( fn.size() );
		_window = 0;
		_graphs.clear();
		if constexpr( windowed )
		{
			// the longest window that suits every net and whose LDS leaves room for four workgroups
			// on a CU
			int widest = 64;
			_window = WINDOW_MAX;
			for( auto * n : _nets )
			{
				_window = std::min( _window, window_cap<Model>( n->params().delay ) );
				widest = std::max( widest, int( n->get_launch().tile_w ) );
				_logged = _logged || n->logged();
			}
			auto bytes = [&]( int w ) { return _fixed ? window_lds<Model, true>::bytes( window_block, widest, w ) : window_lds<Model, false>::bytes( window_block, widest, w ); };
			while( _window > 1 && bytes( _window ) > LDS_PER_CU / 4 ) _window = window_steps( _window - 1 );
			_lds = bytes( _window );
			if( !_windows ) _window = 0;
			allow_lds( _fixed ? reinterpret_cast<void const *>( &k_batch_window<Model, true, window_block> ) : reinterpret_cast<void const *>( &k_batch_window<Model, false, window_block> ),
			           _lds );
		}
		// all tables in one buffer and one copy
		std::vector<unsigned char> all;
		auto put = [&]( auto const & h ) { // the place of h's copy
			std::size_t const at = ( all.size() + 255 ) / 256 * 256;
			all.resize( at + h.size() * sizeof( h[0] ) );
			if( !h.empty() ) std::memcpy( all.data() + at, h.data(), h.size() * sizeof( h[0] ) );
			return at;
		};
		std::size_t at[7], at_views[CLOCK_SLOTS];
		{
			int k = 0;
			for( auto const * h : { &tn, &tl, &bn, &bl, &fn, &fl, &fc } ) at[k++] = put( *h );
		}
		for( int p = 0; p < CLOCK_SLOTS; p++ ) at_views[p] = put( vs[p] );
		_tables.resize( all.size() );
		SPICE_HIP( hipMemcpyAsync( _tables.data(), all.data(), all.size(), hipMemcpyHostToDevice, _s ) );
		{
			int k = 0;
			for( auto * table : { &_tile_net, &_tile_local, &_block_net, &_block_local, &_flush_net, &_flush_local, &_flush_count } )
				*table = reinterpret_cast<std::int32_t const *>( _tables.data() + at[k++] );
		}
		for( int p = 0; p < CLOCK_SLOTS; p++ ) _views[p] = reinterpret_cast<dview const *>( _tables.data() + at_views[p] );
		_grid_tiles = std::min( _ntiles, ( recv_block == 256 ? SPICE_BATCH_GRID_PER_CU : SPICE_BATCH_GRID_PER_CU / 4 ) * device_cu_count() );
		for( auto * n : _nets ) n->synchronize();
		SPICE_HIP( hipStreamSynchronize( _s ) );
		_built = true;
	}

	// The tables are those of the nets as they are now.
	void ready()
	{
		bool stale = !_built;
		if constexpr( factored_v<Model> )
			for( auto * n : _nets ) stale = stale || ( _windows && n->lazy() );
		if( !stale ) return;
		synchronize();
		build();
	}

	// Delivery tile width of a net of n neurons (at `tile_w` now) in a batch of nnets. Many nets
	// already fill the GPU, so then a batched net does not need many small delivery tiles: fewer
	// workgroups, each with a fixed staging cost (every tile stages all of a window's arrivals). A
	// batch of a few nets keeps its nets' own tiles. Fixed-point results do not depend on the tile
	// width (fp32 sums are reordered, as by any launch shape); a net keeps wider tiles it already
	// has (of up to TILE_MAX, what the batched kernels hold), and keeps the new width afterwards.
	// Static nets step by step (delay 1) 192 at least, as fewer tiles reserve their spikes' places on a net's one
	// counter (us per step with 64 and 192: 20 nets of up to 10,000 neurons, brunel_3pop 9.2, 8.7,
	// synth 8.5, 8.1, Vogels 8.5, 8.1). Two-kernel steps: about max(64, 64 x CUs / nets) tiles per net (on a sweep of two 256-net
	// batches 64 tiles per net beat 16, 32, 128 and 256).
	static int batch_tile_w( std::int64_t n, int tile_w, std::int64_t nnets, int delay )
	{
		std::int64_t const tiles = windowed ? std::max<std::int64_t>( 1, window_tiles_per_cu * device_cu_count() / nnets )
		                                    : std::max<std::int64_t>( 64, std::int64_t( SPICE_BATCH_ITEMS_PER_CU ) * device_cu_count() / nnets );
		int const least = windowed && !plastic && window_cap<Model>( delay ) == 1 ? BATCH_TILE : 64;
		int const tw = int( std::clamp<std::int64_t>( ( n / tiles + 63 ) / 64 * 64, least, TILE_MAX ) );
		return std::min( std::max( tw, tile_w ), TILE_MAX );
	}

	~hip_batch() override
	{
		if( _s ) (void)hipStreamSynchronize( _s );
		_owned.clear(); // (before the graphs, as in hip_net)
		_graphs.clear();
		_queue.clear();
		if( _s && _own_stream ) (void)hipStreamDestroy( _s );
	}

	void run( std::int64_t n ) override
	{
		if( n < 0 ) throw std::invalid_argument( "negative step count" );
		if( n == 0 ) return;
		ready();
		for( auto * net : _nets ) net->require_whole();
		// (state imported into a net may ask for a few steps one by one)
		std::int64_t single = 0;
		for( auto * net : _nets ) single = std::max( single, net->single_steps_left() );
		single = std::min( single, n );
		if( single ) launch_windows( _step, single, 1, true );
		_step += single;
		for( auto * net : _nets ) net->advance_host( single );
		n -= single;
		if( n == 0 ) return;
		if( _window > 1 )
		{
			launch_windows( _step, n, _window );
			_step += n;
			for( auto * net : _nets ) net->advance_host( n );
			return;
		}
		if( _graphs.empty() ) _graphs.capture( _s, [&]( int t, int len ) { launch_steps( t, len ); } );
		_graphs.run( _s, _step, n, [&] { _step++; } );
		for( auto * net : _nets ) net->advance_host( n );
	}

	void begin_spike_log( std::int64_t nsteps ) override
	{
		for( auto * net : _nets ) net->note_spike_log( nsteps ); // validates nsteps first
		ready();
		std::int32_t const n = std::int32_t( _nets.size() );
		SPICE_LAUNCH( k_batch_log_window<<<unsigned( ( n + 255 ) / 256 ), 256, 0, _s>>>( _views[_step & ( CLOCK_SLOTS - 1 )], n, nsteps ) );
	}

	void synchronize() override
	{
		SPICE_HIP( hipStreamSynchronize( _s ) );
	}
	int size() const override { return int( _nets.size() ); }
	net_iface * net( int i ) override
	{
		if( i < 0 || i >= size() ) throw std::invalid_argument( "net index out of range" );
		return _nets[i];
	}

private:
	std::vector<hip_net<Model> *> _nets;
	std::vector<std::unique_ptr<hip_net<Model>>> _owned;
	hipStream_t _s = nullptr;
	bool _own_stream = false;
	step_graphs _graphs;
	bool _fixed = false;
	bool _windows = false; // steps run as windows
	bool _built = false;   // build() went through
	// windows of up to _window steps (0: two-kernel steps)
	static constexpr int window_block = 256;
	// tiles of all nets, per CU: 48 nets of 1e4 to 1e7 synapses take, at 4 / 8 / 16 / 64, 2.6 / 1.8 /
	// 1.8 / 1.9 us per step in windows of 15 steps and 11.0 / 10.6 / 14.5 / 18.3 step by step (10.3
	// and 14.7 with a delivery and an update kernel, or an overlapped one, per step)
	static constexpr std::int64_t window_tiles_per_cu = 8;
	int _window = 0;
	bool _logged = false; // some net has a spike log
	std::size_t _lds = 0;
	launch_queue _queue;
	std::int64_t _step = 0;
	std::int32_t _ntiles = 0, _nblocks = 0, _nflush = 0;
	int _grid_tiles = 0;
	dbuf<unsigned char> _tables; // all of these:
	std::int32_t const *_tile_net = nullptr, *_tile_local = nullptr, *_block_net = nullptr, *_block_local = nullptr;
	std::int32_t const *_flush_net = nullptr, *_flush_local = nullptr, *_flush_count = nullptr;
	dview const * _views[CLOCK_SLOTS] = {};

	// n steps from batch step t in windows of up to `most`; each appends its predecessor's spikes
	// to the nets' logs, and a last kernel the last one's. alone: the passes before each in kernels
	// of their own.
	void launch_windows( std::int64_t t, std::int64_t n, int most, bool alone = false )
	{
		int before = 0;
		while( n > 0 )
		{
			int const w = window_steps( std::min<std::int64_t>( n, most ) );
			if( alone )
				for( auto * net : _nets ) net->launch_passes( net->host_step() + ( t - _step ), _s );
			if( _fixed )
				launch_window_t<true>( t, w, before, alone );
			else
				launch_window_t<false>( t, w, before, alone );
			if( _window > 1 ) _queue.launched( _s );
			before = w;
			t += w;
			n -= w;
		}
		if( _logged ) SPICE_LAUNCH( k_batch_log<<<unsigned( _nets.size() ), 256, 0, _s>>>( _views[t & ( CLOCK_SLOTS - 1 )], before ) );
	}

	template <bool F>
	void launch_window_t( std::int64_t t, int w, int before, bool alone )
	{
		std::int32_t const nplast = alone ? 0 : _nflush;
		unsigned const grid = unsigned( _ntiles + nplast ) + ( _logged && before ? unsigned( _nets.size() ) : 0u );
		if constexpr( windowed )
			SPICE_LAUNCH( ( k_batch_window<Model, F, window_block><<<grid, window_block, _lds, _s>>>(
			    _views[t & ( CLOCK_SLOTS - 1 )], _tile_net, _tile_local, _ntiles, w, before, _flush_net,
			    _flush_local, _flush_count, nplast ) ) );
	}

	// Same schedules as hip_net::launch_steps: windows of one step, or two kernels per step
	// (delivery with step t - 1's plasticity, update).
	void launch_steps( std::int64_t t, std::int64_t len )
	{
		if( _windows )
		{
			launch_windows( t, len, 1 );
			return;
		}
		for( std::int64_t k = 0; k < len; k++ )
			if( _fixed )
				launch_step_t<true>( t + k );
			else
				launch_step_t<false>( t + k );
	}

	template <bool F>
	void launch_step_t( std::int64_t t )
	{
		if constexpr( !windowed || factored_v<Model> )
		{
			dview const * v = _views[t & ( CLOCK_SLOTS - 1 )];
			unsigned const grid = unsigned( _grid_tiles + ( plastic ? _nflush : 0 ) );
			SPICE_LAUNCH( k_batch_receive<Model, F, recv_block><<<grid, recv_block, 0, _s>>>( v, _tile_net, _tile_local, _ntiles, _grid_tiles,
			                                                                                    _flush_net, _flush_local, _flush_count ) );
			SPICE_LAUNCH( k_batch_update<Model, F><<<_nblocks, 256, 0, _s>>>( v, _block_net, _block_local ) );
		}
	}
};

// Builds the nets of a batch (each gets its own stream for setup) and the batch, which owns
// them and `s`.
template <typename Model>
batch_iface * make_batch( std::vector<net_params> const & ps, std::vector<csr_dev> && gs, hipStream_t s )
{
	std::vector<std::unique_ptr<hip_net<Model>>> nets;
	std::vector<hip_net<Model> *> raw;
	for( std::size_t k = 0; k < ps.size(); k++ )
	{
		hipStream_t ns = nullptr;
		SPICE_HIP( hipStreamCreateWithFlags( &ns, hipStreamNonBlocking ) );
		try
		{
			launch_cfg first; // at the width that the batch will want
			first.tile_w = hip_batch<Model>::batch_tile_w( gs[k].n, default_tile_w<Model>( gs[k].n, gs[k].targets, ps[k].delay, device_cu_count() ), std::int64_t( ps.size() ), ps[k].delay );
			net_params p = ps[k];
			p.batched = true;
			nets.emplace_back( new hip_net<Model>( p, std::move( gs[k] ), ns, first ) );
		}
		catch( ... )
		{
			(void)hipStreamDestroy( ns );
			throw;
		}
		raw.push_back( nets.back().get() );
	}
	return new hip_batch<Model>( std::move( raw ), std::move( nets ), s, true );
}

// A batch over nets owned elsewhere (all of model `Model`); `s` stays the caller's.
template <typename Model>
batch_iface * make_group( std::vector<net_iface *> const & nets, hipStream_t s )
{
	std::vector<hip_net<Model> *> raw;
	for( auto * n : nets )
	{
		auto * h = dynamic_cast<hip_net<Model> *>( n );
		if( !h ) throw std::invalid_argument( "batch nets must all be of the batch's model" );
		raw.push_back( h );
	}
	return new hip_batch<Model>( std::move( raw ), {}, s, false );
}
} // namespace spice::hipx
