#pragma once
// Host side of one simulated network on one GPU: owns every device buffer, the HIP stream
// and the captured step graphs, and launches the kernels of kernels.h.
//
// Reference counterpart: cuda::snn<Model> (spice/cuda/snn.h:16-77, spice/cuda/snn.d.cpp).
#include "common.h"
#include "dview.h"
#include "graph.h"
#include "graphs.h"
#include "kernels.h"
#include "rules.h"
#include "window.h"

#include <spice/models/model.h>
#include <spice/util/graphgen.h>
#include <spice/util/numeric.h>
#include <spice_hip.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace spice::hipx
{
struct net_params
{
	int model;
	float dt;
	int delay;
	std::uint64_t seed;
	std::uint32_t flags;
	float param[4];
	bool batched = false;   // made for a batch: no segment records (memory for speed), tiles that a batch keeps
	bool own_stream = true; // the net destroys its stream (on failure: make_net does)
};

// Pinned memory through which the nets of this process read small answers back (their number and
// `words` words): one buffer, held by the nets that use it.
struct host_stage
{
	static constexpr std::uint32_t words = 16384;
	std::uint32_t * host = nullptr;
	std::mutex busy;

	host_stage() = default;
	host_stage( host_stage const & ) = delete;
	~host_stage()
	{
		if( host ) (void)hipHostFree( host );
	}

	// nullptr: no memory
	static std::shared_ptr<host_stage> get()
	{
		static std::mutex m;
		static std::weak_ptr<host_stage> last;
		std::lock_guard<std::mutex> g( m );
		if( auto s = last.lock() ) return s;
		auto s = std::make_shared<host_stage>();
		void * p = nullptr;
		if( hipHostMalloc( &p, ( words + 1 ) * 4, hipHostMallocPortable ) != hipSuccess )
		{
			(void)hipGetLastError();
			return nullptr;
		}
		s->host = static_cast<std::uint32_t *>( p );
		last = s;
		return s;
	}
};

struct launch_cfg
{
	std::int32_t tile_w = 0, flush_slots = 0, flush_grid = 0, recv_block = 0, recv_parts = 0;
};

// Model-independent interface used by the C ABI.
struct net_iface
{
	virtual ~net_iface() = default;
	virtual void step( std::int32_t ** dspk, std::uint32_t ** dcnt ) = 0;
	virtual void run( std::int64_t n ) = 0;
	virtual void run_profiled( std::int64_t n, double * kernel_ms ) = 0;
	virtual void copy_spikes( std::int32_t * out, std::uint64_t cap, std::uint64_t * count ) = 0;
	virtual void synchronize() = 0;
	virtual net_params const & params() const = 0;
	virtual std::int64_t num_neurons() const = 0;
	virtual std::int64_t width() const = 0;
	virtual std::int64_t num_edges() const = 0;
	virtual void get_clock( std::int64_t * step, float * sum, float * c ) const = 0;
	virtual void set_clock( std::int64_t step, float sum, float c ) = 0;
	virtual void get_stats( spice_stats * out ) = 0;
	virtual void reset_stats() = 0;
	virtual void export_csr( std::int64_t * row_ptr, std::int32_t * col ) = 0;
	// rows [r0, r1): r1 - r0 + 1 absolute offsets, and (col != nullptr) their target ids
	virtual void export_csr_rows( std::int64_t r0, std::int64_t r1, std::int64_t * row_ptr, std::int32_t * col, std::uint64_t col_cap ) = 0;
	virtual void export_adj( std::int32_t * ell, std::uint64_t cap ) = 0;
	virtual void export_neuron_attr( int a, void * out, std::uint64_t bytes ) = 0;
	virtual void import_neuron_attr( int a, void const * in, std::uint64_t bytes ) = 0;
	virtual void export_synapse_attr( int a, void * out, std::uint64_t bytes, bool ell ) = 0;
	virtual void import_synapse_attr( int a, void const * in, std::uint64_t bytes, bool ell ) = 0;

	// Spike log (served jobs). enable_spike_log allocates a log of `cap` ids for windows of at
	// most `max_steps` steps (before the first run); begin_spike_log opens a window over the
	// next `nsteps` steps; once the net has run exactly those steps, read_spike_log copies the
	// window out, to pinned memory: off[0..nsteps] (off[k] = first id of step t0+k, off[nsteps] =
	// total) and the ids, and returns the total (> cap: the log overflowed, ids past cap were
	// dropped). No step of the net may be in flight during begin/read.
	virtual void enable_spike_log( std::uint64_t cap, std::int64_t max_steps ) = 0;
	virtual void begin_spike_log( std::int64_t nsteps ) = 0;
	virtual std::uint64_t read_spike_log( std::uint64_t * off, std::int32_t * ids, std::uint64_t cap ) = 0;
	virtual std::uint64_t device_bytes() const = 0;
	virtual std::int64_t host_step() const = 0;

	// Launch shapes (see hip_net::apply_launch) and a copy of the net (graph, neuron and
	// synapse state as stored; clock and plasticity bookkeeping start afresh) for tuning them.
	virtual launch_cfg get_launch() const = 0;
	virtual void set_launch( launch_cfg c ) = 0;
	virtual net_iface * clone() const = 0;
	virtual bool is_plastic() const = 0;
	virtual int max_tile_w() const = 0; // widest tile_w set_launch accepts
	virtual bool splits_delivery() const = 0; // whether the steps' kernels depend on recv_parts
};

inline int device_cu_count()
{
	static int cus = [] {
		int dev = 0;
		SPICE_HIP( hipGetDevice( &dev ) );
		hipDeviceProp_t p;
		SPICE_HIP( hipGetDeviceProperties( &p, dev ) );
		return p.multiProcessorCount > 0 ? p.multiProcessorCount : 256;
	}();
	return cus;
}

// Longest window of steps one kernel may run (k_window).
template <typename Model>
int window_cap( int delay )
{
	return windowed_v<Model> && delay >= 2 ? std::max( 1, window_steps( std::min( delay, longest_window_v<Model> ) ) ) : 1;
}

constexpr int REC_TILE = 768; // widest tile that segment records alone are a reason for (default_launch)
constexpr int BATCH_TILE = 192; // narrowest tile of a batch's nets that run step by step (hip_batch::batch_tile_w)

// Targets per delivery tile of a new network (rules.h).
template <typename Model>
int default_tile_w( std::int64_t n, std::int64_t targets, int delay, int cus )
{
	return windowed_v<Model> ? window_tile_w( n, targets, is_plastic_v<Model>, overlap_capable_v<Model> && delay >= 2, cus ) : lazy_tile_w( n, cus );
}

template <typename Model>
class hip_net final : public net_iface
{
	using N = typename Model::neuron;
	using S = typename Model::synapse;
	static constexpr bool plastic = is_plastic_v<Model>;
	static constexpr bool traced = plastic && has_neuron_traces_v<S>;
	static constexpr bool windowed = windowed_v<Model>; // steps run as windows (static models: at most launch shapes)
	static constexpr bool factored = factored_v<Model>; // factored traces (a net may go back to the per-synapse contract)
	static constexpr bool eager = traced || factored;   // traces kept per neuron

public:
	// first: launch shapes to start with (zero fields: the defaults)
	hip_net( net_params const & p, csr_dev && g, hipStream_t stream, launch_cfg first = {} )
	    : _p( p )
	    , _g( std::move( g ) )
	    , _s( stream )
	    , _lazy( plastic && !eager )
	{
		if( !( p.dt > 0.0f ) ) throw std::invalid_argument( "dt must be positive" );
		if( p.flags & ~std::uint32_t( SPICE_FLAG_FIXED_POINT ) ) throw std::invalid_argument( "unknown flags" );
		if( p.delay < 1 ) throw std::invalid_argument( "delay must be >= 1" );
		if( plastic && p.delay > HISTORY - 1 )
			throw std::invalid_argument( "plastic models support delays of at most 255 steps" );
		if( _g.n < 1 || _g.n > INT_MAX - 1024 ) throw std::invalid_argument( "invalid neuron count" );
		static_assert( N::size <= MAXA && S::size <= MAXA, "at most 16 neuron/synapse attributes" );
		_ahead = overlap_capable_v<Model> && p.delay >= 2;
		arena::scope const small( _arena );
		allocate( first );
		initialize();
	}

	~hip_net() override
	{
		if( _s ) (void)hipStreamSynchronize( _s );
		// the large buffers first, so that the little that graphs hold stays among the freed memory that
		// the runtime keeps at hand (Brunel, 10,000 neurons, delay 1, after a run: 0.54 ms, 2.7 with the
		// graphs first)
		_recs.release();
		_col16.release();
		_segs.release();
		_offs.release();
		_tp_ent.release();
		for( auto & b : _sa ) b.release();
		_g.col.release();
		_graphs.clear();
		_queue.clear();
		if( _s && _p.own_stream ) (void)hipStreamDestroy( _s );
	}

	// ---- simulation ----
	void step( std::int32_t ** dspk, std::uint32_t ** dcnt ) override
	{
		require_whole();
		std::int64_t const t = _step;
		if( t < _single_until )
			launch_window( t, 1, nullptr, nullptr, true );
		else
			launch_steps( t, 1 );
		tick();
		int const slot = int( t % _v.rsize );
		if( dspk ) *dspk = _ring.data() + std::int64_t( slot ) * _g.n;
		if( dcnt ) *dcnt = _counts.data() + slot * COUNT_STRIDE;
	}

	// Replays captured step graphs (all of them captured at the first run; see graphs.h).
	void run( std::int64_t n ) override
	{
		if( n < 0 ) throw std::invalid_argument( "negative step count" );
		require_whole();
		while( n > 0 && _step < _single_until )
		{
			launch_window( _step, 1, nullptr, nullptr, true );
			_queue.launched( _s );
			tick();
			n--;
		}
		if( n == 0 ) return;
		if( _window > 1 )
		{
			// windows are long enough to be launched one by one (a launch costs the host a few us)
			while( n > 0 )
			{
				int const w = window_steps( std::min<std::int64_t>( n, _window ) );
				launch_window( _step, w, nullptr, nullptr );
				_queue.launched( _s );
				for( int i = 0; i < w; i++ ) tick();
				n -= w;
			}
			return;
		}
		if( _graphs.empty() ) _graphs.capture( _s, [&]( int t, int len ) { launch_steps( t, len ); } );
		_graphs.run( _s, _step, n, [&] { tick(); } );
	}

	// Runs n steps eagerly, each kernel with HIP events attached to its dispatch on the net's
	// stream, and adds the summed kernel durations (ms) to kernel_ms[0..2]: receive (delivery,
	// with the previous step's plasticity), update, and 0. Windows of static models: 0, 0 and the
	// window kernels; of plastic ones: the first window, the last one, and those between (a run
	// of fewer than three windows: all in [2]).
	void run_profiled( std::int64_t n, double * kernel_ms ) override
	{
		if( n < 0 ) throw std::invalid_argument( "negative step count" );
		require_whole();
		if( _window )
			run_profiled_windows( n, kernel_ms );
		else
			run_profiled_steps( n, kernel_ms );
	}

	void copy_spikes( std::int32_t * out, std::uint64_t cap, std::uint64_t * count ) override
	{
		if( _step == 0 )
		{
			*count = 0;
			return;
		}
		int const slot = int( ( _step - 1 ) % _v.rsize );
		std::int32_t const * ids = _ring.data() + std::int64_t( slot ) * _g.n;
		std::uint32_t const * cnt = _counts.data() + slot * COUNT_STRIDE;
		std::uint32_t c = 0;
		bool const staged = stage_to_host( ids, cnt, host_stage::words, [&]( std::uint32_t const * words, std::uint32_t n ) {
			c = n;
			if( out && c <= cap && c <= host_stage::words ) std::memcpy( out, words, std::size_t( c ) * 4 );
		} );
		if( !staged )
		{
			SPICE_HIP( hipMemcpyAsync( &c, cnt, 4, hipMemcpyDeviceToHost, _s ) );
			SPICE_HIP( hipStreamSynchronize( _s ) );
		}
		*count = c;
		if( out && c )
		{
			if( c > cap ) throw std::invalid_argument( "spike buffer too small" );
			if( staged && c <= host_stage::words ) return;
			SPICE_HIP( hipMemcpyAsync( out, ids, std::size_t( c ) * 4, hipMemcpyDeviceToHost, _s ) );
			SPICE_HIP( hipStreamSynchronize( _s ) );
		}
	}

	void synchronize() override { SPICE_HIP( hipStreamSynchronize( _s ) ); }

	// ---- queries ----
	net_params const & params() const override { return _p; }
	std::int64_t num_neurons() const override { return _g.n; }
	std::int64_t width() const override { return _g.width; }
	std::int64_t num_edges() const override { return _g.nnz; }

	void get_clock( std::int64_t * step, float * sum, float * c ) const override
	{
		*step = _step;
		*sum = float( _clock );
		*c = _clock.compensation();
	}

	// Moves the clock (conversion constructor / resume). Spikes in flight and the
	// plasticity bookkeeping are reset, after the plasticity of the steps before is done: synapse
	// state is current through step-1.
	void set_clock( std::int64_t step, float sum, float c ) override
	{
		if( step < 0 || step > INT_MAX - 2 ) throw std::invalid_argument( "invalid step index" );
		sync_synapses();
		if( factored && !_lazy )
		{
			// (the traces are synapse state: kept, as windows number them from 0 again)
			std::int64_t const from = trace_slot() * _g.n;
			if( from )
				for( auto * b : { &_xtr, &_ytr } ) SPICE_HIP( hipMemcpy( b->data(), b->data() + from, std::size_t( _g.n ) * 4, hipMemcpyDeviceToDevice ) );
		}
		ctl_t ctl{ step, sum, c, std::int32_t( step % _v.rsize ), 0, 0, 0.0f, 0.0f };
		SPICE_HIP( hipMemcpy( _ctl.data() + ( step & ( CLOCK_SLOTS - 1 ) ), &ctl, sizeof( ctl ), hipMemcpyHostToDevice ) );
		SPICE_HIP( hipMemset( _counts.data(), 0, _counts.bytes() ) );
		if constexpr( plastic )
		{
			SPICE_HIP( hipMemset( _hring.data(), 0, _hring.bytes() ) );
			SPICE_HIP( hipMemset( _fl_count.data(), 0, _fl_count.bytes() ) );
			reset_caught();
			if constexpr( eager ) reset_eager( traced );
			if( _lazy ) reset_lazy( std::int32_t( step - 1 ) );
		}
		_single_until = 0;
		_step = step;
		_clock.set( sum, c );
		_dt_last = 0.0f;
	}

	void get_stats( spice_stats * out ) override
	{
		sync_counted();
		std::vector<unsigned long long> b( _bstats.size() );
		SPICE_HIP( hipMemcpyAsync( b.data(), _bstats.data(), _bstats.bytes(), hipMemcpyDeviceToHost, _s ) );
		SPICE_HIP( hipStreamSynchronize( _s ) );
		unsigned long long t[NSTAT] = {};
		for( std::size_t i = 0; i < b.size(); i++ ) t[i % NSTAT] += b[i];
		*out = { std::uint64_t( _step - _stats_step0 ), t[ST_SPIKES], t[ST_EVENTS], t[ST_PLASTIC], t[ST_FLUSH_ROWS],
		         t[ST_FLUSH_SYN], t[ST_FLUSH_SLOTS], t[ST_FLUSH_WRITTEN] };
	}
	void reset_stats() override
	{
		sync_counted();
		SPICE_HIP( hipMemsetAsync( _bstats.data(), 0, _bstats.bytes(), _s ) );
		synchronize();
		_stats_step0 = _step;
	}

	// ---- export / import ----
	void export_csr( std::int64_t * row_ptr, std::int32_t * col ) override
	{
		synchronize();
		SPICE_HIP( hipMemcpy( row_ptr, _g.row_ptr.data(), ( _g.n + 1 ) * 8, hipMemcpyDeviceToHost ) );
		if( _g.nnz ) SPICE_HIP( hipMemcpy( col, _g.col.data(), _g.nnz * 4, hipMemcpyDeviceToHost ) );
	}

	void export_csr_rows( std::int64_t r0, std::int64_t r1, std::int64_t * row_ptr, std::int32_t * col, std::uint64_t col_cap ) override
	{
		synchronize();
		SPICE_HIP( hipMemcpy( row_ptr, _g.row_ptr.data() + r0, std::size_t( r1 - r0 + 1 ) * 8, hipMemcpyDeviceToHost ) );
		if( !col ) return;
		std::int64_t const cnt = row_ptr[r1 - r0] - row_ptr[0];
		if( std::uint64_t( cnt ) > col_cap ) throw std::invalid_argument( "column buffer too small for the row range" );
		if( cnt ) SPICE_HIP( hipMemcpy( col, _g.col.data() + row_ptr[0], std::size_t( cnt ) * 4, hipMemcpyDeviceToHost ) );
	}

	void export_adj( std::int32_t * ell, std::uint64_t cap ) override
	{
		if( cap < std::uint64_t( _g.n * _g.width ) ) throw std::invalid_argument( "adjacency buffer too small" );
		std::vector<std::int64_t> rp( _g.n + 1 );
		std::vector<std::int32_t> col( _g.nnz );
		export_csr( rp.data(), col.data() );
		for( std::int64_t r = 0; r < _g.n; r++ )
		{
			std::int64_t const len = rp[r + 1] - rp[r];
			std::copy( col.begin() + rp[r], col.begin() + rp[r + 1], ell + r * _g.width );
			std::fill( ell + r * _g.width + len, ell + ( r + 1 ) * _g.width, INT_MAX );
		}
	}

	void export_neuron_attr( int a, void * out, std::uint64_t bytes ) override
	{
		check_attr( a, int( N::size ) );
		if( bytes != std::uint64_t( _g.n ) * attr_bytes<N>( a ) ) throw std::invalid_argument( "buffer size mismatch" );
		if( bytes % 4 == 0 && bytes / 4 <= host_stage::words &&
		    stage_to_host( _na[a].data(), nullptr, std::uint32_t( bytes / 4 ), [&]( std::uint32_t const * words, std::uint32_t ) { std::memcpy( out, words, bytes ); } ) )
			return;
		synchronize();
		SPICE_HIP( hipMemcpy( out, _na[a].data(), bytes, hipMemcpyDeviceToHost ) );
	}
	void import_neuron_attr( int a, void const * in, std::uint64_t bytes ) override
	{
		check_attr( a, int( N::size ) );
		if( bytes != std::uint64_t( _g.n ) * attr_bytes<N>( a ) ) throw std::invalid_argument( "buffer size mismatch" );
		synchronize();
		if constexpr( plastic && windowed )
			if( _step > 0 && !_lazy )
			{
				// The imported state need not keep the refractory promise towards spikes before it:
				// until those have arrived, steps run one by one, the passes of each before the next.
				sync_synapses();
				_single_until = _step + _p.delay + _v.wcap;
			}
		SPICE_HIP( hipMemcpy( _na[a].data(), in, bytes, hipMemcpyHostToDevice ) );
	}

	void export_synapse_attr( int a, void * out, std::uint64_t bytes, bool ell ) override
	{
		check_attr( a, int( S::size ) );
		std::size_t const sz = attr_bytes<S>( a );
		if( bytes != ( ell ? std::uint64_t( _g.n * _g.width ) : std::uint64_t( _g.nnz ) ) * sz )
			throw std::invalid_argument( "buffer size mismatch" );
		sync_synapses();
		dbuf<float> expanded; // a factored trace as synapse attribute
		char const * src = _sa[a].data();
		if constexpr( factored )
			if( !_lazy && is_factored_attr<S>( a ) )
			{
				expanded.resize( std::size_t( _g.nnz ) + 1 );
				expand_trace( a, expanded.data() );
				src = reinterpret_cast<char const *>( expanded.data() );
			}
		if( !ell )
		{
			if( _g.nnz ) SPICE_HIP( hipMemcpy( out, src, bytes, hipMemcpyDeviceToHost ) );
			return;
		}
		std::vector<char> csr( _g.nnz * sz );
		if( _g.nnz ) SPICE_HIP( hipMemcpy( csr.data(), src, csr.size(), hipMemcpyDeviceToHost ) );
		std::vector<std::int64_t> rp( _g.n + 1 );
		SPICE_HIP( hipMemcpy( rp.data(), _g.row_ptr.data(), rp.size() * 8, hipMemcpyDeviceToHost ) );
		char * o = static_cast<char *>( out );
		std::memset( o, 0, bytes );
		for( std::int64_t r = 0; r < _g.n; r++ )
			std::memcpy( o + r * _g.width * sz, csr.data() + rp[r] * sz, ( rp[r + 1] - rp[r] ) * sz );
	}

	void import_synapse_attr( int a, void const * in, std::uint64_t bytes, bool ell ) override
	{
		check_attr( a, int( S::size ) );
		std::size_t const sz = attr_bytes<S>( a );
		if( bytes != ( ell ? std::uint64_t( _g.n * _g.width ) : std::uint64_t( _g.nnz ) ) * sz )
			throw std::invalid_argument( "buffer size mismatch" );
		sync_synapses();
		if( !ell )
		{
			store_synapse_attr( a, in );
			return;
		}
		std::vector<std::int64_t> rp( _g.n + 1 );
		SPICE_HIP( hipMemcpy( rp.data(), _g.row_ptr.data(), rp.size() * 8, hipMemcpyDeviceToHost ) );
		std::vector<char> csr( _g.nnz * sz );
		char const * src = static_cast<char const *>( in );
		for( std::int64_t r = 0; r < _g.n; r++ )
			std::memcpy( csr.data() + rp[r] * sz, src + r * _g.width * sz, ( rp[r + 1] - rp[r] ) * sz );
		store_synapse_attr( a, csr.data() );
	}

	// ---- spike log ----
	void enable_spike_log( std::uint64_t cap, std::int64_t max_steps ) override
	{
		if( !_graphs.empty() || _slog_ctl.size() ) throw std::logic_error( "the spike log is enabled once, before the first run" );
		if( max_steps < 1 ) throw std::invalid_argument( "spike log window must hold at least one step" );
		arena::scope const small( _arena );
		_slog_ctl.resize( 1 );
		_slog_ids.resize( std::max<std::uint64_t>( cap, 1 ) );
		_slog_off.resize( std::size_t( max_steps ) );
		_slog_cap = cap;
		_slog_max = max_steps;
		slog_t const w{ 0, 0, cap }; // empty window
		SPICE_HIP( hipMemcpy( _slog_ctl.data(), &w, sizeof( w ), hipMemcpyHostToDevice ) );
		for( dview * v : { &_v, &_vs[0], &_vs[1], &_vs[2], &_vs[3] } )
		{
			v->slog = _slog_ctl.data();
			v->slog_ids = _slog_ids.data();
			v->slog_off = _slog_off.data();
		}
	}

	void begin_spike_log( std::int64_t nsteps ) override
	{
		if( !_slog_ctl.size() ) throw std::logic_error( "spike log not enabled" );
		if( nsteps < 0 || nsteps > _slog_max ) throw std::invalid_argument( "spike log window too long" );
		slog_t const w{ _step, nsteps, _slog_cap };
		SPICE_HIP( hipMemcpy( _slog_ctl.data(), &w, sizeof( w ), hipMemcpyHostToDevice ) );
		note_spike_log( nsteps );
	}

	// Host bookkeeping of a window whose device side a batch opened (k_batch_log_window).
	void note_spike_log( std::int64_t nsteps )
	{
		if( !_slog_ctl.size() ) return;
		if( nsteps < 0 || nsteps > _slog_max ) throw std::invalid_argument( "spike log window too long" );
		_slog_t0 = _step;
		_slog_n = nsteps;
	}

	std::uint64_t read_spike_log( std::uint64_t * off, std::int32_t * ids, std::uint64_t cap ) override
	{
		if( !_slog_ctl.size() ) throw std::logic_error( "spike log not enabled" );
		if( _step != _slog_t0 + _slog_n ) throw std::logic_error( "spike log window not completed" );
		off[0] = 0;
		if( _slog_n == 0 ) return 0;
		SPICE_LAUNCH( k_log_out<<<16, 1024, 0, _s>>>( _slog_off.data(), _slog_n, _counts.data() + ( _step - 1 ) % _v.rsize * COUNT_STRIDE, _slog_ids.data(),
		                                              std::min( _slog_cap, cap ), off, ids ) );
		SPICE_HIP( hipStreamSynchronize( _s ) );
		std::uint64_t const total = off[_slog_n];
		return total;
	}

	std::uint64_t device_bytes() const override
	{
		std::uint64_t b = _g.row_ptr.bytes() + _g.col.bytes();
		for( int a = 0; a < MAXA; a++ ) b += _na[a].bytes() + _acc[a].bytes() + _sa[a].bytes();
		b += _ring.bytes() + _counts.bytes() + _hring.bytes() + _last_spk.bytes() + _synced.bytes() + _pend.bytes() +
		     _fl_id.bytes() + _fl_synced.bytes() + _fl_pend.bytes() + _hasp.bytes() + _pl_lo.bytes() + _pl_hi.bytes() +
		     _fl_count.bytes() + _xtr.bytes() + _ytr.bytes() + _fl8.bytes() + _xpost.bytes() + _sp8.bytes() + _po_id.bytes() + _po_count.bytes() +
		     _tp_ptr.bytes() + _caught.bytes() + _tp_ent.bytes() + _ctl.bytes() + _bstats.bytes() +
		     _segs.bytes() + _offs.bytes() + _recs.bytes() + _col16.bytes() + _slog_ctl.bytes() + _slog_ids.bytes() + _slog_off.bytes();
		return b;
	}

	// ---- launch shapes ----
	launch_cfg get_launch() const override { return _lc; }
	void set_launch( launch_cfg c ) override
	{
		synchronize();
		apply_launch( c );
	}
	bool is_plastic() const override { return plastic; }
	// (windows of several steps, and of plastic models, have one workgroup per tile whatever it says)
	bool splits_delivery() const override { return !windowed || _lazy || ( !plastic && !_ahead ); }
	// widest delivery tile: wide tiles for static models that run step by step
	int max_tile_w() const override { return !plastic && !_ahead ? TILE_WIDE : TILE_MAX; }

	net_iface * clone() const override
	{
		// the original is only read (its lazily updated synapses are copied as they are)
		const_cast<hip_net *>( this )->synchronize();
		hipStream_t s = nullptr;
		SPICE_HIP( hipStreamCreateWithFlags( &s, hipStreamNonBlocking ) );
		try
		{
			csr_dev g;
			g.n = _g.n;
			g.nnz = _g.nnz;
			g.width = _g.width;
			g.targets = _g.targets;
			g.row_ptr.resize( _g.row_ptr.size() );
			g.col.resize( _g.col.size() );
			SPICE_HIP( hipMemcpyAsync( g.row_ptr.data(), _g.row_ptr.data(), _g.row_ptr.bytes(), hipMemcpyDeviceToDevice, s ) );
			SPICE_HIP( hipMemcpyAsync( g.col.data(), _g.col.data(), _g.col.bytes(), hipMemcpyDeviceToDevice, s ) );
			SPICE_HIP( hipStreamSynchronize( s ) );
			net_params p = _p;
			p.own_stream = true;
			auto * c = new hip_net( p, std::move( g ), s );
			s = nullptr; // owned by c
			if constexpr( factored )
			{
				if( _lazy )
					c->make_lazy();
				else
				{
					std::int64_t const from = trace_slot() * _g.n;
					SPICE_HIP( hipMemcpy( c->_xtr.data(), _xtr.data() + from, std::size_t( _g.n ) * 4, hipMemcpyDeviceToDevice ) );
					SPICE_HIP( hipMemcpy( c->_ytr.data(), _ytr.data() + from, std::size_t( _g.n ) * 4, hipMemcpyDeviceToDevice ) );
				}
			}
			for( int a = 0; a < MAXA; a++ )
			{
				if( _na[a].bytes() ) SPICE_HIP( hipMemcpy( c->_na[a].data(), _na[a].data(), _na[a].bytes(), hipMemcpyDeviceToDevice ) );
				if( _sa[a].bytes() ) SPICE_HIP( hipMemcpy( c->_sa[a].data(), _sa[a].data(), _sa[a].bytes(), hipMemcpyDeviceToDevice ) );
			}
			c->apply_launch( _lc );
			return c;
		}
		catch( ... )
		{
			if( s ) (void)hipStreamDestroy( s );
			throw;
		}
	}

	// ---- used by hip_batch (batched stepping of many nets) ----
	dview const & view( int slot ) const { return _vs[slot & ( CLOCK_SLOTS - 1 )]; }
	int num_tiles() const { return _v.nact; } // the delivery's tiles (those with incoming synapses)
	int num_all_tiles() const { return _v.ntiles; }
	std::int64_t single_steps_left() const { return std::max<std::int64_t>( 0, _single_until - _step ); }
	bool lazy() const { return _lazy; }

	// The passes due before step t in a kernel of their own.
	void launch_passes( std::int64_t t, hipStream_t s )
	{
		if constexpr( plastic && windowed )
		{
			dview const & v = _vs[t & ( CLOCK_SLOTS - 1 )];
			if( fixed() )
				SPICE_LAUNCH( ( k_window_passes<Model, true><<<_grid_flush, 256, 0, s>>>( v ) ) );
			else
				SPICE_LAUNCH( ( k_window_passes<Model, false><<<_grid_flush, 256, 0, s>>>( v ) ) );
		}
	}

	// Factored traces back to the per-synapse contract: the traces become synapse attributes, and
	// steps run as two kernels with lazy plasticity. For a layout whose plastic synapses join
	// neurons that do not keep the refractory promise, and for imported synapse state that is not of
	// the factored form.
	void make_lazy()
	{
		if constexpr( factored )
		{
			if( _lazy ) return;
			bool const fresh = _step == 0;
			sync_synapses();
			// All memory first, beside the by-target index, or else in its place; if it does not fit
			// there either, the index comes back and the net stays as it was.
			constexpr int traces[2] = { int( S::pre_trace ), int( S::post_trace ) };
			dbuf<char> kept[2];
			auto take = [&] {
				try
				{
					for( auto & b : kept ) b.resize( std::size_t( _g.nnz + COL_PAD ) * sizeof( float ) );
					alloc_lazy();
				}
				catch( ... )
				{
					for( auto & b : kept ) b.release();
					throw;
				}
			};
			try
			{
				take();
			}
			catch( std::bad_alloc const & )
			{
				if( !_tp_ent.size() ) throw;
				_whole = false;
				_tp_ent.release();
				try
				{
					take();
				}
				catch( ... )
				{
					build_by_target();
					throw;
				}
			}
			for( int k = 0; k < 2; k++ )
			{
				expand_trace( traces[k], reinterpret_cast<float *>( kept[k].data() ) );
				_sa[traces[k]] = std::move( kept[k] );
				_v.sa[traces[k]] = _sa[traces[k]].data();
			}
			_whole = false; // until the views are right
			_tp_ent.release();
			_tp_total = _tp_targets = 0;
			_lazy = true;
			_single_until = 0;
			reset_lazy( std::int32_t( _step - 1 ) );
			SPICE_HIP( hipMemset( _fl_count.data(), 0, _fl_count.bytes() ) );
			apply_launch( fresh ? launch_cfg{} : _lc );
		}
	}
	void require_whole() const
	{
		if( !_whole ) throw std::runtime_error( "the network lost buffers when memory ran out: set its launch shapes, or make it anew" );
	}
	bool logged() const { return _slog_ctl.size() > 0; }
	int num_receive_parts() const { return _v.rparts; }
	int num_update_blocks() const { return _grid_update; }
	// flush workgroups of this net inside a batch: about two per expected work item wave
	// (lazy: rows reach their flush about every FLUSH_AGE steps, and once after each arrival
	// of their spike; eager: arriving rows and spiking targets), at most the net's own grid
	int num_batch_flush_blocks() const
	{
		std::int64_t const items = !_lazy ? ( _g.n / 256 + 1 ) * _v.wcap * ( _v.fparts + _v.pparts ) : ( _g.n / FLUSH_AGE + _g.n / 256 + 1 ) * _v.fparts;
		return int( std::clamp<std::int64_t>( ( items + 1 ) / 2, 1, _grid_flush ) );
	}
	bool fixed() const { return ( _p.flags & SPICE_FLAG_FIXED_POINT ) != 0; }
	std::int64_t host_step() const override { return _step; }
	void advance_host( std::int64_t n )
	{
		for( std::int64_t k = 0; k < n; k++ ) tick();
	}

private:
	net_params _p;
	arena _arena; // the small ones of the buffers below
	csr_dev _g;
	hipStream_t _s = nullptr;
	step_graphs _graphs;

	dbuf<char> _na[MAXA], _acc[MAXA], _sa[MAXA];
	dbuf<std::int32_t> _ring;
	dbuf<std::uint32_t> _counts;
	dbuf<unsigned long long> _hring;
	dbuf<std::int32_t> _last_spk;
	dbuf<std::int32_t> _synced, _pend, _fl_id, _fl_synced, _fl_pend;
	dbuf<std::uint8_t> _hasp;
	dbuf<std::int32_t> _pl_lo, _pl_hi;
	dbuf<std::uint32_t> _fl_count;
	dbuf<std::uint32_t> _xpost;                // eager windows: see dview
	dbuf<float> _xtr, _ytr;                    // eager: traces, [2][N] by step parity or [4][N] by window
	dbuf<std::uint8_t> _fl8, _sp8;             // eager: [2][N] step flags, or the windows' arrivals and spikes
	dbuf<std::int32_t> _po_id;                 // eager: [2][N] spiking targets
	dbuf<std::uint32_t> _po_count;             // eager: [4]
	dbuf<std::int64_t> _tp_ptr;                // eager: by-target index offsets
	dbuf<std::int64_t> _caught;                // plastic: step whose plasticity a synchronization did
	dbuf<tp_entry> _tp_ent;                    // eager: by-target index entries
	std::int64_t _caught_host = -1;
	std::int64_t _tp_total = 0, _tp_targets = 0;
	dbuf<ctl_t> _ctl;
	dbuf<unsigned long long> _bstats;
	std::int64_t _stats_step0 = 0;
	dview _v{};                // step views: _vs[p] reads clock slot p
	dview _vs[CLOCK_SLOTS]{};

	int _grid_update = 0, _grid_flush = 0, _grid_tiles = 0;
	int _grid_upd = 0; // workgroups of this net's own update kernel (_upd_block threads)
	int _upd_block = SPICE_UPDATE_BLOCK;
	int _grid_plast = 0; // plasticity workgroups of the delivery kernel
	bool _ahead = false; // the delivery of a step may run before the updates of earlier steps
	std::int64_t _single_until = 0; // steps run one by one before this step (see import_neuron_attr)
	bool _lazy = false; // plasticity by the per-synapse contract
	bool _whole = false; // all buffers are there (see shape)
	int _window = 0;       // longest window of the window kernels that run the steps (0: none)
	launch_queue _queue;
	launch_cfg _lc{};
	std::shared_ptr<host_stage> _stage; // see stage_to_host
	int _staged = 0;                    // calls that asked for it
	dbuf<std::uint64_t> _segs;  // the segment table,
	dbuf<std::uint32_t> _offs;  // or offsets in its place
	dbuf<unsigned char> _recs; // segment records
	dbuf<std::uint16_t> _col16;       // low halves of the row store
	dbuf<std::int32_t> _tile_ids;
	std::int64_t _step = 0;
	util::kahan_sum<float> _clock;
	float _dt_last = 0.0f; // compensated dt of the last step (what its kernels used)

	// the host's copy of the clock advances with every enqueued step, as the device's does
	void tick()
	{
		_step++;
		_dt_last = _clock.add( _p.dt );
	}

	dbuf<slog_t> _slog_ctl;
	dbuf<std::int32_t> _slog_ids;
	dbuf<std::uint64_t> _slog_off;
	std::uint64_t _slog_cap = 0;
	std::int64_t _slog_max = 0, _slog_t0 = 0, _slog_n = 0;

	template <typename Decl>
	static std::size_t attr_bytes( int a )
	{
		std::size_t r = 0;
		util::for_n<Decl::size>( [&]( auto I ) {
			if( int( I ) == a ) r = sizeof( typename Decl::template type<I> );
		} );
		return r;
	}
	static void check_attr( int a, int n )
	{
		if( a < 0 || a >= n ) throw std::invalid_argument( "attribute index out of range" );
	}

	void allocate( launch_cfg const & first )
	{
		std::int64_t const n = _g.n;
		util::for_n<N::size>( [&]( auto I ) {
			using A = typename N::template type<I>;
			_na[I].resize( n * sizeof( A ) );
			if constexpr( ( ( receive_mask_v<N> >> I ) & 1u ) != 0 )
			{
				std::size_t const asz = ( std::is_floating_point_v<A> && true ) ? ( fixed() ? 8 : sizeof( A ) ) : sizeof( A );
				_acc[I].resize( 2 * n * asz ); // by step parity
				SPICE_HIP( hipMemsetAsync( _acc[I].data(), 0, _acc[I].bytes(), _s ) );
			}
		} );
		util::for_n<S::size>( [&]( auto I ) {
			using A = typename S::template type<I>;
			if constexpr( !factored || !is_factored_attr<S>( int( I ) ) ) _sa[I].resize( ( _g.nnz + COL_PAD ) * sizeof( A ) ); // (read in pieces like the row store)
		} );
		_v.wcap = window_cap<Model>( _p.delay );
		_v.rsize = ring_entries( _p.delay, _v.wcap );
		_ring.resize( std::size_t( _v.rsize ) * n );
		_counts.resize( std::size_t( _v.rsize ) * COUNT_STRIDE );
		SPICE_HIP( hipMemsetAsync( _counts.data(), 0, _counts.bytes(), _s ) );
		if constexpr( plastic )
		{
			_hring.resize( std::size_t( HWORDS ) * n );
			_hasp.resize( n );
			_pl_lo.resize( n );
			_pl_hi.resize( n );
			_fl_id.resize( 2 * n ); // lists of steps of both parities
			_fl_count.resize( CLOCK_SLOTS );
			_caught.resize( 1 );
			SPICE_HIP( hipMemsetAsync( _hring.data(), 0, _hring.bytes(), _s ) );
			SPICE_HIP( hipMemsetAsync( _fl_count.data(), 0, _fl_count.bytes(), _s ) );
			reset_caught();
			if constexpr( eager )
			{
				_xtr.resize( ( windowed ? 4 : 2 ) * n );
				_ytr.resize( ( windowed ? 4 : 2 ) * n );
				_fl8.resize( 2 * n );
				if( windowed ) _xpost.resize( 2 * n );
				if( windowed ) _sp8.resize( 2 * n );
				_po_id.resize( 2 * n );
				_po_count.resize( CLOCK_SLOTS );
				_tp_ptr.resize( n + 2 ); // (then the number of targets that have any)
				reset_eager( true );
			}
			if( _lazy )
			{
				alloc_lazy();
				reset_lazy( -1 );
			}
		}
		_ctl.resize( CLOCK_SLOTS );
		SPICE_HIP( hipMemsetAsync( _ctl.data(), 0, _ctl.bytes(), _s ) );

		dview & v = _v;
		v.N = std::int32_t( n );
		v.D = _p.delay;
		v.width = std::int32_t( std::min<std::int64_t>( _g.width, INT_MAX ) );
		v.shift = 40;
		v.DT = _p.dt;
		v.flags = _p.flags;
		v.seed = _p.seed;
		for( int k = 0; k < 4; k++ ) v.param[k] = _p.param[k];
		v.row_ptr = _g.row_ptr.data();
		v.col = _g.col.data();
		for( int a = 0; a < MAXA; a++ )
		{
			v.na[a] = _na[a].data();
			v.acc[a] = _acc[a].data();
			v.sa[a] = _sa[a].data();
		}
		v.ring = _ring.data();
		v.counts = _counts.data();
		v.hring = _hring.data();
		v.last_spk = _last_spk.data();
		v.synced = _synced.data();
		v.pend = _pend.data();
		v.hasp = _hasp.data();
		v.pl_lo = _pl_lo.data();
		v.pl_hi = _pl_hi.data();
		v.fl_id = _fl_id.data();
		v.fl_synced = _fl_synced.data();
		v.fl_pend = _fl_pend.data();
		v.fl_count = _fl_count.data();
		v.xtr = _xtr.data();
		v.ytr = _ytr.data();
		v.fl8 = _fl8.data();
		v.xpost = _xpost.data();
		v.sp8 = _sp8.data();
		v.po_id = _po_id.data();
		v.po_count = _po_count.data();
		v.tp_ptr = _tp_ptr.data();
		v.caught = _caught.data();
		v.ctl0 = _ctl.data();
		v.ctl = _ctl.data();
		v.ctl_next = _ctl.data() + 1;

		_grid_update = int( ( n + 255 ) / 256 );
		_upd_block = n >= UPDATE_LARGE_N ? UPDATE_BLOCK_LARGE : SPICE_UPDATE_BLOCK;
		_grid_upd = int( ( n + _upd_block - 1 ) / _upd_block );
		apply_launch( first );
	}

	// Eager plasticity state at a clock (re)start: initial traces (if asked), no flags or lists.
	void reset_eager( bool traces )
	{
		if( traces )
			for( auto * b : { &_xtr, &_ytr } )
			{
				if constexpr( factored )
					SPICE_LAUNCH( k_fill<<<unsigned( ( b->size() + 255 ) / 256 ), 256, 0, _s>>>( b->data(), std::int64_t( b->size() ), S::trace_init ) );
				else
					SPICE_HIP( hipMemsetAsync( b->data(), 0, b->bytes(), _s ) );
			}
		SPICE_HIP( hipMemsetAsync( _fl8.data(), 0, _fl8.bytes(), _s ) );
		if( windowed ) SPICE_HIP( hipMemsetAsync( _sp8.data(), 0, _sp8.bytes(), _s ) );
		SPICE_HIP( hipMemsetAsync( _po_count.data(), 0, _po_count.bytes(), _s ) );
	}

	// Lazy plasticity's bookkeeping, every row current through step `synced`.
	void alloc_lazy()
	{
		std::int64_t const n = _g.n;
		_last_spk.resize( n );
		_synced.resize( n );
		_pend.resize( n );
		_fl_synced.resize( 2 * n );
		_fl_pend.resize( 2 * n );
		_v.last_spk = _last_spk.data();
		_v.synced = _synced.data();
		_v.pend = _pend.data();
		_v.fl_synced = _fl_synced.data();
		_v.fl_pend = _fl_pend.data();
	}
	void reset_lazy( std::int32_t synced )
	{
		SPICE_HIP( hipMemsetAsync( _last_spk.data(), 0xff, _last_spk.bytes(), _s ) ); // -1
		SPICE_HIP( hipMemsetAsync( _pend.data(), 0, _pend.bytes(), _s ) );
		std::vector<std::int32_t> rows( _g.n, synced );
		SPICE_HIP( hipMemcpyAsync( _synced.data(), rows.data(), _synced.bytes(), hipMemcpyHostToDevice, _s ) );
		SPICE_HIP( hipStreamSynchronize( _s ) ); // `rows` is a host temporary
	}

	// The place (0 .. 3) of the current traces: that of the next window's number.
	std::int64_t trace_slot() const
	{
		ctl_t c{};
		SPICE_HIP( hipMemcpy( &c, _ctl.data() + ( _step & ( CLOCK_SLOTS - 1 ) ), sizeof( c ), hipMemcpyDeviceToHost ) );
		return c.wseq & 3;
	}

	// Factored trace attribute a of every synapse (synapses synchronized).
	void expand_trace( int a, float * out )
	{
		if constexpr( factored )
		{
			std::int64_t const at = trace_slot() * _g.n;
			SPICE_LAUNCH( k_expand_trace<Model><<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( _v, _xtr.data() + at, _ytr.data() + at, a, out ) );
			SPICE_HIP( hipStreamSynchronize( _s ) );
		}
	}

	// Imported attribute a of every synapse, in CSR order (synapses synchronized).
	void store_synapse_attr( int a, void const * in )
	{
		std::size_t const bytes = std::size_t( _g.nnz ) * attr_bytes<S>( a );
		if constexpr( factored )
			if( !_lazy && _g.nnz )
			{
				dbuf<char> tmp( bytes );
				SPICE_HIP( hipMemcpy( tmp.data(), in, bytes, hipMemcpyHostToDevice ) );
				unsigned const rows = unsigned( ( _g.n + 3 ) / 4 );
				dbuf<std::int32_t> bad( 1 );
				SPICE_HIP( hipMemsetAsync( bad.data(), 0, 4, _s ) );
				dbuf<float> t( std::size_t( _g.n ) );
				dbuf<float> & kept = a == S::pre_trace ? _xtr : _ytr;
				std::int64_t const at = trace_slot() * _g.n;
				if( is_factored_attr<S>( a ) )
				{
					SPICE_HIP( hipMemcpyAsync( t.data(), kept.data() + at, t.bytes(), hipMemcpyDeviceToDevice, _s ) );
					SPICE_LAUNCH( k_gather_trace<Model><<<rows, 256, 0, _s>>>( _v, a, reinterpret_cast<float const *>( tmp.data() ), t.data() ) );
				}
				SPICE_LAUNCH( k_check_factored<Model><<<rows, 256, 0, _s>>>( _v, a, tmp.data(), t.data(), bad.data() ) );
				std::int32_t b = 0;
				SPICE_HIP( hipMemcpyAsync( &b, bad.data(), 4, hipMemcpyDeviceToHost, _s ) );
				SPICE_HIP( hipStreamSynchronize( _s ) );
				if( b )
				{
					tmp.release();
					make_lazy();
				}
				else if( is_factored_attr<S>( a ) )
				{
					SPICE_HIP( hipMemcpy( kept.data() + at, t.data(), t.bytes(), hipMemcpyDeviceToDevice ) );
					return;
				}
			}
		if( bytes ) SPICE_HIP( hipMemcpy( _sa[a].data(), in, bytes, hipMemcpyHostToDevice ) );
	}

	// Nothing synchronized yet (plastic models).
	void reset_caught()
	{
		std::int64_t const none = -1;
		SPICE_HIP( hipMemcpyAsync( _caught.data(), &none, 8, hipMemcpyHostToDevice, _s ) );
		SPICE_HIP( hipStreamSynchronize( _s ) ); // `none` is a host temporary
		_caught_host = -1;
	}

	// By-target index of the plastic synapses: count per target, prefix sums, fill (after the
	// tiles and the rows' plastic flags are known).
	void build_by_target()
	{
		std::int64_t const n = _g.n;
		if( n > ( std::int64_t( 1 ) << 24 ) ) throw std::bad_alloc(); // (its segment table did not fit either)
		dbuf<std::uint32_t> cnt( n );
		SPICE_HIP( hipMemsetAsync( cnt.data(), 0, cnt.bytes(), _s ) ); // (tiles without inputs are not walked)
		SPICE_LAUNCH( ( k_tp_tile<Model, true><<<unsigned( _v.nact ), TP_BLOCK, 0, _s>>>( _v, cnt.data(), nullptr ) ) );
		SPICE_LAUNCH( k_tp_scan<<<1, 1024, 0, _s>>>( cnt.data(), _tp_ptr.data(), n ) );
		std::int64_t ends[2];
		SPICE_HIP( hipMemcpyAsync( ends, _tp_ptr.data() + n, 16, hipMemcpyDeviceToHost, _s ) );
		SPICE_HIP( hipStreamSynchronize( _s ) );
		_tp_total = ends[0];
		_tp_ent.resize( std::size_t( std::max<std::int64_t>( _tp_total, 1 ) ) );
		_v.tp_ent = _tp_ent.data();
		if( _tp_total > 0 ) SPICE_LAUNCH( ( k_tp_tile<Model, false><<<unsigned( _v.nact ), TP_BLOCK, 0, _s>>>( _v, nullptr, _tp_ent.data() ) ) );
		// targets with incoming plastic synapses (the mean in-degree sets the post-pass split)
		_tp_targets = ends[1];
		SPICE_HIP( hipStreamSynchronize( _s ) );
		apply_launch( _lc ); // the views, and the post pass's split
	}

	// Launch shapes (zero fields: the defaults). tile_w: targets per delivery tile (the
	// receive workgroup's LDS accumulators; see default_tile_w); flush_slots: target
	// slots per flush work item (one wave), so a flushed row of length L is split into about
	// L / flush_slots items; flush_grid: persistent flush workgroups (8 per CU by default).
	launch_cfg default_launch() const
	{
		int const cus = device_cu_count();
		std::int64_t const n = _g.n;
		launch_cfg c;
		c.tile_w = _lazy ? lazy_tile_w( n, cus ) : default_tile_w<Model>( n, _g.targets, _p.delay, cus );
		if( _p.batched && windowed && !plastic && _v.wcap == 1 ) c.tile_w = std::max( c.tile_w, BATCH_TILE );
		if constexpr( input_classes_v<Model> > 0 )
			if( _v.wcap == 1 && !_p.batched && _g.targets > 0 && double( _g.nnz ) / double( n ) * REC_TILE / double( _g.targets ) <= 18.0 )
				// Step by step, with segment records that fit: rather fewer and wider tiles, as all of
				// them reserve their spikes' places on one address, 9 ns apart (us per step of Vogels
				// nets of 22,361, 70,711 and 100,000 neurons: 6.6, 7.0 and 7.9 with a tile per CU, 5.8,
				// 6.6 and 7.4 with 768 targets; 4,000: 5.5 with 64, 5.75 with 768. Brunel, 100,000, whose
				// segments of 77 targets in such a tile have no records: 11.1 with 256, 11.4 with 768)
				c.tile_w = int( std::clamp<std::int64_t>( ( ( _g.targets + 95 ) / 96 + 63 ) / 64 * 64, c.tile_w, std::max( c.tile_w, REC_TILE ) ) );
		// plasticity beside a window's tiles: four workgroups of 256 threads per CU; work items of 128
		// slots or entries, which one round of a wave's loads holds twice over (STDP 1e8, delay 1:
		// 13.0 us per step, 16.2 with 256, 23.6 with 512), or of 512 where a window has items enough
		// for every wave anyway (1e9, delay 15, steps 2,000-12,000: 24.9, 25.3 with 256, 26.5 with 128;
		// brunel_with_plasticity 6e8: 13.1, 13.9 and 15.9)
		double const mean_row = n > 0 ? double( _g.nnz ) / double( n ) : 0.0;
		bool const win = windowed && !_lazy;
		c.flush_slots = !win ? 256 : _v.wcap > 1 && mean_row >= 5000.0 ? 512 : 128;
		std::int64_t const fparts = std::max( 1, int( mean_row / c.flush_slots + 0.5 ) );
		c.flush_grid = int( std::min<std::int64_t>( ( win ? 4 : 8 ) * cus, std::max<std::int64_t>( 1, ( n * fparts + 3 ) / 4 ) ) );
		c.recv_parts = 1;
		if( !plastic )
		{
			// window kernels: 16 waves where a workgroup has a CU to itself, 8 where several share one
			// or, step by step, the tile is small. us per step with 16 and 8 waves, Vogels 1e9 (delay 8,
			// 250 tiles of 896): 5.9, 9.0; brunel_3pop 1e9 (224 of 448): 2.8, 3.6, and 1e7 (248 of 128):
			// 1.2, 1.4; Brunel 1e10 (495 of 640): 18.7, 18.0; brunel_3pop 4e7 (313 of 64): 1.7, 1.2.
			// (workgroups of tiles without inputs come after the others: where those have a CU each and
			// are no small ones, 16 waves too -- Brunel, 400,000 neurons, 481 tiles of 832: 9.9, 14.5)
			std::int64_t const room = std::int64_t( cus ) * c.tile_w;
			bool const alone = c.tile_w >= 256 ? _g.targets <= room : n <= room;
			c.recv_block = c.tile_w > 2048 || ( alone && ( _v.wcap > 1 || c.tile_w >= 512 ) ) ? 1024 : 512;
		}
		else if( win )
			c.recv_block = 512; // (STDP 1e9: 24.3 us per step, 27.4 with 1,024 threads)
		else
			// small nets: few events per tile, so more and smaller delivery workgroups
			c.recv_block = n <= 65536 ? 256 : 1024;
		return c;
	}

	void apply_launch( launch_cfg c )
	{
		launch_cfg const d = default_launch();
		if( c.tile_w == 0 ) c.tile_w = d.tile_w;
		if( c.flush_slots == 0 ) c.flush_slots = d.flush_slots;
		if( c.flush_grid == 0 ) c.flush_grid = d.flush_grid;
		if( c.recv_block == 0 ) c.recv_block = d.recv_block;
		if( c.recv_parts == 0 ) c.recv_parts = d.recv_parts;
		if( c.recv_block != 256 && c.recv_block != 512 && c.recv_block != 1024 )
			throw std::invalid_argument( "recv_block must be 256, 512 or 1024" );
		if( c.recv_parts < 1 || c.recv_parts > 16 ) throw std::invalid_argument( "recv_parts must be in [1, 16]" );
		int const cus = device_cu_count();
		if( c.tile_w < 64 || c.tile_w > max_tile_w() || c.tile_w % 64 )
			throw std::invalid_argument( max_tile_w() > TILE_MAX ? "tile_w must be a multiple of 64 in [64, 8192]"
			                                                    : "tile_w must be a multiple of 64 in [64, 1024] (wider tiles: models without plasticity that run two kernels per step)" );
		if( c.flush_slots < 64 || c.flush_slots > ( 1 << 20 ) || c.flush_slots % 64 )
			throw std::invalid_argument( "flush_slots must be a multiple of 64 in [64, 2^20]" );
		if( c.flush_grid < 1 || c.flush_grid > 64 * cus ) throw std::invalid_argument( "flush_grid must be in [1, 64 x CUs]" );
		if( !_lc.tile_w )
		{
			shape( c ); // (a new network: nothing to go back to)
			return;
		}
		launch_cfg const before = _lc;
		try
		{
			shape( c );
		}
		catch( ... )
		{
			shape( before ); // (its buffers fitted)
			throw;
		}
	}

	// The buffers, views and windows of launch shapes c. If an allocation fails on the way the network
	// is not whole until a call succeeds, and is not stepped.
	void shape( launch_cfg const & c )
	{
		int const cus = device_cu_count();
		std::int64_t const n = _g.n;
		dview & v = _v;
		bool const retile = c.tile_w != v.tile_w || !( v.segs || v.offs );
		int const had_window = _window;
		_whole = false;
		if( retile )
		{
			std::int32_t const ntiles = std::int32_t( ( n + c.tile_w - 1 ) / c.tile_w );
			v.tile_w = c.tile_w;
			v.ntiles = ntiles;
			allocate_table();
			double const mean = double( _g.nnz ) / double( n ) * double( c.tile_w ) / double( std::max<std::int64_t>( _g.targets, 1 ) );
			bool const records = input_classes_v<Model> > 0 && _v.wcap == 1 && record_size( mean ) <= 6;
			if( !records && v.segs && ntiles <= PASS_TILES && !_col16.size() && wants_halves( mean ) && allocate_halves() )
			{
				std::uint32_t const d = std::uint32_t( c.tile_w ) / 64, magic = d == 1 ? 0u : std::uint32_t( ( ( std::uint64_t( 1 ) << 32 ) + d - 1 ) / d );
				SPICE_LAUNCH( k_segments_halves<<<unsigned( ( n + 3 ) / 4 ), 256, 16 * std::size_t( ntiles + 1 ), _s>>>( _v, _g.nnz, magic, _col16.data() ) );
			}
			else
				SPICE_LAUNCH( k_segments<<<unsigned( ( n + 3 ) / 4 ), 256, 0, _s>>>( _v ) );
			find_active_tiles(); // (synchronizes)
		}
		double const mean_row = n > 0 ? double( _g.nnz ) / double( n ) : 0.0;
		v.fparts = std::max( 1, int( mean_row / c.flush_slots + 0.5 ) );
		double const mean_in = _tp_targets > 0 ? double( _tp_total ) / double( _tp_targets ) : 0.0;
		v.pparts = std::max( 1, int( mean_in / c.flush_slots + 0.5 ) );
		v.rparts = c.recv_parts;
		_grid_flush = c.flush_grid;
		_grid_tiles = std::max( 1, std::min( v.nact * v.rparts, ( 16 * 1024 / c.recv_block ) * cus ) );
		_grid_plast = plastic ? std::max( 1, _grid_flush * 256 / c.recv_block ) : 0; // the same waves as flush_grid
		_lc = c;
		choose_window();
		if( retile || ( _window > 0 ) != ( had_window > 0 ) ) build_records();
		build_halves();
		// statistics slots: one per workgroup of the widest step kernel (receive: per work item;
		// plasticity: after those, one per plasticity workgroup or synchronization block; windows:
		// one per tile, then the passes' workgroups; update: per block)
		std::size_t const slots =
		    std::size_t( std::max( { _grid_update, _grid_upd, 2 * _grid_flush, 2 * _grid_tiles,
		                             v.ntiles * v.rparts + std::max( _grid_plast, _grid_flush ) } ) ) *
		    NSTAT;
		if( slots > _bstats.size() )
		{
			std::vector<unsigned long long> keep( NSTAT, 0ull );
			if( _bstats.size() )
			{
				std::vector<unsigned long long> b( _bstats.size() );
				SPICE_HIP( hipMemcpyAsync( b.data(), _bstats.data(), _bstats.bytes(), hipMemcpyDeviceToHost, _s ) );
				SPICE_HIP( hipStreamSynchronize( _s ) );
				for( std::size_t i = 0; i < b.size(); i++ ) keep[i % NSTAT] += b[i];
			}
			dbuf<unsigned long long> more( slots );
			SPICE_HIP( hipMemsetAsync( more.data(), 0, more.bytes(), _s ) );
			SPICE_HIP( hipMemcpyAsync( more.data(), keep.data(), NSTAT * 8, hipMemcpyHostToDevice, _s ) );
			SPICE_HIP( hipStreamSynchronize( _s ) ); // `keep` is a host temporary
			_bstats = std::move( more );
			v.bstats = _bstats.data();
		}
		for( int p = 0; p < CLOCK_SLOTS; p++ )
		{
			_vs[p] = _v;
			_vs[p].ctl = _ctl.data() + p;
			_vs[p].ctl_next = _ctl.data() + ( ( p + 1 ) & ( CLOCK_SLOTS - 1 ) );
			_vs[p].ctl_prev = _ctl.data() + ( ( p + CLOCK_SLOTS - 1 ) & ( CLOCK_SLOTS - 1 ) );
		}
		SPICE_HIP( hipStreamSynchronize( _s ) );
		_graphs.clear(); // the captured launches hold the old shapes
		_whole = true;
	}

	// Whether `bytes` of optional memory fit beside what this net still needs (rules.h).
	bool fits( std::uint64_t bytes ) const
	{
		if( bytes <= OPTIONAL_SMALL ) return true;
		std::size_t room = 0, all = 0;
		SPICE_HIP( hipMemGetInfo( &room, &all ) );
		return optional_fits( bytes, room, eager && !_lazy && !_tp_ent.size() ? 8 * std::uint64_t( _g.nnz ) : 0 );
	}

	// The segment table of the view's tiles, or offsets in its place (kernels.h, segment_of).
	void allocate_table()
	{
		_segs.release();
		_offs.release();
		_v.segs = nullptr;
		_v.offs = nullptr;
		std::uint64_t const entries = seg_entries( _g.n, _v.ntiles );
		if( _g.width < ( std::int64_t( 1 ) << 24 ) && ( _p.batched ? 8 * entries <= TABLE_BATCHED : fits( 8 * entries ) ) )
			try
			{
				_segs.resize( entries );
				_v.segs = _segs.data();
				return;
			}
			catch( std::bad_alloc const & )
			{
			}
		_offs.resize( std::size_t( _g.n ) * std::size_t( _v.ntiles + 1 ) );
		_v.offs = _offs.data();
	}

	// The delivery's tiles: those that some row has a target in (a population that no
	// connection targets gets no delivery workgroups); at least one, so that every step has a
	// delivery work item. Runs right after the segment table is built, before the views are copied.
	void find_active_tiles()
	{
		dview & v = _v;
		dbuf<std::uint8_t> flag( std::size_t( v.ntiles ) );
		SPICE_HIP( hipMemsetAsync( flag.data(), 0, flag.bytes(), _s ) );
		SPICE_LAUNCH( k_tile_active<<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( v, flag.data() ) );
		std::vector<std::uint8_t> f( std::size_t( v.ntiles ) );
		SPICE_HIP( hipMemcpyAsync( f.data(), flag.data(), f.size(), hipMemcpyDeviceToHost, _s ) );
		SPICE_HIP( hipStreamSynchronize( _s ) );
		std::vector<std::int32_t> ids;
		for( std::int32_t t = 0; t < v.ntiles; t++ )
			if( f[std::size_t( t )] ) ids.push_back( t );
		if( ids.empty() ) ids.push_back( 0 );
		v.nact = std::int32_t( ids.size() );
		for( std::int32_t t = 0; t < v.ntiles; t++ )
			if( !f[std::size_t( t )] && ( t != ids[0] || v.nact > 1 ) ) ids.push_back( t );
		_tile_ids.resize( ids.size() );
		SPICE_HIP( hipMemcpy( _tile_ids.data(), ids.data(), ids.size() * 4, hipMemcpyHostToDevice ) );
		v.tile_ids = _tile_ids.data();
	}

	// Window kernels (_window: their longest window, 0: none) run the steps of models whose
	// delivery may run before its targets' update in windows of up to the delay, as long as the
	// accumulators fit; other static models' step by step where one workgroup delivers a tile
	// (recv_parts = 1) of at most 4 workgroup widths.
	void choose_window()
	{
		_window = 0;
		{
			// lanes per segment: the power of two whose reads hold a segment two standard deviations
			// longer than the mean, so that few take a second round (Vogels 1e9, delay 8, 17.9
			// targets per segment: 8.9 us per step with 4 lanes, 7.5 with 8, 8.3 with 16)
			double const mean = _g.n > 0 ? double( _g.nnz ) / double( _g.n ) / _v.nact : 0.0;
			_v.wlanes = 0;
			while( _v.wlanes < 5 && double( WIN_VEC << _v.wlanes ) < mean + 2.0 * std::sqrt( mean ) ) _v.wlanes++;
		}
		if constexpr( windowed )
		{
			if( plastic && _lazy ) return;
			if( !plastic && !_ahead && ( _lc.recv_parts != 1 || _lc.tile_w > 4 * _lc.recv_block ) ) return;
			_window = 1;
			with_window_kernel( IDS32, [&]( auto, auto bytes, int ) {
				// the LDS of a CU, shared by the workgroups that a CU gets
				std::size_t const per_cu = std::size_t( std::clamp( ( _v.ntiles + device_cu_count() - 1 ) / device_cu_count(), 1, 3 ) );
				std::size_t const room = LDS_DYNAMIC / per_cu;
				int w = _v.wcap;
				while( w > 1 && bytes( w ) > room ) w = window_steps( w - 1 );
				_window = w;
			} );
			for( int form : { IDS32, IDS16, IDS16X8, RECORDS, IDS32_OFFSETS } )
				with_window_kernel( form, [&]( auto kernel, auto bytes, int ) { allow_lds( reinterpret_cast<void const *>( kernel ), bytes( _window ) ); } );
		}
	}

	// take(words, their number) of *count words of src (n of them without a count; n given at most),
	// by way of the pinned buffer: one small kernel and one wait in place of a copy of the count, a
	// wait, a copy of the words and another wait (a step of 4,000 neurons and its spikes: 47.6 us
	// with the copies, 22 without). false: nothing was done, as another thread has the buffer, or
	// there is none -- the second call gets it, as allocating it takes longer than a few copies.
	template <typename F>
	bool stage_to_host( void const * src, std::uint32_t const * count, std::uint32_t n, F && take )
	{
		if( !_stage )
		{
			if( ++_staged < 2 ) return false;
			_stage = host_stage::get();
			if( !_stage ) return false;
		}
		std::unique_lock<std::mutex> one( _stage->busy, std::try_to_lock );
		if( !one ) return false;
		SPICE_LAUNCH( k_stage<<<4, 1024, 0, _s>>>( static_cast<std::uint32_t const *>( src ), count, n, _stage->host ) );
		SPICE_HIP( hipStreamSynchronize( _s ) );
		take( _stage->host + 1, _stage->host[0] );
		return true;
	}

	// The low halves of the row store (window.h), for windows without records. us per step without
	// them, with 4 per lane and with 8, at this mean length of a segment: 2.6 (Vogels, 30,000
	// neurons, delay 2) 3.9, 4.1, 4.3; 6 (brunel_3pop 1e6) 0.86, 0.85, 0.93; 18 (Vogels 1e9, delay
	// 8) 5.8, 4.8, 5.3; 45 (brunel_3pop 1e9) 2.8, 2.5, 2.5; 50 (200,000 neurons) 3.4, 3.0, 3.2; 64
	// (Brunel 1e10) 17.2, 14.9, 12.5; beside weights, 26 (brunel_with_plasticity 6e8) 12.5, 11.6, 45
	// (brunel_3pop_stdp 1e9, steps 2,000 on) 24.9, 24.3. None if they took more than a fifth of the free memory; none for
	// the nets of a batch, whose kernel reads the row store.
	bool wants_halves( double mean ) const
	{
		return ( input_classes_v<Model> > 0 || ( plastic && windowed && !_lazy ) ) && !_p.batched && _g.nnz > 0 && mean >= 4.0;
	}
	bool allocate_halves()
	{
		std::size_t const n = std::size_t( _g.nnz ) + 8;
		if( !fits( 2 * n ) ) return false;
		try
		{
			_col16.resize( n );
		}
		catch( std::bad_alloc const & )
		{
			return false;
		}
		return true;
	}
	void build_halves()
	{
		_v.col16 = nullptr;
		double const mean = double( _g.nnz ) / double( _g.n ) / _v.nact;
		if( _window == 0 || _v.rec_lg || _v.offs || !wants_halves( mean ) )
		{
			_col16.release();
			return;
		}
		if( !_col16.size() )
		{
			if( !allocate_halves() ) return;
			SPICE_LAUNCH( k_halves<<<unsigned( std::min<std::size_t>( ( std::size_t( _g.nnz ) / 8 + 256 ) / 256, 256 * 32 ) ), 256, 0, _s>>>( _g.col.data(), _g.nnz, _col16.data() ) );
		}
		_v.col16 = _col16.data();
		_v.vec16 = !plastic && mean >= 56.0 ? 8 : 4;
		// (lanes per segment: see choose_window)
		_v.wlanes = 0;
		while( _v.wlanes < 5 && double( _v.vec16 << _v.wlanes ) < mean + ( mean < 20.0 ? 2.0 : 1.0 ) * std::sqrt( mean ) + ( _v.vec16 == 8 ? 4.0 : 0.0 ) ) _v.wlanes++;
	}

	// log2 of the smallest record that holds a segment 2.9 standard deviations longer than the mean
	// (8: none does)
	static int record_size( double mean )
	{
		int lg = 4;
		while( lg < 8 && rec_capacity( lg ) < mean + 2.9 * std::sqrt( mean ) ) lg++;
		return lg;
	}
	// Segment records (window.h) of networks that run step by step, where segments are short: 64 bytes
	// hold one (with 128, brunel_3pop of 90,000 neurons at p = 0.08 took 8.2 us per step instead of 9.2,
	// but 7.6 ms to build instead of 3.9). Not if the records took over twice the row store's memory, or more than a fifth of the free memory, or if over 1 %
	// of the segments did not fit (rows of very different lengths); not for the nets of a batch.
	void build_records()
	{
		_recs.release();
		_v.recs = nullptr;
		_v.rec_lg = 0;
		if constexpr( input_classes_v<Model> > 0 )
		{
			int const lg = record_size( double( _g.nnz ) / double( _g.n ) / _v.nact );
			std::uint64_t const segs = seg_entries( _g.n, _v.ntiles ), bytes = segs << lg;
			if( _v.wcap > 1 || _window == 0 || _p.batched || _v.offs || lg > 6 || _g.nnz == 0 || bytes > std::max<std::uint64_t>( 64 << 20, 8 * std::uint64_t( _g.nnz ) ) ) return;
			if( !fits( bytes ) ) return;
			try
			{
				_recs.resize( bytes );
			}
			catch( std::bad_alloc const & )
			{
				return;
			}
			dbuf<unsigned long long> longs( 1 );
			SPICE_HIP( hipMemsetAsync( longs.data(), 0, 8, _s ) );
			SPICE_LAUNCH( k_records<<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( _v, _recs.data(), lg, longs.data() ) );
			unsigned long long n = 0;
			SPICE_HIP( hipMemcpyAsync( &n, longs.data(), 8, hipMemcpyDeviceToHost, _s ) );
			SPICE_HIP( hipStreamSynchronize( _s ) );
			if( n > segs / 100 )
			{
				_recs.release();
				return;
			}
			_v.recs = _recs.data();
			_v.rec_lg = lg;
		}
	}

	void initialize()
	{
		SPICE_LAUNCH( k_init_neurons<Model><<<_grid_update, 256, 0, _s>>>( _v ) );
		if constexpr( plastic )
		{
			dbuf<std::int32_t> broken( 1 );
			SPICE_HIP( hipMemsetAsync( broken.data(), 0, 4, _s ) );
			SPICE_LAUNCH( k_init_synapses<Model><<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( _v, broken.data() ) );
			std::int32_t b = 0;
			SPICE_HIP( hipMemcpyAsync( &b, broken.data(), 4, hipMemcpyDeviceToHost, _s ) );
			SPICE_HIP( hipStreamSynchronize( _s ) );
			if( b )
				make_lazy();
			else if constexpr( eager )
				build_by_target();
		}
		SPICE_HIP( hipStreamSynchronize( _s ) );
	}

	// Enqueues steps t .. t + len - 1: windows of one step, or two kernels per step. The passes of
	// the last step of a plastic model are left to the next kernel (or a synchronization).
	void launch_steps( std::int64_t t, std::int64_t len )
	{
		for( std::int64_t k = 0; k < len; k++ )
			if( _window )
				launch_window( t + k, 1, nullptr, nullptr );
			else
				launch_step( t + k );
	}

	// Enqueues the kernels of step `t` (t mod 4 selects the clock slot): delivery (plastic
	// models: with step t - 1's plasticity work in the same kernel), then the neuron update.
	void launch_step( std::int64_t t )
	{
		[[maybe_unused]] dview const & v = _vs[t & ( CLOCK_SLOTS - 1 )];
		if constexpr( !plastic || !windowed || factored )
		{
			if( fixed() )
			{
				launch_receive<true>( v );
				launch_update<true>( v, nullptr, nullptr );
			}
			else
			{
				launch_receive<false>( v );
				launch_update<false>( v, nullptr, nullptr );
			}
		}
	}

	// run_profiled for two-kernel steps
	void run_profiled_steps( std::int64_t n, double * kernel_ms )
	{
		constexpr int batch = 128, ev_per_step = 4;
		synchronize(); // profiled steps run serially on the main stream
		std::vector<hipEvent_t> ev( batch * ev_per_step, nullptr );
		try
		{
			for( auto & e : ev ) SPICE_HIP( hipEventCreate( &e ) );
			for( std::int64_t done = 0; done < n; )
			{
				int const k = int( std::min<std::int64_t>( batch, n - done ) );
				for( int i = 0; i < k; i++ )
				{
					hipEvent_t * e = &ev[i * ev_per_step];
					if constexpr( !plastic || !windowed || factored )
					{
						if( fixed() )
							launch_step_events<true>( e, _vs[_step & ( CLOCK_SLOTS - 1 )] );
						else
							launch_step_events<false>( e, _vs[_step & ( CLOCK_SLOTS - 1 )] );
					}
					tick();
				}
				SPICE_HIP( hipStreamSynchronize( _s ) );
				for( int i = 0; i < k; i++ )
				{
					hipEvent_t * e = &ev[i * ev_per_step];
					for( int q = 0; q < 2; q++ ) // kernel_ms[2] stays 0: plasticity runs inside the delivery kernel
					{
						float ms = 0;
						SPICE_HIP( hipEventElapsedTime( &ms, e[2 * q], e[2 * q + 1] ) );
						kernel_ms[q] += ms;
					}
				}
				done += k;
			}
		}
		catch( ... )
		{
			for( auto & e : ev )
				if( e ) (void)hipEventDestroy( e );
			throw;
		}
		for( auto & e : ev ) (void)hipEventDestroy( e );
	}

	// the neuron update kernel of the two-kernel step (workgroups of _upd_block threads), with
	// HIP events attached to its dispatch when start is not null
	template <bool F>
	void launch_update( dview const & v, hipEvent_t start, hipEvent_t stop )
	{
		if( _upd_block == UPDATE_BLOCK_LARGE )
		{
			if( start )
				launch_timed( reinterpret_cast<void const *>( &k_update<Model, F, UPDATE_BLOCK_LARGE> ), unsigned( _grid_upd ), UPDATE_BLOCK_LARGE, start, stop, v );
			else
				SPICE_LAUNCH( ( k_update<Model, F, UPDATE_BLOCK_LARGE><<<_grid_upd, UPDATE_BLOCK_LARGE, 0, _s>>>( v ) ) );
		}
		else
		{
			if( start )
				launch_timed( reinterpret_cast<void const *>( &k_update<Model, F> ), unsigned( _grid_upd ), SPICE_UPDATE_BLOCK, start, stop, v );
			else
				SPICE_LAUNCH( ( k_update<Model, F><<<_grid_upd, SPICE_UPDATE_BLOCK, 0, _s>>>( v ) ) );
		}
	}

	// The window of w steps from step t, with HIP events attached to its dispatch when start is not
	// null. alone: the passes before it in a kernel of their own first.
	void launch_window( std::int64_t t, int w, hipEvent_t start, hipEvent_t stop, bool alone = false )
	{
		if constexpr( windowed )
		{
			if( alone ) launch_passes( t, _s );
			if( _slog_ctl.size() ) throw std::logic_error( "nets with a spike log are stepped by a batch" );
			dview v = _vs[t & ( CLOCK_SLOTS - 1 )];
			with_window_kernel( v.offs ? IDS32_OFFSETS : v.rec_lg ? RECORDS : !v.col16 ? IDS32 : v.vec16 == 8 ? IDS16X8 : IDS16, [&]( auto kernel, auto bytes, int bs ) {
				std::int32_t W = w;
				void * args[] = { &v, &W };
				void const * fn = reinterpret_cast<void const *>( kernel );
				if( start )
					SPICE_HIP( hipExtLaunchKernel( fn, dim3( unsigned( v.ntiles + ( alone ? 0 : _grid_plast ) ) ), dim3( unsigned( bs ) ), args, bytes( w ), _s, start, stop, 0 ) );
				else
					SPICE_HIP( hipLaunchKernel( fn, dim3( unsigned( v.ntiles + ( alone ? 0 : _grid_plast ) ) ), dim3( unsigned( bs ) ), args, bytes( w ), _s ) );
			} );
		}
	}

	// f(window kernel, its LDS bytes for w steps, workgroup size) of the launch shape
	template <typename F>
	void with_window_kernel( int form, F && f )
	{
		auto go = [&]( auto fx, auto b ) {
			constexpr bool FX = decltype( fx )::value;
			constexpr int BS = decltype( b )::value;
			constexpr bool cl = input_classes_v<Model> > 0;
			f( form == RECORDS ? &k_window<Model, FX, BS, cl ? RECORDS : IDS32> : form == IDS16 ? &k_window<Model, FX, BS, cl || plastic ? IDS16 : IDS32> : form == IDS16X8 ? &k_window<Model, FX, BS, cl ? IDS16X8 : IDS32> : form == IDS32_OFFSETS ? &k_window<Model, FX, BS, IDS32_OFFSETS> : &k_window<Model, FX, BS>,
			   [&]( int w ) { return window_lds<Model, FX>::bytes( BS, _lc.tile_w, w ); }, BS );
		};
		auto by_block = [&]( auto fx ) {
			int const bs = _lc.recv_block;
			bs == 256 ? go( fx, std::integral_constant<int, 256>{} ) : bs == 512 ? go( fx, std::integral_constant<int, 512>{} ) : go( fx, std::integral_constant<int, 1024>{} );
		};
		fixed() ? by_block( std::true_type{} ) : by_block( std::false_type{} );
	}

	// run_profiled for windows
	void run_profiled_windows( std::int64_t n, double * kernel_ms )
	{
		constexpr int batch = 128;
		synchronize(); // profiled steps run serially on the main stream
		std::vector<hipEvent_t> ev( 2 * batch, nullptr );
		try
		{
			for( auto & e : ev ) SPICE_HIP( hipEventCreate( &e ) );
			double first = 0.0, last = 0.0, sum = 0.0;
			std::int64_t windows = 0;
			while( n > 0 )
			{
				int k = 0;
				for( ; k < batch && n > 0; k++ )
				{
					bool const single = _step < _single_until;
					int const w = single ? 1 : window_steps( std::min<std::int64_t>( n, _window ) );
					launch_window( _step, w, ev[2 * k], ev[2 * k + 1], single );
					for( int i = 0; i < w; i++ ) tick();
					n -= w;
				}
				SPICE_HIP( hipStreamSynchronize( _s ) );
				for( int i = 0; i < k; i++ )
				{
					float ms = 0;
					SPICE_HIP( hipEventElapsedTime( &ms, ev[2 * i], ev[2 * i + 1] ) );
					if( windows++ == 0 ) first = ms;
					last = ms;
					sum += ms;
				}
			}
			bool const ends = plastic && windows >= 3;
			kernel_ms[0] += ends ? first : 0.0;
			kernel_ms[1] += ends ? last : 0.0;
			kernel_ms[2] += ends ? sum - first - last : sum;
		}
		catch( ... )
		{
			for( auto & e : ev )
				if( e ) (void)hipEventDestroy( e );
			throw;
		}
		for( auto & e : ev ) (void)hipEventDestroy( e );
	}

	// delivery workgroups, plus (plastic models) the previous step's plasticity workgroups
	template <bool F>
	void launch_receive( dview const & v )
	{
		launch_receive_events<F>( v, nullptr, nullptr );
	}

	// the delivery kernel at the launch shape's workgroup size and tile capacity (wide tiles:
	// static models only), with HIP events attached to its dispatch when start is not null
	template <bool F>
	void launch_receive_events( dview const & v, hipEvent_t start, hipEvent_t stop )
	{
		unsigned const grid = unsigned( _grid_tiles + _grid_plast );
		std::int32_t const tiles = _grid_tiles;
		auto go = [&]( auto bs, auto tm ) {
			constexpr int BS = decltype( bs )::value, TM = decltype( tm )::value;
			if( start )
				launch_timed( reinterpret_cast<void const *>( &k_receive_tiled<Model, F, BS, TM> ), grid, BS, start, stop, v, tiles );
			else
				SPICE_LAUNCH( ( k_receive_tiled<Model, F, BS, TM><<<grid, BS, 0, _s>>>( v, tiles ) ) );
		};
		auto by_block = [&]( auto tm ) {
			if( _lc.recv_block == 256 )
				go( std::integral_constant<int, 256>{}, tm );
			else if( _lc.recv_block == 512 )
				go( std::integral_constant<int, 512>{}, tm );
			else
				go( std::integral_constant<int, 1024>{}, tm );
		};
		if constexpr( !plastic )
			if( _lc.tile_w > TILE_MAX )
			{
				by_block( std::integral_constant<int, TILE_WIDE>{} );
				return;
			}
		by_block( std::integral_constant<int, TILE_MAX>{} );
	}

	// Launches `fn` on the net's stream with `start`/`stop` attached to the dispatch itself, so
	// that their elapsed time is the kernel's own duration (no launch gap, unlike events
	// recorded between launches). args: the kernel's exact parameter types.
	template <typename... A>
	void launch_timed( void const * fn, unsigned grid, unsigned block, hipEvent_t start, hipEvent_t stop, A... a )
	{
		void * args[] = { static_cast<void *>( &a )... };
		SPICE_HIP( hipExtLaunchKernel( fn, dim3( grid ), dim3( block ), args, 0, _s, start, stop, 0 ) );
	}

	// e[0], e[1] time the delivery kernel, e[2], e[3] the neuron update
	template <bool F>
	void launch_step_events( hipEvent_t * e, dview const & v )
	{
		launch_receive_events<F>( v, e[0], e[1] );
		launch_update<F>( v, e[2], e[3] );
	}

	// Before the counters are read or cleared: windows of different lengths leave different amounts of
	// plasticity due, and all of it counts to the steps before.
	void sync_counted()
	{
		if( windowed && !_lazy )
			sync_synapses();
		else
			synchronize();
	}

	// Brings all plastic synapses up to date through the last completed step.
	void sync_synapses()
	{
		synchronize();
		if constexpr( plastic )
		{
			if( _step > 0 && _caught_host != _step - 1 )
			{
				require_whole();
				// the last step's plasticity work, which the next delivery kernel would run, then
				// (eager) its events of the rows arriving next or (lazy) every row's replay up to it;
				// recorded in `caught` so the next delivery kernel skips the former
				std::int64_t const now = _step - 1;
				dview const & v = _vs[_step & ( CLOCK_SLOTS - 1 )]; // a view of step now + 1
				[[maybe_unused]] std::int64_t const slot0 = std::int64_t( v.ntiles ) * v.rparts;
				if( windowed && !_lazy )
					launch_passes( _step, _s );
				else if constexpr( traced && !windowed )
				{
					if( fixed() )
						SPICE_LAUNCH( k_stdp<Model, true><<<_grid_flush, 256, 0, _s>>>( v, now, slot0 ) );
					else
						SPICE_LAUNCH( k_stdp<Model, false><<<_grid_flush, 256, 0, _s>>>( v, now, slot0 ) );
					// deferred events of the rows arriving next
					SPICE_LAUNCH( k_sync_eager<Model><<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( _v, now ) );
				}
				else if constexpr( !traced )
				{
					if( fixed() )
						SPICE_LAUNCH( k_flush<Model, true><<<_grid_flush, 256, 0, _s>>>( v, now, slot0 ) );
					else
						SPICE_LAUNCH( k_flush<Model, false><<<_grid_flush, 256, 0, _s>>>( v, now, slot0 ) );
					// dt of the last completed step (the step that moved the clock to its state)
					SPICE_LAUNCH( k_sync_all<Model><<<unsigned( ( _g.n + 3 ) / 4 ), 256, 0, _s>>>( _v, std::int32_t( now ), _last_dt() ) );
				}
				SPICE_HIP( hipMemcpyAsync( _caught.data(), &now, 8, hipMemcpyHostToDevice, _s ) );
				SPICE_HIP( hipStreamSynchronize( _s ) ); // `now` is a host temporary
				_caught_host = now;
			}
		}
		synchronize();
	}

	// Compensated dt of step _step - 1 (the last enqueued step), as its kernels computed it
	// from the device clock; the nominal dt before any step (no replay needs it then).
	float _last_dt() const { return _step > 0 && _dt_last > 0.0f ? _dt_last : _p.dt; }
};
} // namespace spice::hipx
