#pragma once
// Device-side view of one network: plain pointers and sizes passed by value to every
// kernel. All step-dependent values (step index, Kahan clock, ring slot) are read from
// device memory (ctl), so the kernels of a step take identical arguments every step and a
// captured HIP graph can be replayed.
//
// HBM layout of one net:
//   row_ptr  int64[N+1], col int32[E]           CSR adjacency, rows sorted by target
//   na[a]    attribute a of every neuron          structure of arrays
//   acc[a]   receive accumulators of attribute a  [2][N] by step parity: fp32 / int64 (fixed
//                        point) / int32
//   sa[a]    attribute a of every synapse         CSR order (plastic models only)
//   ring     int32[rsize * N], counts uint32[rsize * COUNT_STRIDE] spike ids of the last steps (entry t mod
//                        rsize; rsize > D + 2 wcap (rules.h): a window of W <= wcap steps from T
//                        clears the entries of the wcap steps after it, while those of steps T - D
//                        and T - wcap - 1 may still be read; never-written entries are empty)
//   hring    uint64[HWORDS * N]  spike-history ring: bit (t mod H) of word (t mod H)/64 of
//                        neuron i set iff i spiked at step t (H = 256 steps, plastic models)
//   hasp     uint8[N]    row s has at least one plastic synapse
//   pl_lo/hi int32[N]    first / one-past-last plastic slot of row s (offsets in the row)
//   segs     uint64[N * ntiles]  per row and target tile: place in col and number of the row's targets
//                        in the tile, 8 tiles of a row side by side (kernels.h, seg_at); or
//   offs     uint32[N * (ntiles + 1)]  offsets of the tiles' first targets in the row
//   tile_ids int32[ntiles] the tiles: first the nact ones that some row has targets in (at least
//                        one), then the rest
// lazy plasticity (per-synapse contract):
//   last_spk int32[N]    latest spike step
//   synced   int32[N]    row s is up to date through this step
//   pend     int32[N]    row s has an undelivered pre event at synced+1
//   fl_*     int32[2][N] rows queued at this step (spike arrived, or history window full),
//                        with their (synced, pend) at that time; lists by step parity,
//                        counters [4] by step mod 4
// eager plasticity (neuron-trace synapses) with deferred events, all [2][N] by step parity:
//   xtr/ytr  f32[2][N]   neuron-local pre/post traces after step T
//   fl8      u8[2][N]    bit 0: spiked at T, bit 1: its spike arrives at T, bit 2: at T + 1
//   fl_id    int32[2][N] rows whose spike arrived at T and does not arrive at T + 1
//   po_id    int32[2][N] neurons that spiked at T and have incoming plastic synapses
// eager plasticity in windows (refractory endpoints), k = the window's number:
//   xtr/ytr  f32[4][N]   traces before the window's first step, by k mod 4
//   xpost    u32[2][N]   by k mod 2: what the post pass needs of a source in one gather
//   fl8      u8[2][N]    by k mod 2: 1 + the step of the window at which the neuron's spike
//                        arrived (0: none)
//   sp8      u8[2][N]    by k mod 2: 1 + the step of the window at which the neuron spiked
//   fl_id    int32[2][N] rows whose spike arrived in the window
//   po_id    int32[2][N] neurons that spiked in the window and have incoming plastic synapses
//                        (their counters by k mod 4)
// both:
//   tp_ptr   int64[N+1], tp_ent {src, place}[P]: the P plastic synapses by target
// both:
//   caught   int64       step whose plasticity work (and, eager, deferred events of the rows
//                        arriving next) a synchronization already did
//   slog_ids int32[cap]  spike log (served jobs): ids of steps t0 .. t0+nsteps-1, step by step
//   slog_off u64[nsteps] offset of step t0+k in slog_ids
#include <cstdint>

namespace spice::hipx
{
constexpr int MAXA = 16;

// Device clock. Four slots: the kernels of step T (the window from T on) read slot T & 3, and the
// window kernel or the neuron update writes the next one's, (T + W) & 3, so the clock advances
// without atomics or an extra kernel (a window's length is never a multiple of 4), the plasticity
// work of a two-kernel step, in the next delivery kernel, still reads its own slot (ctl_prev), and
// a captured graph of a multiple of 4 steps replays.
constexpr int CLOCK_SLOTS = 4;
struct ctl_t
{
	std::int64_t step; // index of the step being executed
	float sum;         // Kahan sum of dt over completed steps
	float c;           // Kahan compensation
	std::int32_t rslot; // spike ring entry of this step: step mod rsize
	// windows of plastic models: this window's number, and of the window before it (the one whose
	// plasticity passes are due) the steps (0: none) and the clock at its start
	std::int32_t wseq, wprev;
	float psum, pc;
};

// Device counters live in per-block slots: block b of any step kernel adds its block-reduced
// counts to bstats[b * NSTAT + k] with a plain read-add-write (no other block touches the
// slot, kernels of a stream never overlap), so no same-address atomics are needed. The host
// sums the slots when it reads statistics.
enum stat_index
{
	ST_SPIKES = 0,
	ST_EVENTS,
	ST_PLASTIC,
	ST_FLUSH_ROWS,
	ST_FLUSH_SYN,
	ST_FLUSH_SLOTS,
	ST_FLUSH_WRITTEN, // plastic synapses whose state the plasticity passes wrote back
	NSTAT = 8
};

// Spike log window of a net (device memory, set by the host between runs): steps
// t0 .. t0 + nsteps - 1 append their spike ids to the log, at most cap ids in all.
struct slog_t
{
	std::int64_t t0;
	std::int64_t nsteps;
	std::uint64_t cap;
};

// One plastic synapse of the by-target index: its source row (the upper 24 bits: a plastic network of
// 2^24 neurons would need 2 TB for its segment table) and its place among the synapses (40 bits).
using tp_entry = std::uint64_t;
constexpr std::uint32_t X_ARRIVED = 0xffffffffu; // (a NaN that no arithmetic gives)

// The spike counters of successive steps lie this many words apart: all tiles reserve their places
// of all of a window's steps at about the same time, and atomics on one line wait for each other, 9
// ns each (us per step with the counters side by side and apart: Vogels 1e9, delay 8, 250 tiles: 7.5
// and 5.8; Brunel 1e10, 495 tiles: 18.0 and 17.2; brunel_with_plasticity 6e8: 13.1 and 12.5).
constexpr int COUNT_STRIDE = 64;

struct dview
{
	std::int32_t N, D, width, shift;
	float DT;
	std::int32_t fparts; // work items per flushed row
	std::int32_t pparts; // work items per spiking target (eager plasticity)
	std::int32_t rparts; // delivery workgroups per tile (the step's spike list split between them)
	std::int32_t rsize;     // entries of the spike ring
	std::int32_t wcap;      // longest window of steps run by one kernel
	std::int32_t wlanes;    // windows: log2 of the lanes that walk a row segment
	std::uint32_t flags;
	std::uint64_t seed;
	float param[4]; // per-net model parameters (snn_info::param)

	std::int64_t const * row_ptr;
	std::int32_t const * col;

	void * na[MAXA];
	void * acc[MAXA];
	void * sa[MAXA];

	std::int32_t * ring;
	std::uint32_t * counts;

	unsigned long long * hring; // [HWORDS][N] spike-history ring
	std::int32_t * last_spk;    // [N] latest spike step (-1: none)
	std::int32_t * synced;
	std::int32_t * pend;
	std::uint8_t * hasp;
	std::int32_t * pl_lo; // plastic slots of row r lie in [row_ptr[r] + pl_lo[r], row_ptr[r] + pl_hi[r])
	std::int32_t * pl_hi;
	std::int32_t * fl_id;
	std::int32_t * fl_synced;
	std::int32_t * fl_pend;
	std::uint32_t * fl_count; // [4]
	float * xtr;
	float * ytr;
	std::uint32_t * xpost; // windows: [2][N] pre trace at the window's start, X_ARRIVED if the spike arrived in it
	std::uint8_t * fl8;
	std::uint8_t * sp8;
	std::int32_t * po_id;
	std::uint32_t * po_count; // [4]
	std::int64_t const * tp_ptr;
	tp_entry const * tp_ent;
	std::int64_t * caught;

	ctl_t * ctl0;     // the clock slots
	ctl_t * ctl;      // this step's clock
	ctl_t * ctl_next; // the next step's clock (written by k_update)
	ctl_t * ctl_prev; // the previous step's clock (its dt for the lazy flush of that step)
	unsigned long long * bstats; // [nblocks_max * NSTAT]

	std::uint64_t * segs; // the segment table: where row r's targets in tile t are (kernels.h, segment_of)
	std::uint32_t * offs; // in its place if it is nullptr: offsets in the row
	std::int32_t ntiles, tile_w;
	std::int32_t * tile_ids; // [ntiles]: the tiles with incoming synapses (the delivery's), then the others
	std::int32_t nact;

	// segment records (window.h): per row and tile 2^rec_lg bytes, the
	// segment's length and targets in 16 bits (0: none built, the segments are read from col)
	unsigned char const * recs;
	std::int32_t rec_lg;

	std::uint16_t const * col16; // the low halves of col (window.h); nullptr: none
	std::int32_t vec16;          // of them per lane: 4 or 8

	slog_t * slog; // nullptr: no spike log
	std::int32_t * slog_ids;
	std::uint64_t * slog_off;
};
} // namespace spice::hipx
