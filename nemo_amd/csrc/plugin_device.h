/*
 * Device helpers shared by the neuron-model plugin kernels.
 *
 * An update kernel runs one block of NEMO_TILE threads per tile of its neuron
 * type, one neuron per thread, and every thread of a block calls
 *   UpdateLds& L = update_lds<CO>();            (CO: the launch carries propagate blocks)
 *   if(!CO && b.direct.ring && direct_block(b, g, L)) return;
 *   h = load_history(b, ng, valid);
 *   gather_input(b, g, L);                      (block barriers inside)
 * or, in a launch of NEMO_COLAUNCH_BLOCK-thread blocks whose tile blocks keep
 * their other waves (colaunched_block<true>), those waves help to gather:
 *   if(!gather_input<NEMO_COLAUNCH_BLOCK>(b, g, L)) return;
 *   take_current(b, L.input, ng, E, I);         (valid threads)
 *   record_firing<CO>(b, L, ng, valid, fired, h); (every thread; pushes the delay-1 events when asked)
 *   stdp_tile(b, L, ng, valid, h);              (every thread; barriers inside)
 */
#ifndef NEMO_AMD_PLUGIN_DEVICE_H
#define NEMO_AMD_PLUGIN_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nemo_hip_plugin.h"
#include "glibc_math.h"

#define NEMO_UPDATE_BLOCK NEMO_TILE
/* Launch bounds of an update kernel, compiled with CO true for launches that
 * carry propagate blocks and false otherwise. */
#define NEMO_UPDATE_BOUNDS(CO) \
	__launch_bounds__((CO) ? NEMO_COLAUNCH_BLOCK : NEMO_UPDATE_BLOCK, (CO) ? NEMO_COLAUNCH_WAVES : 1)

namespace nemo_dev {

/* The step base.  No kernel that calls this changes the clock, so it is read
 * as a constant: once per wave, where an ordinary load would be repeated
 * after every store, each time in the launch's chain of dependent phases. */
__device__ inline uint64_t clock_base(const nemo_hip_clock* clock)
{
	typedef const __attribute__((address_space(4))) nemo_hip_clock* constant_clock;
	return reinterpret_cast<constant_clock>(reinterpret_cast<uintptr_t>(clock))->base_step;
}

__device__ inline uint64_t current_step(const nemo_hip_step_buffers& b)
{
	return clock_base(b.clock) + b.step_offset;
}

/* Inclusive sum over the lanes of a wave, all of them active: within rows of
 * 16 by DPP shifts, then each row's last lane broadcast into the rows after
 * it (row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3).  Six
 * additions, where shuffles take six round trips of the LDS crossbar. */
__device__ inline uint32_t wave_inclusive_sum(uint32_t x)
{
	int v = int(x);
	v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
	v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
	return uint32_t(v);
}

/* Room for x entries per lane in a list that the block's waves fill in
 * whatever order they come: *counter (LDS) grows by the wave's total, the
 * lane's entries start where returned.  Every lane of the wave calls it. */
__device__ inline uint32_t wave_append(uint32_t* counter, uint32_t x)
{
	const uint32_t upto = wave_inclusive_sum(x);
	const uint32_t all = uint32_t(__builtin_amdgcn_readlane(int(upto), 63));
	uint32_t base = 0;
	if(all) {
		if((threadIdx.x & 63) == 0) base = atomicAdd(counter, all);
		base = uint32_t(__builtin_amdgcn_readfirstlane(int(base)));
	}
	return base + upto - x;
}

/* Exclusive scan of one value per thread over a block of THREADS threads;
 * returns the thread's prefix and sets *total. */
template<unsigned THREADS = NEMO_TILE>
__device__ inline uint32_t block_exclusive_scan(uint32_t x, uint32_t* total)
{
	__shared__ uint32_t s_wave[THREADS / 64];
	const unsigned lane = threadIdx.x & 63;
	const unsigned wave = threadIdx.x >> 6;
	const uint32_t v = wave_inclusive_sum(x);
	if(lane == 63) s_wave[wave] = v;
	__syncthreads();
	uint32_t before = 0, all = 0;
#pragma unroll
	for(unsigned w = 0; w < THREADS / 64; ++w) {
		const uint32_t t = s_wave[w];
		before += w < wave ? t : 0;
		all += t;
	}
	__syncthreads();
	*total = all;
	return before + v - x;
}

/* For each of K items x, the largest i < n with arr[i] <= x, for a
 * non-decreasing arr with arr[0] <= x and 1 <= n <= MAXN (a power of two): a
 * fixed number of steps, in lock-step, so that the K LDS reads of a step are
 * in flight together. */
template<unsigned MAXN, int K>
__device__ inline void last_not_above_k(const uint32_t* arr, unsigned n, const uint32_t (&x)[K], unsigned (&lo)[K])
{
#pragma unroll
	for(int u = 0; u < K; ++u) lo[u] = 0;
#pragma unroll
	for(unsigned step = MAXN / 2; step >= 1; step >>= 1) {
		uint32_t v[K];
#pragma unroll
		for(int u = 0; u < K; ++u) {
			const unsigned probe = lo[u] + step;
			v[u] = arr[probe < n ? probe : n - 1];
		}
#pragma unroll
		for(int u = 0; u < K; ++u) {
			const unsigned probe = lo[u] + step;
			lo[u] = (probe < n && v[u] <= x[u]) ? probe : lo[u];
		}
	}
}

/* Synaptic input of one tile for the current step. */
struct TileInput {
	long long E[NEMO_TILE];
	long long I[NEMO_TILE];
};

/* Columns of the bin table a group of lanes gathers at a time, an event per
 * lane each in flight. */
constexpr int GATHER_ILP = 4;

/* Pieces (of up to 64 events) of fired rows that a block delivering directly
 * lists in LDS at a time. */
constexpr unsigned DIRECT_CHUNKS = 256;

/* The LDS an update block uses: its tile's input sums, the lists of direct
 * delivery, and the per-tile STDP lists.  A kernel takes it
 * from update_lds<DYNAMIC>(): a static array, or -- in launches that also run
 * propagate blocks -- the start of the launch's dynamic LDS, which those
 * blocks use for their own purposes, so that a block of either kind needs
 * only the larger of the two. */
struct UpdateLds {
	TileInput input;
	uint2 chunk[DIRECT_CHUNKS]; /* direct delivery: pieces of the fired rows, events per delay, pieces listed */
	uint32_t count[64];
	uint32_t chunks;
	int32_t fn[128];
	uint32_t rb[NEMO_TILE];
	uint32_t pos[NEMO_TILE + 1];
	uint2 push_rows[NEMO_TILE]; /* the tile's rows to push, read ahead */
};

template<bool DYNAMIC>
__device__ inline UpdateLds& update_lds()
{
	if constexpr(DYNAMIC) {
		extern __shared__ uint64_t nemo_update_lds_dyn[];
		return *reinterpret_cast<UpdateLds*>(nemo_update_lds_dyn);
	} else {
		__shared__ UpdateLds lds;
		return lds;
	}
}

struct Nothing {
	__device__ void operator()() const {}
};

/* The delay-1 row of device index ng when the launch pushes (co.push, or
 * direct delivery), for L.push_rows[threadIdx.x]: gather_input reads it
 * ahead; a kernel that records firing without gathering calls begin_push. */
__device__ inline uint2 push_row(const nemo_hip_step_buffers& b, unsigned ng)
{
	return b.direct.ring ? b.direct.first_rows[ng] : b.co.push ? b.co.push_rows[ng] : make_uint2(0, 0);
}

__device__ inline void begin_push(const nemo_hip_step_buffers& b, UpdateLds& L, unsigned ng)
{
	L.push_rows[threadIdx.x] = push_row(b, ng);
	if(threadIdx.x < 64) L.count[threadIdx.x] = 0;
	if(threadIdx.x == 64) L.chunks = 0;
	__syncthreads();
}

/* The step's slot of the ring of a directly delivered network: the tile's
 * sums are there already.  One round trip, where the binned gather takes
 * three (table row, bins, sums).  The neuron's state (prefetch) is requested
 * first, which needs no clock; the tile's event counter is touched last and
 * without waiting for it. */
template<typename Prefetch, typename Meanwhile>
__device__ inline void gather_direct(const nemo_hip_step_buffers& b, UpdateLds& L, unsigned tile, Prefetch prefetch,
		Meanwhile meanwhile)
{
	const nemo_hip_direct& r = b.direct;
	const unsigned tid = threadIdx.x;
	const unsigned ng = tile * NEMO_TILE + tid;
	/* every argument the launch uses, loaded in one go: where each is used,
	 * a cold line of the argument block at a time, they cost the chain a
	 * round trip of the scalar cache each */
	asm volatile("" ::"s"(r.ring), "s"(r.first_rows), "s"(r.fcm), "s"(r.delay), "s"(r.arrivals), "s"(r.events),
			"s"(r.mask), "s"(r.tiles), "s"(b.acc_pitch), "s"(b.hist), "s"(b.hist_pitch), "s"(b.fired_bits),
			"s"(b.fired_words), "s"(b.fbits), "s"(b.ext_current), "s"(b.fstim), "s"(b.debug_current),
			"s"(b.stdp.rcm_ptr), "s"(clock_base(b.clock)));
	const uint2 prow = push_row(b, ng);
	prefetch();
	const uint32_t slot = uint32_t(current_step(b)) & r.mask;
	int64_t* acc = r.ring + size_t(slot) * 2 * b.acc_pitch;
	const int64_t oe = acc[ng];
	const int64_t oi = acc[b.acc_pitch + ng];
	uint32_t* arrived = r.arrivals + size_t(slot) * r.tiles + tile;
	const uint32_t n = tid == 0 ? *arrived : 0;
	if(tid < 64) L.count[tid] = 0;
	if(tid == 64) L.chunks = 0;
	meanwhile();
	L.input.E[tid] = oe;
	L.input.I[tid] = oi;
	L.push_rows[tid] = prow;
	if(oe) acc[ng] = 0;
	if(oi) acc[b.acc_pitch + ng] = 0;
	if(n) {
		*arrived = 0;
		atomicAdd(&r.events[ng >> 6], (unsigned long long)n);
	}
	__syncthreads(); /* count and chunks, for record_firing */
}

/* Sum the tile's input of this step into LDS: the overflow accumulators of
 * its neurons (cleared here, cpu/Simulation.cpp:279-288) and the binned events
 * of every delivery column (integer sums, so the order of the 64-bit LDS
 * atomics does not matter).  The whole table row is read (or, bin_ranged, the
 * tile's two ranges of it): columns whose window does not hold the tile keep
 * a zero count, and reading them costs less than a dependent load of the
 * tile's column range.
 *
 * A group of lanes takes a column: its entry, then its events, a lane each,
 * four columns in flight per group.  Two round trips and no barrier between
 * them, where one event per thread needs the columns' prefix (a block scan)
 * and a search for each event's column.  The lanes per group are what a block
 * has for two rounds of four columns: 16 at 100k neurons x 1000 synapses (245
 * columns of about 8 of the tile's events).  Measured (us a step, graphs, scan
 * and search before): 100k x 1000 17.06 -> 16.14 without STDP, 19.7 -> 19.3
 * with it, a batch of 32 networks 19.1 -> 17.9; one round of six columns 16.5
 * and 19.3, of eight spills (72 VGPRs) and gains nothing.
 *
 * prefetch() is called once the row's entries and the accumulators are
 * requested: the loads it issues (the model's state, say) queue behind them,
 * so that waiting for the entries does not wait for them too.  meanwhile()
 * runs in the tile's own threads, all of them, while the ring's slot is on
 * its way (direct delivery) or the block's other waves still sum events: work
 * on what prefetch loaded that needs no input, such as a neuron's noise.
 *
 * THREADS threads of the block take part: the tile's NEMO_TILE (one per
 * neuron, which alone read the accumulators and, through prefetch, their
 * neuron's state) and, in a block of NEMO_COLAUNCH_BLOCK threads, helpers that
 * only load and sum events.  Returns false for the helpers, which take no
 * further part in the step. */
template<unsigned THREADS = NEMO_TILE, typename Prefetch = Nothing, typename Meanwhile = Nothing>
__device__ inline bool gather_input(const nemo_hip_step_buffers& b, const nemo_hip_neuron_group& g, UpdateLds& L,
		Prefetch prefetch = Prefetch(), Meanwhile meanwhile = Meanwhile())
{
	static_assert(THREADS % 64 == 0 && THREADS >= NEMO_TILE, "whole waves beyond the tile");
	TileInput& in = L.input;
	const unsigned tid = threadIdx.x;
	const bool lead = THREADS == NEMO_TILE || tid < NEMO_TILE; /* uniform per wave */
	const unsigned tile = g.start / NEMO_TILE + blockIdx.x;
	if constexpr(THREADS == NEMO_TILE) {
		/* a launch that carries propagate blocks is never direct */
		if(b.direct.ring) {
			gather_direct(b, L, tile, prefetch, meanwhile);
			return true;
		}
	}
	const size_t parity = current_step(b) & 1;
	int64_t* acc = b.acc + parity * 2 * b.acc_pitch;
	const unsigned ng = tile * NEMO_TILE + tid;
	const unsigned BB = b.bin_blocks;
	const char* row = reinterpret_cast<const char*>(b.bin_table + (parity * b.tiles + tile) * BB);
	const uint32_t cap = b.bin_capacity;
	const char* bins = reinterpret_cast<const char*>(b.bins + parity * BB * size_t(cap));
	/* the columns read: the whole row, or (bin_ranged) the tile's two ranges,
	 * column first0 + i for i < n0, then first1 + i - n0 */
	const unsigned BR = b.bin_first_set ? b.bin_first_set : BB; /* columns holding events */
	unsigned B = BR, first0 = 0, n0 = BR, first1 = 0;
	if(b.bin_ranged) {
		const uint32_t r0 = b.bin_range[tile], r1 = b.bin_range[b.tiles + tile];
		first0 = r0 & 0xffffu;
		n0 = (r0 >> 16) - first0;
		first1 = r1 & 0xffffu;
		B = n0 + (b.bin_first_set ? 0u : (r1 >> 16) - first1);
	}
	/* groups of 1 << shift lanes take a column each, as many lanes as two
	 * rounds of GATHER_ILP columns per group leave them */
	constexpr int ILP = GATHER_ILP;
	unsigned shift = 6;
	while(shift > 2 && (B << shift) > 2 * ILP * THREADS) --shift;
	const unsigned lanes = 1u << shift, lane = tid & (lanes - 1);
	const unsigned groups = THREADS >> shift, group = tid >> shift;
	uint32_t ent[ILP]; /* count << 16 | offset */
	auto column = [&](unsigned i) { return i < n0 ? first0 + i : first1 + (i - n0); };
	auto read_row = [&](unsigned c0) {
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			const unsigned i = c0 + u * groups + group;
			ent[u] = i < B ? *reinterpret_cast<const uint32_t*>(row + column(i) * uint32_t(sizeof(uint32_t))) : 0u;
		}
	};
	read_row(0);
	int64_t oe = 0, oi = 0;
	if(lead) {
		oe = acc[ng];
		oi = acc[b.acc_pitch + ng];
		const uint2 prow = push_row(b, ng);
		prefetch();
		in.E[tid] = 0;
		in.I[tid] = 0;
		L.push_rows[tid] = prow;
	}
	__syncthreads(); /* the sums are cleared; the loads stay on their way */
	for(unsigned c0 = 0; c0 < B; c0 += ILP * groups) {
		if(c0) read_row(c0);
		uint32_t at[ILP]; /* byte offset of the lane's next event: below 2^28 */
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			at[u] = (column(c0 + u * groups + group) * cap + (ent[u] & 0xffffu) + lane) * uint32_t(sizeof(int2));
			ent[u] >>= 16;
		}
		/* events lane, lane + lanes, ... of every column: one round while no
		 * column holds more events than its group has lanes */
		bool more = true;
		for(uint32_t e = lane; __any(more); e += lanes) {
			int2 ev[ILP];
			more = false;
#pragma unroll
			for(int u = 0; u < ILP; ++u) {
				ev[u] = make_int2(-1, 0);
				if(e < ent[u]) ev[u] = *reinterpret_cast<const int2*>(bins + at[u]);
				at[u] += lanes * uint32_t(sizeof(int2));
				more = more || e - lane + lanes < ent[u];
			}
#pragma unroll
			for(int u = 0; u < ILP; ++u) {
				if(ev[u].x >= 0) {
					long long* dst = ev[u].y >= 0 ? &in.E[ev[u].x] : &in.I[ev[u].x];
					atomicAdd(reinterpret_cast<unsigned long long*>(dst), (unsigned long long)(long long)ev[u].y);
				}
			}
		}
	}
	if(lead) {
		if(oe) acc[ng] = 0;
		if(oi) acc[b.acc_pitch + ng] = 0;
		meanwhile();
	}
	__syncthreads();
	if(lead) {
		in.E[tid] += oe;
		in.I[tid] += oi;
	}
	return lead;
}

/* Saturate a 64-bit fixed-point sum to the int32 range and convert to float,
 * as NeMo's wfx_toFloat (src/nemo/fixedpoint.cpp:40-49). */
__device__ inline float wfx_to_float(int64_t v, unsigned fbits)
{
	v = v > int64_t(INT32_MAX) ? int64_t(INT32_MAX) : v;
	v = v < int64_t(INT32_MIN) ? int64_t(INT32_MIN) : v;
	/* the product with the power of two is the quotient, exactly */
	return float(int32_t(v)) * __uint_as_float((127u - fbits) << 23);
}

/* Excitatory and inhibitory current of neuron ng (thread threadIdx.x of the
 * tile), as gathered by gather_input. */
__device__ inline void take_current(const nemo_hip_step_buffers& b, const TileInput& in, unsigned ng, float& E, float& I)
{
	E = wfx_to_float(in.E[threadIdx.x], b.fbits);
	I = wfx_to_float(in.I[threadIdx.x], b.fbits);
	if(b.debug_current) {
		b.debug_current[ng] = E;
		b.debug_current[b.acc_pitch + ng] = I;
	}
}

/* User current for this step, cleared after use (Izhikevich.cpp:61-64). */
__device__ inline float take_external(const nemo_hip_step_buffers& b, unsigned ng)
{
	if(!b.ext_current) return 0.0f;
	float v = b.ext_current[ng];
	b.ext_current[ng] = 0.0f;
	return v;
}

__device__ inline bool stimulated(const nemo_hip_step_buffers& b, unsigned ng)
{
	return b.fstim && ((b.fstim[ng >> 5] >> (ng & 31)) & 1u);
}

/* Marsaglia xorshift128 (src/nemo/RNG.cpp:9-19) */
__device__ inline uint32_t urand(uint4& s)
{
	uint32_t t = s.x ^ (s.x << 11);
	s.x = s.y;
	s.y = s.z;
	s.z = s.w;
	s.w = (s.w ^ (s.w >> 19)) ^ (t ^ (t >> 8));
	return s.w;
}

/* Box-Muller, sine branch only, bit-exact with glibc (src/nemo/RNG.cpp:25-33) */
__device__ inline float nrand(uint4& s)
{
	float a = float(urand(s)) * 1.4629180792671596810513378043098e-9f;
	float b = float(urand(s)) * 0.00000000023283064365386962890625f;
	float r = __builtin_sqrtf(-2.0f * nemo_math::logf_exact(1.0f - b));
	return nemo_math::sinf_exact(a) * r;
}

/* The same for every lane of a wave at once, all of them active, without a
 * branch or a load: lane i holds entry i % 16 of logf's tables (noise_table,
 * loaded ahead with the neuron's state), which the lanes look up by shuffle.
 * As a chain of branches over both routes of sinf and logf's special cases,
 * with the table in memory, the deviate took 0.9 us of a step's launch. */
struct NoiseTable {
	double invc, logc;
};

__device__ inline NoiseTable noise_table()
{
	NoiseTable t;
	t.invc = nemo_math::logf_invc(threadIdx.x & 15);
	t.logc = nemo_math::logf_logc(threadIdx.x & 15);
	return t;
}

__device__ inline float nrand_wave(uint4& s, const NoiseTable& t)
{
	const float a = float(urand(s)) * 1.4629180792671596810513378043098e-9f;
	const float b = float(urand(s)) * 0.00000000023283064365386962890625f;
	const float l = nemo_math::logf_unit(1.0f - b, [&t](unsigned i, double* invc, double* logc) {
		*invc = __shfl(t.invc, int(i));
		*logc = __shfl(t.logc, int(i));
	});
	return nemo_math::sinf_turn(a) * __builtin_sqrtf(-2.0f * l);
}

/* Write the tile's words of the step's firing bitmap (one ballot per wave;
 * device indices of a wave are 64-aligned). */
__device__ inline void store_firing(const nemo_hip_step_buffers& b, unsigned ng, bool valid, bool fired)
{
	const uint64_t mask = __ballot(valid && fired);
	if((threadIdx.x & 63) == 0) {
		const uint64_t slot = current_step(b) & (NEMO_STEP_RING - 1);
		b.fired_bits[slot * b.fired_words + (ng >> 6)] = mask;
	}
}

/* History of neuron ng before this step (after the previous one). */
__device__ inline uint64_t load_history(const nemo_hip_step_buffers& b, unsigned ng, bool valid)
{
	return valid ? b.hist[NEMO_HIST_INDEX(ng, current_step(b) - 1, b.hist_pitch)] : 0;
}

/* Delay-1 delivery of this step's firing for the next step, straight into
 * that step's overflow accumulators (nemo_hip_colaunch.push), as the delay-1
 * part of cpu::Simulation::deliverSpikes (src/nemo/cpu/Simulation.cpp:
 * 259-308).  Each wave spreads the delay-1 rows of its fired neurons (read
 * ahead into L.push_rows by gather_input) over its lanes, PUSH_ILP loads in
 * flight per lane before their 64-bit atomics; the sums are integer, so
 * their order does not matter.  Every thread of the wave calls it. */
constexpr int PUSH_ILP = 4;
__device__ inline void push_delay1(const nemo_hip_step_buffers& b, const UpdateLds& L, unsigned ng, bool valid,
		bool fired)
{
	const nemo_propagate_args& a = b.co.args;
	const bool f = valid && fired;
	if(!__any(f)) return;
	const unsigned lane = threadIdx.x & 63;
	uint32_t rb = 0, len = 0;
	if(f) {
		const uint2 r = L.push_rows[threadIdx.x];
		rb = r.x;
		len = r.y - r.x;
	}
	const uint32_t incl = wave_inclusive_sum(len);
	const uint32_t total = uint32_t(__builtin_amdgcn_readlane(int(incl), 63));
	const uint32_t excl = incl - len;
	int64_t* acc = a.acc + ((current_step(b) + 1) & 1) * 2 * a.acc_pitch;
	for(uint32_t e0 = 0; e0 < total; e0 += 64 * PUSH_ILP) {
		int2 ev[PUSH_ILP];
#pragma unroll
		for(int u = 0; u < PUSH_ILP; ++u) {
			const uint32_t e = e0 + u * 64 + lane;
			/* the lane whose row holds event e: the first whose inclusive
			 * prefix exceeds e (the prefix is non-decreasing over lanes) */
			unsigned s = 0;
#pragma unroll
			for(unsigned step = 32; step >= 1; step >>= 1) {
				if(__shfl(incl, int(s + step - 1)) <= e) s += step;
			}
			const uint32_t srb = __shfl(rb, int(s));
			const uint32_t sex = __shfl(excl, int(s));
			ev[u] = make_int2(0, 0);
			if(e < total) ev[u] = a.fcm[srb + (e - sex)];
		}
#pragma unroll
		for(int u = 0; u < PUSH_ILP; ++u) {
			if(e0 + u * 64 + lane < total) {
				int64_t* dst = acc + (ev[u].y >= 0 ? size_t(0) : a.acc_pitch) + uint32_t(ev[u].x);
				atomicAdd(reinterpret_cast<unsigned long long*>(dst), (unsigned long long)(int64_t)ev[u].y);
			}
		}
	}
	/* the wave's own counter: atomics of many waves on one address queue */
	if(lane == 0) atomicAdd(&a.block_events[NEMO_MAX_BIN_BLOCKS + (ng >> 6)], (unsigned long long)total);
}

/* Direct delivery of the rows (one per thread, [row.x, row.y), empty for
 * neurons that did not fire) of tile `tile` that fired in step t, this
 * block's part of them: every thread of a block of NEMO_TILE calls it, with
 * count (64 entries) and *chunks in LDS cleared and seen by all; chunk is
 * LDS too.  The chip does 23 G 64-bit atomics a second to random words,
 * whatever their scope and place, so this pays while a step has few events; a
 * bin round trip costs a network of any size its chain of dependent phases
 * instead.
 *
 * What counts here is the length of the chain: a thread lists in LDS those
 * pieces of its row, of 64 events, that are this part's, and after one
 * barrier each wave takes every fourth of them, a lane an event, with no scan
 * and no search (which took 1.3 us of a step's launch).  The parts agree on
 * their pieces by neuron and piece number; the order within a part is free. */
constexpr int DIRECT_ILP = 8;
__device__ inline void deliver_direct(const nemo_hip_direct& r, size_t acc_pitch, uint2 row, uint64_t t, unsigned tile,
		unsigned part, unsigned parts, uint2* chunk, uint32_t* chunks, uint32_t* count)
{
	constexpr unsigned WAVES = NEMO_TILE / 64;
	const unsigned tid = threadIdx.x, lane = tid & 63;
	/* pieces before, before + parts, ... of the row */
	const uint32_t pieces = (row.y - row.x + 63) / 64;
	const uint32_t before = parts == 1 ? 0 : (part + parts - tid % parts) % parts;
	const uint32_t mine = before < pieces ? (pieces - before + parts - 1) / parts : 0;
	const uint32_t first = mine ? atomicAdd(chunks, mine) : 0;
	uint32_t total = 0;
	for(uint32_t lo = 0;; lo += DIRECT_CHUNKS) {
		for(uint32_t q = max(first, lo); q < min(first + mine, lo + DIRECT_CHUNKS); ++q) {
			const uint32_t base = row.x + 64 * (before + (q - first) * parts);
			chunk[q - lo] = make_uint2(base, min(64u, row.y - base));
		}
		__syncthreads();
		total = *chunks;
		const uint32_t here = min(total - min(total, lo), DIRECT_CHUNKS);
		for(uint32_t c0 = tid / 64; c0 < here; c0 += DIRECT_ILP * WAVES) {
			int2 ev[DIRECT_ILP];
			unsigned d[DIRECT_ILP];
			bool live[DIRECT_ILP];
#pragma unroll
			for(int u = 0; u < DIRECT_ILP; ++u) {
				const uint32_t c = c0 + u * WAVES;
				const uint2 piece = chunk[min(c, here - 1)];
				live[u] = c < here && lane < piece.y;
				ev[u] = make_int2(0, 0);
				d[u] = 0;
				if(live[u]) {
					ev[u] = r.fcm[piece.x + lane];
					d[u] = r.delay[piece.x + lane];
				}
			}
#pragma unroll
			for(int u = 0; u < DIRECT_ILP; ++u) {
				if(!live[u]) continue;
				const uint32_t slot = uint32_t(t + 1 + d[u]) & r.mask;
				int64_t* dst = r.ring + (size_t(slot) * 2 + (ev[u].y >= 0 ? 0 : 1)) * acc_pitch + uint32_t(ev[u].x);
				atomicAdd(reinterpret_cast<unsigned long long*>(dst), (unsigned long long)(int64_t)ev[u].y);
				atomicAdd(&count[d[u]], 1u);
			}
		}
		if(lo + DIRECT_CHUNKS >= total) break;
		__syncthreads(); /* the list is rewritten */
	}
	if(!total) return;
	__syncthreads();
	if(tid < 64 && count[tid]) {
		atomicAdd(&r.arrivals[size_t(uint32_t(t + 1 + tid) & r.mask) * r.tiles + tile], count[tid]);
	}
}

/* In an update launch with direct delivery: run this block as one of those
 * after the group's tiles and return true, or return false in a tile's block.
 * The block reads a tile's firing of the step before from the bitmap and
 * delivers its part of the events of delays 2.. (the delay-1 events went out
 * with that step).  Beside the tiles' work, and split over parts, a tile that
 * fires a lot does not hold the step up. */
__device__ inline bool direct_block(const nemo_hip_step_buffers& b, const nemo_hip_neuron_group& g, UpdateLds& L)
{
	const unsigned tiles = (g.count + NEMO_TILE - 1) / NEMO_TILE;
	if(blockIdx.x < tiles) return false;
	const nemo_hip_direct& r = b.direct;
	const uint64_t t = current_step(b);
	if(t == 0) return true;
	const unsigned k = blockIdx.x - tiles;
	const unsigned tile = k / r.parts; /* of the network */
	const unsigned tid = threadIdx.x;
	const unsigned ng = tile * NEMO_TILE + tid;
	const uint64_t word = b.fired_bits[((t - 1) & (NEMO_STEP_RING - 1)) * b.fired_words + (ng >> 6)];
	const uint2 late = r.late_rows[ng];
	if(tid < 64) L.count[tid] = 0;
	if(tid == 64) L.chunks = 0;
	__syncthreads();
	const bool fired = (word >> (ng & 63)) & 1u;
	deliver_direct(r, b.acc_pitch, fired ? late : make_uint2(0, 0), t - 1, tile, k % r.parts, r.parts, L.chunk, &L.chunks,
			L.count);
	return true;
}

/* Blocks of an update launch of a group: its tiles, then the propagate blocks
 * it carries, or the blocks of direct delivery. */
inline unsigned update_blocks(const nemo_hip_neuron_group* g, const nemo_hip_step_buffers* b)
{
	const unsigned tiles = (g->count + NEMO_TILE - 1) / NEMO_TILE;
	return tiles + b->co.deliver_blocks + b->co.stdp_blocks + b->direct.late_blocks;
}

/* Store the shifted history (h as from load_history) and write the step's
 * firing bitmap. */
__device__ inline void record_firing(const nemo_hip_step_buffers& b, unsigned ng, bool valid, bool fired, uint64_t h)
{
	if(valid) {
		b.hist[NEMO_HIST_INDEX(ng, current_step(b), b.hist_pitch)] = (h << 1) | uint64_t(fired ? 1 : 0);
	}
	store_firing(b, ng, valid, fired);
}

/* The same in an update block whose input gather_input summed into L: with
 * co.push, or with direct delivery (never in a launch that carries propagate
 * blocks, CO), also deliver the firing's delay-1 events. */
template<bool CO>
__device__ inline void record_firing(const nemo_hip_step_buffers& b, UpdateLds& L, unsigned ng, bool valid,
		bool fired, uint64_t h)
{
	record_firing(b, ng, valid, fired, h);
	if constexpr(!CO) {
		if(b.direct.ring) {
			deliver_direct(b.direct, b.acc_pitch, valid && fired ? L.push_rows[threadIdx.x] : make_uint2(0, 0),
					current_step(b), ng / NEMO_TILE, 0, 1, L.chunk, &L.chunks, L.count);
			return;
		}
	}
	if(b.co.push) push_delay1(b, L, ng, valid, fired);
}

/* StdpProcess::updateRegion (StdpProcess.cpp:86-111): within one region of
 * arrivals, the nearest presynaptic arrival on either side of the
 * postsynaptic spike wins; a tie gives nothing. */
__device__ inline int32_t stdp_update_region(uint64_t arrivals, unsigned post_window, uint64_t pre_post,
		uint64_t post_pre, const int32_t* fn_pre, const int32_t* fn_post)
{
	if(!arrivals) return 0;
	const unsigned NONE = ~0u;
	const uint64_t pre = arrivals & pre_post;
	const uint64_t post = arrivals & post_pre;
	const unsigned dt_pre = pre ? unsigned(__builtin_ctzll(pre >> post_window)) : NONE;
	const unsigned dt_post = post ? unsigned(__builtin_clzll(post << (64 - post_window))) : NONE;
	if(dt_pre < dt_post) return fn_pre[dt_pre];
	if(dt_post < dt_pre) return fn_post[dt_post];
	return 0;
}

__device__ inline int32_t stdp_wrap_add(int32_t x, int32_t y)
{
	return int32_t(uint32_t(x) + uint32_t(y));
}

/* The STDP accumulation of the previous step for this tile's neurons (the
 * contract of nemo_hip_stdp).  h is the thread's neuron history after the
 * previous step (load_history).  Every thread of the block calls it. */
__device__ inline void stdp_tile(const nemo_hip_step_buffers& b, UpdateLds& L, unsigned ng, bool valid, uint64_t h)
{
	constexpr int ILP = 8;
	const nemo_hip_stdp& st = b.stdp;
	if(!st.rcm_ptr) return;
	const uint64_t t = current_step(b);
	if(t == 0) return;
	const uint64_t r = t - 1;
	if(r < st.post_window || r == b.clock->stdp_flushed) return;

	int32_t* s_fn = L.fn;
	uint32_t* s_rb = L.rb;
	uint32_t* s_pos = L.pos;
	const unsigned tid = threadIdx.x;
	if(tid < 64) {
		s_fn[tid] = st.fn_pre[tid];
		s_fn[64 + tid] = st.fn_post[tid];
	}
	const bool post = valid && ((h >> st.post_window) & 1u);
	uint32_t rb = 0, len = 0;
	if(post) {
		rb = st.rcm_ptr[ng];
		len = st.rcm_ptr[ng + 1] - rb;
	}
	uint32_t nfired;
	const uint32_t idx = block_exclusive_scan(post ? 1u : 0u, &nfired);
	uint32_t total;
	const uint32_t pos = block_exclusive_scan(len, &total);
	if(post) {
		s_rb[idx] = rb;
		s_pos[idx] = pos;
	}
	if(tid == 0) s_pos[nfired] = total;
	__syncthreads();
	if(total == 0) return;

	const uint64_t* pre_hist = b.hist + NEMO_HIST_INDEX(0, r, b.hist_pitch);
	for(uint32_t e0 = tid; e0 < total; e0 += ILP * NEMO_TILE) {
		uint32_t k[ILP];
		uint32_t sd[ILP];
		int32_t acc[ILP];
#pragma unroll
		for(int u = 0; u < ILP; ++u) k[u] = e0 + u * NEMO_TILE;
		unsigned lo[ILP];
		last_not_above_k<NEMO_TILE>(s_pos, nfired, k, lo);
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			const uint32_t e = k[u];
			k[u] = 0;
			sd[u] = 0;
			acc[u] = 0;
			if(e < total) {
				k[u] = s_rb[lo[u]] + (e - s_pos[lo[u]]);
				sd[u] = st.rcm_sd[k[u]];
				acc[u] = st.rcm_acc[k[u]];
			}
		}
		uint64_t ph[ILP];
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			ph[u] = 0;
			if(e0 + u * NEMO_TILE < total) ph[u] = pre_hist[sd[u] & 0x3ffffffu];
		}
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			if(e0 + u * NEMO_TILE < total) {
				const unsigned d = (sd[u] >> 26) + 1;
				const uint64_t arrivals = d >= 64 ? 0 : (ph[u] >> d);
				const int32_t dw = stdp_wrap_add(
						stdp_update_region(arrivals & st.potentiation, st.post_window, st.pre_post, st.post_pre,
							s_fn, s_fn + 64),
						stdp_update_region(arrivals & st.depression, st.post_window, st.pre_post, st.post_pre,
							s_fn, s_fn + 64));
				if(dw != 0) st.rcm_acc[k[u]] = stdp_wrap_add(acc[u], dw);
			}
		}
	}
	if(tid == 0) atomicAdd(&st.examined[ng / NEMO_TILE], (unsigned long long)total);
}

} // namespace nemo_dev

/* the propagate blocks an update launch may carry (colaunched_block) */
#include "propagate_device.h"

#endif
