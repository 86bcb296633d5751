/*
 * The backend's own gfx950 kernels: the per-step propagate kernel (binned
 * spike delivery), the STDP-only kernel, applyStdp and stimulus helpers.
 * Neuron updates, which also gather the binned input and usually run the
 * STDP accumulation, live in the model plugins (plugins/<Model>.hip).
 *
 * Data layout in HBM.  Device indices number neurons type by type, in
 * insertion order within a type (NeMo's simulation order,
 * src/nemo/cpu/Simulation.cpp:60-77), each type starting at a multiple of
 * NEMO_TILE (256):
 *   fcm        int2[S]     synapse rows (source, delay) back to back; row
 *                          (n, d) = [rowptr[n*D+d-1], rowptr[n*D+d]); entries
 *                          {target, Q11.20 weight}, 8 bytes, so consecutive
 *                          lanes read consecutive 8-byte words of a row
 *   fired_bits uint64[128][N/64]  one firing bitmap per step (ring)
 *   hist       uint64[2][N] firing history (bit k: fired k steps ago); plane
 *                          s % 2 holds the history after step s
 *   stdp_snap  uint64[N][2] two history snapshots per neuron (STDP batches)
 *   bins       int2[2][B][CAP] each delivery block's events, sorted by tile,
 *                          for steps of even and odd parity
 *   bin_table  uint32[2][T][B] count << 16 | offset of tile t in block b's
 *                          bins (entries of the blocks whose window holds t)
 *   acc        int64[2][2][N] overflow accumulators (events beyond CAP)
 *   rcm_*      per target, its plastic incoming synapses (STDP only)
 * and, for a network delivered directly (nemo_hip_direct), the ring of input
 * accumulators int64[slots][2][N] in place of bins, bin_table and acc.
 */
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>

#include "kernels.h"
#include "glibc_math.h"
#include "plugin_device.h"
#include "propagate_device.h"

namespace {

/* threads of a propagate (delivery or STDP) block */
constexpr unsigned PBLOCK = NEMO_PROPAGATE_BLOCK;

using nemo_dev::stdp_wrap_add;

/* delivery blocks, then (when fused into this launch) STDP blocks; at least
 * 6 waves per SIMD (80 VGPRs), so that three 512-thread blocks share a CU */
__global__ void __launch_bounds__(PBLOCK, 6)
propagate_kernel(nemo_propagate_args a)
{
	extern __shared__ uint64_t lds_dyn[];
	unsigned char* lds = reinterpret_cast<unsigned char*>(lds_dyn);
	const uint64_t t = a.clock->base_step + a.step_offset;
	if(blockIdx.x < a.deliver_blocks) {
		nemo_dev::deliver_block<PBLOCK>(a, t, blockIdx.x, lds);
	} else {
		nemo_dev::stdp_step<PBLOCK>(a, t, blockIdx.x - a.deliver_blocks, lds);
	}
}

/* Both delivery sets of one step in one launch: the first set's blocks, the
 * second's, then (when fused into this launch) STDP blocks of the first
 * set's arguments */
__global__ void __launch_bounds__(PBLOCK, 6)
propagate_sets_kernel(nemo_propagate_args a, nemo_propagate_args a2)
{
	extern __shared__ uint64_t lds_dyn[];
	unsigned char* lds = reinterpret_cast<unsigned char*>(lds_dyn);
	const uint64_t t = a.clock->base_step + a.step_offset;
	if(blockIdx.x < a.deliver_blocks) {
		nemo_dev::deliver_block<PBLOCK>(a, t, blockIdx.x, lds);
	} else if(blockIdx.x < a.deliver_blocks + a2.deliver_blocks) {
		nemo_dev::deliver_block<PBLOCK>(a2, t, blockIdx.x - a.deliver_blocks, lds);
	} else {
		nemo_dev::stdp_step<PBLOCK>(a, t, blockIdx.x - a.deliver_blocks - a2.deliver_blocks, lds);
	}
}

/* STDP blocks only */
__global__ void __launch_bounds__(PBLOCK)
stdp_kernel(nemo_propagate_args a)
{
	extern __shared__ uint64_t lds_dyn[];
	nemo_dev::stdp_step<PBLOCK>(a, a.clock->base_step + a.step_offset, blockIdx.x,
			reinterpret_cast<unsigned char*>(lds_dyn));
}

/* The pending STDP accumulation, one block per group of stdp_words bitmap
 * words (stdp_batch_block) */
__global__ void __launch_bounds__(NEMO_STDP_BATCH_BLOCK, NEMO_STDP_BATCH_WAVES)
stdp_batch_kernel(nemo_propagate_args a)
{
	extern __shared__ uint64_t lds_dyn[];
	nemo_dev::stdp_batch_block<NEMO_STDP_BATCH_BLOCK>(a, blockIdx.x, reinterpret_cast<unsigned char*>(lds_dyn));
}

/* The same as a flush, which nothing runs beside: wider blocks with more
 * loads in flight per thread */
__global__ void __launch_bounds__(PBLOCK)
stdp_flush_kernel(nemo_propagate_args a)
{
	extern __shared__ uint64_t lds_dyn[];
	nemo_dev::stdp_batch_block<PBLOCK, nemo_dev::STDP_FLUSH_ILP>(a, blockIdx.x,
			reinterpret_cast<unsigned char*>(lds_dyn));
}

/* A history snapshot after step base + offset into the free slot (the one
 * the last snapshot is not in) */
__global__ void __launch_bounds__(NEMO_BLOCK)
stdp_snapshot_kernel(nemo_propagate_args a, uint64_t offset)
{
	const uint64_t s = a.clock->base_step + offset;
	const unsigned slot = unsigned(a.clock->stdp_snaps + 1) & 1;
	const size_t n = a.fired_words * 64;
	for(size_t i = size_t(blockIdx.x) * NEMO_BLOCK + threadIdx.x; i < n; i += size_t(gridDim.x) * NEMO_BLOCK) {
		a.stdp_snap[2 * i + slot] = a.hist[NEMO_HIST_INDEX(i, s, a.hist_pitch)];
	}
}

/* ... after which the steps since the last snapshot are pending; and the
 * step base moves on by advance (the last node of a graph of steps, so that
 * the next graph needs no copy of its base from the host) */
__global__ void stdp_snapshot_done_kernel(nemo_hip_clock* clock, uint64_t offset, uint64_t advance)
{
	const uint64_t base = clock->base_step;
	const uint64_t s = base + offset;
	clock->stdp_first = clock->stdp_last + 1;
	clock->stdp_count = s - clock->stdp_last;
	clock->stdp_last = s;
	clock->stdp_snaps += 1;
	if(advance) clock->base_step = base + advance;
}

/* ... and after a flush of the pending batch: nothing is pending, and the
 * accumulation of step base + offset has run */
__global__ void stdp_flush_done_kernel(nemo_hip_clock* clock, uint64_t offset)
{
	clock->stdp_count = 0;
	clock->stdp_flushed = clock->base_step + offset;
}

/* applyStdp in forward order: every synapse of the FCM that is plastic
 * (rcm_of[j] its accumulator) takes its weight change; reading the weights in
 * order and the accumulators scattered costs one random read per synapse,
 * where the reverse order costs a random read and write of the weight.  The
 * accumulators are cleared afterwards by a separate fill.
 *
 * The random reads are cache lines that an XCD's L2 does not hold: 1660 us at
 * 1e8 synapses, 8e7 of them plastic.  So in large networks (a.tile) the
 * accumulators are first moved to tiles of APPLY_TILE consecutive FCM synapses
 * each (apply_collect_kernel, which also clears them), and the blocks of an
 * XCD, which are those of one number modulo 8, pass a tile together: it stays
 * in their L2: 372 + 638 us, of 2.3 + 1.3 GB.  Tiles of half or twice the size
 * take the same in sum. */
__device__ inline int32_t applied_weight(const nemo_apply_args& a, int32_t w, int32_t acc)
{
	const int32_t x = stdp_wrap_add(w, int32_t((int64_t(a.reward) * int64_t(acc)) >> a.fbits));
	return w > 0 ? min(a.maxE, max(x, a.minE)) : w < 0 ? min(a.minI, max(x, a.maxI)) : 0;
}

__global__ void __launch_bounds__(NEMO_BLOCK)
apply_stdp_kernel(nemo_apply_args a)
{
	/* APPLY_ILP pairs of synapses per thread at a time: their index and weight
	 * loads, then their accumulator gathers, are in flight together */
	constexpr unsigned APPLY_ILP = 4;
	constexpr size_t PIECE = NEMO_BLOCK * APPLY_ILP; /* pairs */
	constexpr size_t PIECES = NEMO_APPLY_TILE / 2 / PIECE; /* of a tile */
	size_t piece = blockIdx.x;
	if(a.tile) {
		const size_t g = blockIdx.x / 8;
		piece = (g / PIECES * 8 + blockIdx.x % 8) * PIECES + g % PIECES;
	}
	const size_t stride = size_t(gridDim.x) * PIECE;
	const size_t pairs = a.fcm_count / 2;
	const int32_t* source = a.tile ? a.tile : a.rcm_acc;
	const uint2* of = reinterpret_cast<const uint2*>(a.rcm_of);
	int4* fcm = reinterpret_cast<int4*>(a.fcm);
	for(size_t j0 = piece * PIECE + threadIdx.x; j0 < pairs; j0 += stride) {
		uint2 k[APPLY_ILP];
		int4 w[APPLY_ILP];
		int2 acc[APPLY_ILP];
#pragma unroll
		for(unsigned u = 0; u < APPLY_ILP; ++u) {
			const size_t j = j0 + u * NEMO_BLOCK;
			k[u] = j < pairs ? of[j] : make_uint2(~0u, ~0u);
			w[u] = j < pairs ? fcm[j] : make_int4(0, 0, 0, 0);
		}
#pragma unroll
		for(unsigned u = 0; u < APPLY_ILP; ++u) {
			acc[u].x = k[u].x != ~0u && a.reward != 0 ? source[k[u].x] : 0;
			acc[u].y = k[u].y != ~0u && a.reward != 0 ? source[k[u].y] : 0;
		}
#pragma unroll
		for(unsigned u = 0; u < APPLY_ILP; ++u) {
			const int32_t x = k[u].x != ~0u ? applied_weight(a, w[u].y, acc[u].x) : w[u].y;
			const int32_t y = k[u].y != ~0u ? applied_weight(a, w[u].w, acc[u].y) : w[u].w;
			/* in the large networks changed or not: whole lines are written to
			 * memory faster than some words of them (638 against 685 us at 1e8
			 * synapses, a third changed; at 1e7, which stay in the
			 * memory-side cache, 91 against 85) */
			const bool plastic = k[u].x != ~0u || k[u].y != ~0u;
			if(plastic && (a.tile || x != w[u].y || y != w[u].w))
				fcm[j0 + u * NEMO_BLOCK] = make_int4(w[u].x, x, w[u].z, y);
		}
	}
	if(a.fcm_count % 2 && blockIdx.x == 0 && threadIdx.x == 0) {
		const size_t j = a.fcm_count - 1;
		const uint32_t k = a.rcm_of[j];
		if(k != ~0u) a.fcm[j].y = applied_weight(a, a.fcm[j].y, a.reward != 0 ? source[k] : 0);
	}
}

/* The accumulators to their tiles, and cleared: in target order, in which they
 * are read and the places in a tile run on. */
__global__ void __launch_bounds__(NEMO_BLOCK)
apply_collect_kernel(nemo_apply_args a)
{
	constexpr unsigned ILP = 4;
	const size_t quads = a.count / 4;
	const size_t stride = size_t(gridDim.x) * NEMO_BLOCK * ILP;
	for(size_t q0 = size_t(blockIdx.x) * NEMO_BLOCK * ILP + threadIdx.x; q0 < quads; q0 += stride) {
		int4 acc[ILP];
		uint4 at[ILP];
#pragma unroll
		for(unsigned u = 0; u < ILP; ++u) {
			const size_t q = q0 + u * NEMO_BLOCK;
			if(q >= quads) continue;
			acc[u] = reinterpret_cast<const int4*>(a.rcm_acc)[q];
			at[u] = reinterpret_cast<const uint4*>(a.rcm_tile)[q];
		}
#pragma unroll
		for(unsigned u = 0; u < ILP; ++u) {
			const size_t q = q0 + u * NEMO_BLOCK;
			if(q >= quads) continue;
			a.tile[at[u].x] = acc[u].x;
			a.tile[at[u].y] = acc[u].y;
			a.tile[at[u].z] = acc[u].z;
			a.tile[at[u].w] = acc[u].w;
			reinterpret_cast<int4*>(a.rcm_acc)[q] = make_int4(0, 0, 0, 0);
		}
	}
	const size_t k = quads * 4 + threadIdx.x;
	if(blockIdx.x == 0 && k < a.count) {
		a.tile[a.rcm_tile[k]] = a.rcm_acc[k];
		a.rcm_acc[k] = 0;
	}
}

/* The place of every plastic synapse k in the tiles: rcm_tile[k] =
 * rcm_of[rcm_fwd[k]] (rcm_of filled with ~0 before), in tile rcm_fwd[k] /
 * APPLY_TILE, where a block's synapses, of neighbouring targets, follow each
 * other; used counts the places taken of each tile (zero before). */
constexpr unsigned TILE_SPAN = 16384; /* synapses per block */
constexpr unsigned TILE_MAX = 8192;   /* tiles: of 2^32 synapses */

__global__ void __launch_bounds__(NEMO_BLOCK)
assign_tiles_kernel(const uint32_t* rcm_fwd, uint32_t* rcm_of, uint32_t* rcm_tile, uint32_t* used, unsigned tiles,
		size_t count)
{
	__shared__ uint32_t place[TILE_MAX];
	const size_t first = size_t(blockIdx.x) * TILE_SPAN;
	const size_t last = min(count, first + TILE_SPAN);
	for(unsigned t = threadIdx.x; t < tiles; t += NEMO_BLOCK) place[t] = 0;
	__syncthreads();
	for(size_t k = first + threadIdx.x; k < last; k += NEMO_BLOCK) atomicAdd(&place[rcm_fwd[k] / NEMO_APPLY_TILE], 1u);
	__syncthreads();
	for(unsigned t = threadIdx.x; t < tiles; t += NEMO_BLOCK)
		if(place[t]) place[t] = t * NEMO_APPLY_TILE + atomicAdd(&used[t], place[t]);
	__syncthreads();
	for(size_t k = first + threadIdx.x; k < last; k += NEMO_BLOCK) {
		const uint32_t f = rcm_fwd[k];
		const uint32_t at = atomicAdd(&place[f / NEMO_APPLY_TILE], 1u);
		rcm_tile[k] = at;
		rcm_of[f] = at;
	}
}

/* rcm_of[rcm_fwd[k]] = k for every plastic synapse k (rcm_of filled with ~0 before) */
__global__ void __launch_bounds__(NEMO_BLOCK)
invert_rcm_kernel(const uint32_t* rcm_fwd, uint32_t* rcm_of, size_t count)
{
	for(size_t k = size_t(blockIdx.x) * NEMO_BLOCK + threadIdx.x; k < count; k += size_t(gridDim.x) * NEMO_BLOCK) {
		rcm_of[rcm_fwd[k]] = uint32_t(k);
	}
}

/* Tells the host, which polls done->flag in pinned memory, that the kernel's
 * writes to pinned memory are there: by the last of its blocks to get here,
 * every thread of which calls it (done->blocks counts them, and ends at 0). */
__device__ inline void signal_done(const nemo_host_signal& done)
{
	__threadfence_system();
	__syncthreads();
	if(threadIdx.x != 0) return;
	if(gridDim.x > 1) {
		if(atomicAdd(done.blocks, 1u) + 1 < gridDim.x) return;
		*done.blocks = 0;
		__threadfence_system();
	}
	__hip_atomic_store(done.flag, done.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* ------------------------------------------------------ firing readout */

constexpr unsigned READOUT_BLOCK = 512;
/* entries of a step's list that its block puts in order in LDS */
constexpr unsigned READOUT_STAGE = 4096;

/* The neurons fired in step base + offset + blockIdx.x (its firing-bitmap ring
 * slot), in ascending device index: counts[slot] of them, list[slot][..] the
 * first room of them, as index's entries (or, index NULL, device indices).
 * counts and list are pinned host memory, so that the host reads them without
 * a copy: per 64 steps, two copies and the events between the streams took 65
 * us.  The list goes out through LDS, in whole lines. */
__global__ void __launch_bounds__(READOUT_BLOCK)
fired_readout_kernel(const nemo_hip_clock* clock, uint64_t offset, const uint64_t* bits, size_t words,
		const uint32_t* index, uint32_t* counts, uint32_t* list, unsigned room, nemo_host_signal done)
{
	__shared__ uint32_t s_list[READOUT_STAGE];
	const uint64_t base = nemo_dev::clock_base(clock) + offset;
	const size_t slot = (base + blockIdx.x) & (NEMO_STEP_RING - 1);
	const uint64_t* b = bits + slot * words;
	uint32_t* out = list + slot * room;
	/* a contiguous run of words per thread keeps the list in device order */
	const size_t per = (words + READOUT_BLOCK - 1) / READOUT_BLOCK;
	const size_t w0 = min(words, size_t(threadIdx.x) * per), w1 = min(words, w0 + per);
	uint32_t c = 0;
	for(size_t w = w0; w < w1; ++w) c += uint32_t(__popcll(b[w]));
	uint32_t total;
	uint32_t pos = nemo_dev::block_exclusive_scan<READOUT_BLOCK>(c, &total);
	if(threadIdx.x == 0) counts[slot] = total;
	const bool staged = total <= READOUT_STAGE;
	for(size_t w = w0; w < w1; ++w) {
		for(uint64_t x = b[w]; x; x &= x - 1, ++pos) {
			const uint32_t n = uint32_t(w * 64) + uint32_t(__builtin_ctzll(x));
			const uint32_t v = index ? index[n] : n;
			if(staged) s_list[pos] = v;
			else if(pos < room) out[pos] = v;
		}
	}
	if(staged) {
		__syncthreads();
		for(uint32_t i = threadIdx.x; i < min(total, room); i += READOUT_BLOCK) out[i] = s_list[i];
	}
	done.value += base;
	signal_done(done);
}

/* *sum = the total of the n counters (sum in pinned host memory).  One block. */
__global__ void __launch_bounds__(READOUT_BLOCK)
sum_counters_kernel(const unsigned long long* counters, size_t n, uint64_t* sum, nemo_host_signal done)
{
	__shared__ unsigned long long s_sum;
	if(threadIdx.x == 0) s_sum = 0;
	__syncthreads();
	unsigned long long x = 0;
	for(size_t i = threadIdx.x; i < n; i += READOUT_BLOCK) x += counters[i];
	if(x) atomicAdd(&s_sum, x);
	__syncthreads();
	if(threadIdx.x == 0) *sum = s_sum;
	if(done.flag) signal_done(done);
}

/* ------------------------------------------- externally given firing */

/* All tiles as one group, for the blocks that need no more of it. */
__device__ inline nemo_hip_neuron_group whole_group(unsigned tiles)
{
	nemo_hip_neuron_group g = {};
	g.count = tiles * NEMO_TILE;
	return g;
}

/* The firing of step s given from outside (Brian's propagate,
 * cpu/Simulation.cpp:115-137): neuron ng fired if flags[sim] is nonzero for
 * its simulation index sim = dev_to_sim[ng] (~0 for padding), or, without
 * flags, if its bit in bits is set, which is cleared; its history
 * and the step's bitmap word are written as an update would. */
__global__ void __launch_bounds__(NEMO_TILE)
external_fire_kernel(nemo_hip_step_buffers b, const uint32_t* flags, uint32_t* bits, const uint32_t* dev_to_sim)
{
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<false>();
	if(b.direct.ring && nemo_dev::direct_block(b, whole_group(b.direct.tiles), L)) return;
	const unsigned ng = blockIdx.x * NEMO_TILE + threadIdx.x;
	const uint32_t sim = dev_to_sim[ng];
	const bool valid = sim != ~0u;
	const uint64_t h = nemo_dev::load_history(b, ng, valid);
	nemo_dev::begin_push(b, L, ng);
	const bool fired = valid && (flags ? flags[sim] != 0u : ((bits[ng >> 5] >> (ng & 31)) & 1u) != 0u);
	nemo_dev::record_firing<false>(b, L, ng, valid, fired, h);
	/* the wave has read its two words */
	if(!flags && (threadIdx.x & 31) == 0) bits[ng >> 5] = 0;
}

/* ------------------------------------------------------ direct delivery */

/* The events that arrive from step t0 on of the firing of step t0 - j, j =
 * 1 .. D (blockIdx.y + 1), of source tile blockIdx.x: of a neuron that fired
 * then, the rows of delays j .. D, which follow each other in the FCM; of the
 * last step's firing the delay-1 row only, as the update of step t0 delivers
 * the others. */
__global__ void __launch_bounds__(NEMO_TILE)
direct_rebuild_kernel(nemo_hip_direct r, size_t acc_pitch, const uint32_t* rowptr, unsigned D,
		const uint64_t* fired_bits, size_t fired_words, uint64_t t0)
{
	__shared__ uint2 s_chunk[nemo_dev::DIRECT_CHUNKS];
	__shared__ uint32_t s_count[64], s_chunks;
	const unsigned tile = blockIdx.x, j = blockIdx.y + 1, tid = threadIdx.x;
	if(t0 < j) return;
	const uint64_t t = t0 - j;
	const uint64_t word = fired_bits[(t & (NEMO_STEP_RING - 1)) * fired_words + size_t(tile) * (NEMO_TILE / 64) + tid / 64];
	const bool fired = (word >> (tid & 63)) & 1u;
	if(tid < 64) s_count[tid] = 0;
	if(tid == 64) s_chunks = 0;
	if(!__syncthreads_or(fired)) return;
	uint2 row = make_uint2(0, 0);
	if(fired) {
		const size_t n = size_t(tile) * NEMO_TILE + tid;
		row.x = rowptr[n * D + j - 1];
		row.y = rowptr[n * D + (j == 1 ? 1 : D)];
	}
	nemo_dev::deliver_direct(r, acc_pitch, row, t, tile, 0, 1, s_chunk, &s_chunks, s_count);
}

/* The synaptic input of a step, gathered per tile as the neuron updates
 * gather it (overflow accumulators cleared), converted to float and written
 * in simulation order: E[sim], I[sim]. */
__global__ void __launch_bounds__(NEMO_TILE)
gather_currents_kernel(nemo_hip_step_buffers b, const uint32_t* dev_to_sim, float* E, float* I, nemo_host_signal done)
{
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<false>();
	const nemo_hip_neuron_group g = whole_group(gridDim.x);
	const unsigned ng = blockIdx.x * NEMO_TILE + threadIdx.x;
	if(b.direct.ring) {
		/* read, not taken: an update of this step would still find its
		 * input.  The step before passed without one: its slot is cleared
		 * for the steps to come. */
		const nemo_hip_direct& r = b.direct;
		const uint64_t t = nemo_dev::current_step(b);
		const size_t slot = size_t(t) & r.mask, before = size_t(t - 1) & r.mask;
		L.input.E[threadIdx.x] = r.ring[slot * 2 * b.acc_pitch + ng];
		L.input.I[threadIdx.x] = r.ring[(slot * 2 + 1) * b.acc_pitch + ng];
		r.ring[before * 2 * b.acc_pitch + ng] = 0;
		r.ring[(before * 2 + 1) * b.acc_pitch + ng] = 0;
		if(threadIdx.x == 0) {
			r.events[ng >> 6] += r.arrivals[slot * r.tiles + blockIdx.x];
			r.arrivals[before * r.tiles + blockIdx.x] = 0;
		}
	} else {
		nemo_dev::gather_input(b, g, L);
	}
	float e, i;
	nemo_dev::take_current(b, L.input, ng, e, i);
	const uint32_t sim = dev_to_sim[ng];
	if(sim != ~0u) {
		E[sim] = e;
		I[sim] = i;
	}
	if(done.flag) signal_done(done);
}

/* ------------------------------------------------------------ stimulus */

/* The stimulus of a step, read from the host's pinned lists: firing bits set,
 * external currents written (distinct neurons). */
__global__ void __launch_bounds__(NEMO_BLOCK)
stimulus_kernel(uint32_t* bits, const uint32_t* fidx, size_t nf, float* ext, const uint32_t* iidx, const float* ival,
		size_t ni)
{
	const size_t i = size_t(blockIdx.x) * NEMO_BLOCK + threadIdx.x;
	if(i < nf) atomicOr(&bits[fidx[i] >> 5], 1u << (fidx[i] & 31));
	if(i < ni) ext[iidx[i]] = ival[i];
}

/* ... and its end: the step's firing bitmap written to pinned host memory,
 * the firing stimulus cleared (its words hold no other bits).  One block. */
__global__ void __launch_bounds__(NEMO_BLOCK)
step_readout_kernel(const uint64_t* fired, uint64_t* out, size_t words, uint32_t* bits, const uint32_t* fidx, size_t nf,
		nemo_host_signal done)
{
	for(size_t i = threadIdx.x; i < words; i += NEMO_BLOCK) out[i] = fired[i];
	for(size_t i = threadIdx.x; i < nf; i += NEMO_BLOCK) bits[fidx[i] >> 5] = 0;
	signal_done(done);
}

/* out[i] = *src[i], from and to pinned host memory */
__global__ void __launch_bounds__(NEMO_BLOCK)
read_values_kernel(const float* const* src, float* out, size_t n, nemo_host_signal done)
{
	const size_t i = size_t(blockIdx.x) * NEMO_BLOCK + threadIdx.x;
	if(i < n) out[i] = *src[i];
	signal_done(done);
}

/* The step base moved on by the last node of a graph of steps, so that the
 * next graph needs no copy of its base from the host: that copy starts 5 to
 * 15 us after the last kernel, and the next graph 15 to 20 us after it. */
__global__ void advance_clock_kernel(nemo_hip_clock* clock, uint64_t steps)
{
	clock->base_step += steps;
}

__global__ void eval_math_kernel(int fn, const float* in, float* out, size_t n)
{
	const size_t i = size_t(blockIdx.x) * NEMO_BLOCK + threadIdx.x;
	if(i < n) {
		const float x = in[i];
		out[i] = fn == 0 ? nemo_math::logf_exact(x) : fn == 1 ? nemo_math::sinf_exact(x) : nemo_math::expf_exact(x);
	}
}

} // namespace

extern "C" {

size_t nemo_propagate_lds_bytes(unsigned max_window, unsigned bin_capacity)
{
	return nemo_dev::PropagateLds<PBLOCK>::delivery_bytes(bin_capacity, max_window);
}

static bool stdp_batch_args_valid(const nemo_propagate_args* a, unsigned stdp_blocks)
{
	return a->stdp_snap && a->stdp.post_window <= 63 && a->stdp_words > 0 && a->stdp_words <= NEMO_STDP_BATCH_MAX_WORDS
		&& size_t(stdp_blocks) * a->stdp_words >= a->fired_words && a->stdp.rcm_ptr;
}

hipError_t nemo_launch_stdp_batch(hipStream_t st, const nemo_propagate_args* a, unsigned stdp_blocks)
{
	if(stdp_blocks == 0) return hipSuccess;
	if(!stdp_batch_args_valid(a, stdp_blocks)) return hipErrorInvalidValue;
	hipLaunchKernelGGL(stdp_batch_kernel, dim3(stdp_blocks), dim3(NEMO_STDP_BATCH_BLOCK),
			nemo_dev::PropagateLds<NEMO_STDP_BATCH_BLOCK>::stdp_bytes(), st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_stdp_flush(hipStream_t st, const nemo_propagate_args* a, unsigned stdp_blocks, uint64_t offset)
{
	if(stdp_blocks == 0) return hipSuccess;
	if(!stdp_batch_args_valid(a, stdp_blocks)) return hipErrorInvalidValue;
	hipLaunchKernelGGL(stdp_flush_kernel, dim3(stdp_blocks), dim3(PBLOCK), nemo_dev::PropagateLds<PBLOCK>::stdp_bytes(),
			st, *a);
	hipError_t e = hipGetLastError();
	if(e != hipSuccess) return e;
	hipLaunchKernelGGL(stdp_flush_done_kernel, dim3(1), dim3(1), 0, st, const_cast<nemo_hip_clock*>(a->clock), offset);
	return hipGetLastError();
}

hipError_t nemo_launch_stdp_snapshot(hipStream_t st, const nemo_propagate_args* a, uint64_t offset, uint64_t advance)
{
	if(!a->stdp_snap || !a->hist) return hipErrorInvalidValue;
	const size_t n = a->fired_words * 64;
	const unsigned blocks = unsigned(std::min<size_t>(1024, (n + NEMO_BLOCK - 1) / NEMO_BLOCK));
	hipLaunchKernelGGL(stdp_snapshot_kernel, dim3(blocks), dim3(NEMO_BLOCK), 0, st, *a, offset);
	hipError_t e = hipGetLastError();
	if(e != hipSuccess) return e;
	hipLaunchKernelGGL(stdp_snapshot_done_kernel, dim3(1), dim3(1), 0, st, const_cast<nemo_hip_clock*>(a->clock),
			offset, advance);
	return hipGetLastError();
}

size_t nemo_colaunch_lds_bytes(unsigned max_window, unsigned bin_capacity, int delivery)
{
	/* the update blocks of the launch take their LDS from the same buffer */
	return std::max(nemo_dev::PropagateLds<NEMO_COLAUNCH_BLOCK>::bytes(delivery != 0,
					bin_capacity, max_window),
			sizeof(nemo_dev::UpdateLds));
}

size_t nemo_propagate_static_lds(void)
{
	hipFuncAttributes fa;
	if(hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(propagate_kernel)) != hipSuccess) return 32768;
	return fa.sharedSizeBytes;
}

hipError_t nemo_launch_propagate(hipStream_t st, const nemo_propagate_args* a, unsigned stdp_blocks, int fuse_stdp,
		hipEvent_t start, hipEvent_t stop)
{
	if(a->deliver_blocks > NEMO_MAX_BIN_BLOCKS) return hipErrorInvalidValue;
	if(a->deliver_blocks && (a->D == 0 || a->D > NEMO_MAX_DELAY || a->bin_capacity == 0
				|| a->bin_capacity > 32768 || a->max_window == 0 || a->max_window > a->tiles
				|| !a->pair_bounds || !a->windows || a->d_first == 0 || a->d_count == 0
				|| a->d_first + a->d_count - 1 > a->D || a->block_base + a->deliver_blocks > a->table_columns
				|| a->table_columns > NEMO_MAX_BIN_BLOCKS)) {
		return hipErrorInvalidValue;
	}
	if(stdp_blocks && (a->stdp.post_window > 63 || a->stdp_words == 0 || a->stdp_words > NEMO_STDP_MAX_WORDS
				|| size_t(stdp_blocks) * a->stdp_words < a->fired_words || !a->stdp.rcm_ptr || !a->hist)) {
		return hipErrorInvalidValue;
	}
	const size_t lds = nemo_dev::PropagateLds<PBLOCK>::bytes(a->deliver_blocks > 0, a->bin_capacity, a->max_window);
	if(fuse_stdp) {
		const unsigned blocks = a->deliver_blocks + stdp_blocks;
		if(blocks == 0) return hipSuccess;
		hipExtLaunchKernelGGL(propagate_kernel, dim3(blocks), dim3(PBLOCK), lds, st, start, stop, 0, *a);
		return hipGetLastError();
	}
	if(stdp_blocks) {
		hipExtLaunchKernelGGL(stdp_kernel, dim3(stdp_blocks), dim3(PBLOCK), nemo_dev::PropagateLds<PBLOCK>::stdp_bytes(),
				st, start, a->deliver_blocks ? nullptr : stop, 0, *a);
		const hipError_t e = hipGetLastError();
		if(e != hipSuccess) return e;
	}
	if(a->deliver_blocks) {
		hipExtLaunchKernelGGL(propagate_kernel, dim3(a->deliver_blocks), dim3(PBLOCK), lds, st,
				stdp_blocks ? nullptr : start, stop, 0, *a);
		return hipGetLastError();
	}
	return hipSuccess;
}

hipError_t nemo_launch_propagate_sets(hipStream_t st, const nemo_propagate_args* a, const nemo_propagate_args* a2,
		unsigned stdp_blocks, hipEvent_t start, hipEvent_t stop)
{
	if(!a2->deliver_blocks) return nemo_launch_propagate(st, a, stdp_blocks, 1, start, stop);
	if(!a->deliver_blocks) {
		if(stdp_blocks) return hipErrorInvalidValue; /* the STDP blocks take the first set's arguments */
		return nemo_launch_propagate(st, a2, 0, 1, start, stop);
	}
	if(a->step_offset != a2->step_offset || a->clock != a2->clock || a->bin_capacity != a2->bin_capacity
			|| a->max_window != a2->max_window || a->table_columns != a2->table_columns
			|| a->deliver_blocks + a2->deliver_blocks > NEMO_MAX_BIN_BLOCKS) {
		return hipErrorInvalidValue;
	}
	for(const nemo_propagate_args* x : {a, a2}) {
		if(x->D == 0 || x->D > NEMO_MAX_DELAY || x->bin_capacity == 0 || x->bin_capacity > 32768
				|| x->max_window == 0 || x->max_window > x->tiles || !x->pair_bounds || !x->windows
				|| x->d_first == 0 || x->d_count == 0 || x->d_first + x->d_count - 1 > x->D
				|| x->block_base + x->deliver_blocks > x->table_columns || x->table_columns > NEMO_MAX_BIN_BLOCKS) {
			return hipErrorInvalidValue;
		}
	}
	if(stdp_blocks && (a->stdp.post_window > 63 || a->stdp_words == 0 || a->stdp_words > NEMO_STDP_MAX_WORDS
				|| size_t(stdp_blocks) * a->stdp_words < a->fired_words || !a->stdp.rcm_ptr || !a->hist)) {
		return hipErrorInvalidValue;
	}
	const size_t lds = nemo_dev::PropagateLds<PBLOCK>::bytes(true, a->bin_capacity, a->max_window);
	const unsigned blocks = a->deliver_blocks + a2->deliver_blocks + stdp_blocks;
	hipExtLaunchKernelGGL(propagate_sets_kernel, dim3(blocks), dim3(PBLOCK), lds, st, start, stop, 0, *a, *a2);
	return hipGetLastError();
}

hipError_t nemo_launch_apply_stdp(hipStream_t st, const nemo_apply_args* a)
{
	if(a->count == 0) return hipSuccess;
	if(a->tile) {
		if(!a->rcm_tile) return hipErrorInvalidValue;
		size_t blocks = (a->count + 16 * NEMO_BLOCK - 1) / (16 * NEMO_BLOCK);
		if(blocks > 16384) blocks = 16384;
		hipLaunchKernelGGL(apply_collect_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, *a);
		hipError_t e = hipGetLastError();
		if(e != hipSuccess) return e;
		/* whole tiles for each XCD */
		const size_t tiles = (a->fcm_count + NEMO_APPLY_TILE - 1) / NEMO_APPLY_TILE;
		blocks = (tiles + 7) / 8 * 8 * (NEMO_APPLY_TILE / (8 * NEMO_BLOCK));
		hipLaunchKernelGGL(apply_stdp_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, *a);
		return hipGetLastError();
	}
	size_t blocks = (a->fcm_count + 8 * NEMO_BLOCK - 1) / (8 * NEMO_BLOCK);
	if(blocks > 16384) blocks = 16384;
	hipLaunchKernelGGL(apply_stdp_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, *a);
	hipError_t e = hipGetLastError();
	if(e != hipSuccess) return e;
	return hipMemsetAsync(a->rcm_acc, 0, a->count * sizeof(int32_t), st);
}

hipError_t nemo_launch_invert_rcm(hipStream_t st, const uint32_t* rcm_fwd, uint32_t* rcm_of, size_t count,
		size_t fcm_count)
{
	hipError_t e = hipMemsetAsync(rcm_of, 0xff, fcm_count * sizeof(uint32_t), st);
	if(e != hipSuccess || count == 0) return e;
	size_t blocks = (count + NEMO_BLOCK - 1) / NEMO_BLOCK;
	if(blocks > 16384) blocks = 16384;
	hipLaunchKernelGGL(invert_rcm_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, rcm_fwd, rcm_of, count);
	return hipGetLastError();
}

hipError_t nemo_launch_assign_tiles(hipStream_t st, const uint32_t* rcm_fwd, uint32_t* rcm_of, uint32_t* rcm_tile,
		uint32_t* used, size_t count, size_t fcm_count)
{
	const size_t tiles = (fcm_count + NEMO_APPLY_TILE - 1) / NEMO_APPLY_TILE;
	if(tiles > TILE_MAX) return hipErrorInvalidValue;
	hipError_t e = hipMemsetAsync(rcm_of, 0xff, fcm_count * sizeof(uint32_t), st);
	if(e == hipSuccess) e = hipMemsetAsync(used, 0, tiles * sizeof(uint32_t), st);
	if(e != hipSuccess || count == 0) return e;
	const size_t blocks = (count + TILE_SPAN - 1) / TILE_SPAN;
	hipLaunchKernelGGL(assign_tiles_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, rcm_fwd, rcm_of, rcm_tile,
			used, unsigned(tiles), count);
	return hipGetLastError();
}

hipError_t nemo_launch_external_fire(hipStream_t st, const nemo_hip_step_buffers* b, const uint32_t* flags, uint32_t* bits,
		const uint32_t* dev_to_sim, unsigned tiles)
{
	if(tiles == 0) return hipSuccess;
	if(b->direct.ring && b->direct.tiles != tiles) return hipErrorInvalidValue;
	const unsigned blocks = tiles + b->direct.late_blocks;
	hipLaunchKernelGGL(external_fire_kernel, dim3(blocks), dim3(NEMO_TILE), 0, st, *b, flags, bits, dev_to_sim);
	return hipGetLastError();
}

hipError_t nemo_launch_direct_rebuild(hipStream_t st, const nemo_hip_direct* r, size_t acc_pitch, const uint32_t* rowptr,
		unsigned D, const uint64_t* fired_bits, size_t fired_words, uint64_t t0)
{
	if(!r->ring || !r->fcm || !r->delay || !r->arrivals || D == 0 || D > NEMO_MAX_DELAY || r->mask < D
			|| (r->mask & (r->mask + 1)) || fired_words != size_t(r->tiles) * (NEMO_TILE / 64)) {
		return hipErrorInvalidValue;
	}
	if(r->tiles == 0) return hipSuccess;
	const size_t slots = size_t(r->mask) + 1;
	hipError_t e = hipMemsetAsync(r->ring, 0, slots * 2 * acc_pitch * sizeof(int64_t), st);
	if(e != hipSuccess) return e;
	e = hipMemsetAsync(r->arrivals, 0, slots * r->tiles * sizeof(uint32_t), st);
	if(e != hipSuccess) return e;
	hipLaunchKernelGGL(direct_rebuild_kernel, dim3(r->tiles, D), dim3(NEMO_TILE), 0, st, *r, acc_pitch, rowptr, D,
			fired_bits, fired_words, t0);
	return hipGetLastError();
}

hipError_t nemo_launch_gather_currents(hipStream_t st, const nemo_hip_step_buffers* b, const uint32_t* dev_to_sim,
		float* E, float* I, unsigned tiles, const nemo_host_signal* done)
{
	if(tiles == 0) return hipErrorInvalidValue; /* no block to signal */
	hipLaunchKernelGGL(gather_currents_kernel, dim3(tiles), dim3(NEMO_TILE), 0, st, *b, dev_to_sim, E, I, *done);
	return hipGetLastError();
}

hipError_t nemo_launch_fired_readout(hipStream_t st, const nemo_hip_clock* clock, uint64_t offset, unsigned k,
		const uint64_t* bits, size_t words, const uint32_t* index, uint32_t* counts, uint32_t* list, unsigned room,
		const nemo_host_signal* done)
{
	if(k == 0 || k > NEMO_STEP_RING || !clock || !bits || !counts || !list || !done->flag) return hipErrorInvalidValue;
	hipLaunchKernelGGL(fired_readout_kernel, dim3(k), dim3(READOUT_BLOCK), 0, st, clock, offset, bits, words, index, counts,
			list, room, *done);
	return hipGetLastError();
}

hipError_t nemo_launch_sum_counters(hipStream_t st, const unsigned long long* counters, size_t n, uint64_t* sum,
		const nemo_host_signal* done)
{
	hipLaunchKernelGGL(sum_counters_kernel, dim3(1), dim3(READOUT_BLOCK), 0, st, counters, n, sum, *done);
	return hipGetLastError();
}

hipError_t nemo_launch_stimulus(hipStream_t st, uint32_t* bits, const uint32_t* fidx, size_t nf, float* ext,
		const uint32_t* iidx, const float* ival, size_t ni)
{
	const size_t n = std::max(nf, ni);
	if(n == 0) return hipSuccess;
	hipLaunchKernelGGL(stimulus_kernel, dim3(unsigned((n + NEMO_BLOCK - 1) / NEMO_BLOCK)), dim3(NEMO_BLOCK), 0, st, bits,
			fidx, nf, ext, iidx, ival, ni);
	return hipGetLastError();
}

hipError_t nemo_launch_step_readout(hipStream_t st, const uint64_t* fired, uint64_t* out, size_t words, uint32_t* bits,
		const uint32_t* fidx, size_t nf, const nemo_host_signal* done)
{
	hipLaunchKernelGGL(step_readout_kernel, dim3(1), dim3(NEMO_BLOCK), 0, st, fired, out, words, bits, fidx, nf, *done);
	return hipGetLastError();
}

hipError_t nemo_launch_read_values(hipStream_t st, const float* const* src, float* out, size_t n,
		const nemo_host_signal* done)
{
	const size_t blocks = std::max<size_t>(1, (n + NEMO_BLOCK - 1) / NEMO_BLOCK);
	hipLaunchKernelGGL(read_values_kernel, dim3(unsigned(blocks)), dim3(NEMO_BLOCK), 0, st, src, out, n, *done);
	return hipGetLastError();
}

hipError_t nemo_launch_advance_clock(hipStream_t st, nemo_hip_clock* clock, uint64_t steps)
{
	hipLaunchKernelGGL(advance_clock_kernel, dim3(1), dim3(1), 0, st, clock, steps);
	return hipGetLastError();
}

hipError_t nemo_launch_eval_math(hipStream_t st, int fn, const float* in, float* out, size_t n)
{
	if(n == 0) return hipSuccess;
	hipLaunchKernelGGL(eval_math_kernel, dim3(unsigned((n + NEMO_BLOCK - 1) / NEMO_BLOCK)), dim3(NEMO_BLOCK), 0, st,
			fn, in, out, n);
	return hipGetLastError();
}

} // extern "C"
