/*
 * Device code of the propagate blocks -- spike delivery of one step and STDP
 * accumulation of the previous one -- shared by the backend's own propagate
 * launches and by neuron-update launches that carry them as extra blocks
 * after their tiles.  Templated on the block width; all LDS comes from one
 * dynamic buffer whose layout PropagateLds describes, so a launch that also
 * runs other blocks pays no static LDS for these.
 *
 * Semantics: delivery as cpu::Simulation::deliverSpikes
 * (src/nemo/cpu/Simulation.cpp:259-308), binned by target tile (the contract
 * of nemo_propagate_args); STDP as ConnectivityMatrix::accumulateStdp
 * (src/nemo/ConnectivityMatrix.cpp:224-258) with StdpProcess::weightChange
 * (src/nemo/StdpProcess.cpp:68-124).
 */
#ifndef NEMO_AMD_PROPAGATE_DEVICE_H
#define NEMO_AMD_PROPAGATE_DEVICE_H

#include "plugin_device.h"

namespace nemo_dev {

constexpr uint64_t PROPAGATE_RING_MASK = NEMO_STEP_RING - 1;
/* independent global loads each thread keeps in flight in the synapse loop
 * of STDP, and in the event loop of delivery */
constexpr int ILP = 8;
/* 8, not 16: with the launch held to 80 VGPRs a CU runs three 512-thread
 * delivery blocks at once instead of two, which pays when there are more
 * blocks than CUs (batches) and costs nothing with one block per CU */
constexpr int EVENT_ILP = 8;
/* The delivery blocks an update launch carries (overlap 3) keep 6: that
 * launch is held to 72 VGPRs (NEMO_COLAUNCH_WAVES), so that beside three of
 * its blocks a CU's SIMDs still hold one wave each of an STDP batch block
 * (NEMO_STDP_BATCH_BLOCK threads, 80 VGPRs).  8 would take all 72 and gains
 * nothing (19.62 against 19.65 us a step at 100k x 1000 with STDP) */
constexpr int CARRIED_EVENT_ILP = 6;
/* independent global loads per thread in the synapse loop of the STDP batch
 * beside the steps, held to 80 VGPRs (NEMO_STDP_BATCH_WAVES waves per SIMD),
 * and of a flush's batch, which nothing runs beside */
constexpr int STDP_BATCH_ILP = 5;
constexpr int STDP_FLUSH_ILP = 8;

/* Synapses per listed target, on average, from which a wave passes a target by
 * itself (stdp_batch_rows; below, its last lanes idle for longer than the
 * search takes).  Flush of 50 steps in us, search / wave per target: 30000
 * neurons of 80 plastic synapses each 13.6 / 14.3, 128 17.2 / 16.3, 200 25.6 /
 * 19.8; 32 networks of 40 to 800 111 / 95; 100000 of 800 287 / 267. */
constexpr uint32_t STDP_WAVE_ROW = 112;
/* staged events per thread the delivery sort keeps in registers */
constexpr unsigned SORT_REGS = 8;

/* LDS of a propagate block of THREADS threads, carved from one buffer:
 * staged events (bin capacity), the fired rows of a batch (ROWS at a time)
 * and the pieces of their events (PIECES at a time: first event, and count <<
 * 25 | place in the stage), the counters of the three, and per-window-tile
 * counts and cursors.  An STDP block uses the start of the same buffer for
 * its weight-change table, row bases and prefix. */
template<unsigned THREADS>
struct PropagateLds {
	static constexpr unsigned PIECE = 16;
	static constexpr unsigned ROWS = THREADS;
	static constexpr unsigned PIECES = 2 * THREADS;
	int2* stage;
	uint2* piece;
	uint32_t* row;
	uint32_t* rows;   /* fired rows of the batch */
	uint32_t* pieces; /* pieces of the chunk of rows */
	uint32_t* fill;   /* events staged, or delivered beyond the stage */
	uint32_t* cnt;
	uint32_t* cur;
	__device__ PropagateLds(unsigned char* p, unsigned cap, unsigned max_window)
	{
		stage = reinterpret_cast<int2*>(p);
		piece = reinterpret_cast<uint2*>(stage + cap);
		row = reinterpret_cast<uint32_t*>(piece + PIECES);
		rows = row + ROWS;
		pieces = rows + 1;
		fill = rows + 2;
		cnt = rows + 4;
		cur = cnt + max_window;
	}
	static constexpr size_t delivery_bytes(unsigned cap, unsigned max_window)
	{
		return size_t(cap) * 8 + size_t(PIECES) * 8 + 4 * (size_t(ROWS) + 4) + 8 * size_t(max_window);
	}
	static constexpr size_t stdp_bytes() { return 128 * 4 + 4 * (2 * size_t(THREADS) + 2) + 8 * size_t(THREADS); }
	static constexpr size_t bytes(bool delivery, unsigned cap, unsigned max_window)
	{
		return delivery && delivery_bytes(cap, max_window) > stdp_bytes() ? delivery_bytes(cap, max_window)
			: stdp_bytes();
	}
};

/* ------------------------------------------------------------ delivery */

/* A delivery block: list the fired rows of its (source tile, delay) pairs,
 * read their row pointers in parallel, list the rows' events in pieces of up
 * to 16, then spread the pieces over groups of 16 lanes, a lane an event and
 * EV_ILP pieces in flight, staging the events in LDS; finally counting-sort the
 * staged events by target tile (relative to the block's window) into the
 * block's bins.
 *
 * The block is a chain of dependent phases (bitmap words, row pointers,
 * events, sort, copy-out), and its length bounds the launch that carries it.
 * So the lists are built with LDS counters in whatever order the waves come
 * (the sums are integer, any order gives the same), where scans over the block
 * took two barriers each and an event its search for the row it belongs to;
 * and a pair is divided into tile and delay once, in 32
 * bits (a pair's number is below tiles * D, at most 2^24).  Measured with the
 * wave sums by DPP (us a step, graphs): 100k neurons x 1000 synapses 18.07 ->
 * 17.14 without STDP, 20.65 -> 19.65 with it; 100k x 400 13.4 -> 12.0; 60k x
 * 600 12.9 -> 11.2.  Pieces of 64, a wave each, were slower than the scans
 * (20.8): rows of 20 to 50 events leave too many lanes idle. */
template<unsigned THREADS, int EV_ILP = EVENT_ILP>
__device__ inline void deliver_block(const nemo_propagate_args& a, uint64_t t, unsigned b, unsigned char* lds)
{
	using Lds = PropagateLds<THREADS>;
	constexpr unsigned ROWS = Lds::ROWS;
	constexpr unsigned PIECES = Lds::PIECES;
	constexpr uint32_t PIECE = Lds::PIECE;
	constexpr unsigned GROUPS = THREADS / PIECE;
	constexpr uint32_t PLACES = (1u << 25) - 1; /* beyond any stage */
	const Lds L(lds, a.bin_capacity, a.max_window);
	int2* stage = L.stage;
	uint32_t* cnt = L.cnt;
	uint32_t* cur = L.cur;

	const unsigned CAP = a.bin_capacity;
	const unsigned D = a.D;
	const unsigned DC = a.d_count;
	const unsigned tid = threadIdx.x;
	const unsigned lane = tid % PIECE;
	const unsigned col = a.block_base + b;
	const size_t parity = t & 1;
	int64_t* acc = a.acc + parity * 2 * a.acc_pitch;
	const uint2 win = a.windows[b];
	const unsigned tlo = win.x;
	const unsigned W = win.y - win.x; /* tiles in the window */
	const uint32_t q0 = a.pair_bounds[b];
	const uint32_t nwords = (a.pair_bounds[b + 1] - q0) * 4;
	for(unsigned p = tid; p < W; p += THREADS) cnt[p] = 0;
	if(tid == 0) *L.fill = 0;

	/* staging of an event at its place: with a count for its tile, or (beyond
	 * capacity or, defensively, outside the window) straight into the
	 * accumulators */
	auto stage_event = [&](int2 ev, uint32_t pos) {
		const uint32_t rel = uint32_t(ev.x) / NEMO_TILE - tlo;
		if(pos < CAP && rel < W) {
			stage[pos] = ev;
			atomicAdd(&cnt[rel], 1u);
		} else {
			if(pos < CAP) stage[pos] = make_int2(-1, 0);
			int64_t* dst = acc + (ev.y >= 0 ? size_t(0) : a.acc_pitch) + uint32_t(ev.x);
			atomicAdd(reinterpret_cast<unsigned long long*>(dst), (unsigned long long)(int64_t)ev.y);
		}
	};

	for(uint32_t wb = 0; wb < nwords; wb += THREADS) {
		/* the bitmap words of this batch, one per thread */
		uint64_t word = 0;
		uint32_t row0 = 0; /* row of the word's first neuron */
		const uint32_t w = wb + tid;
		if(w < nwords) {
			const uint32_t q = q0 + w / 4;
			const uint32_t p = q / DC;
			const uint32_t d = q - p * DC + a.d_first;
			row0 = (p * NEMO_TILE + (w & 3) * 64) * D + (d - 1);
			if(t >= d) word = a.fired_bits[((t - d) & PROPAGATE_RING_MASK) * a.fired_words + size_t(p) * 4 + (w & 3)];
		}
		if(tid == 0) *L.rows = 0;
		__syncthreads();
		const uint32_t fired = uint32_t(__popcll(word));
		const uint32_t mine = wave_append(L.rows, fired);
		for(uint32_t r0 = 0;; r0 += ROWS) {
			/* this chunk's rows */
			uint32_t at = mine;
			for(uint64_t x = word; x; x &= x - 1, ++at) {
				if(at - r0 < ROWS) L.row[at - r0] = row0 + uint32_t(__builtin_ctzll(x)) * D;
			}
			if(tid == 0) *L.pieces = 0;
			__syncthreads();
			const uint32_t R = *L.rows;
			/* a row per thread: its events' pieces and their place */
			uint32_t rb = 0, len = 0;
			if(r0 + tid < R) {
				const size_t row = L.row[tid];
				rb = a.rowptr[row];
				len = a.rowptr[row + 1] - rb;
			}
			const uint32_t np = (len + PIECE - 1) / PIECE;
			const uint32_t first = wave_append(L.pieces, np);
			const uint32_t place = wave_append(L.fill, len);
			for(uint32_t p0 = 0;; p0 += PIECES) {
				/* the pieces of this pass */
				for(uint32_t i = max(first, p0); i < min(first + np, p0 + PIECES); ++i) {
					const uint32_t e = PIECE * (i - first);
					L.piece[i - p0] = make_uint2(rb + e, (min(PIECE, len - e) << 25) | min(PLACES, place + e));
				}
				__syncthreads();
				const uint32_t P = *L.pieces;
				const uint32_t here = min(P - min(P, p0), PIECES);
				for(uint32_t c0 = tid / PIECE; c0 < here; c0 += EV_ILP * GROUPS) {
					int2 ev[EV_ILP];
					uint32_t pos[EV_ILP];
#pragma unroll
					for(int u = 0; u < EV_ILP; ++u) {
						const uint32_t c = c0 + u * GROUPS;
						const uint2 pc = L.piece[min(c, here - 1)];
						const bool live = c < here && lane < (pc.y >> 25);
						pos[u] = live ? (pc.y & PLACES) + lane : ~0u;
						ev[u] = make_int2(0, 0);
						if(live) ev[u] = a.fcm[pc.x + lane];
					}
#pragma unroll
					for(int u = 0; u < EV_ILP; ++u) {
						if(pos[u] != ~0u) stage_event(ev[u], pos[u]);
					}
				}
				if(p0 + PIECES >= P) break;
				__syncthreads(); /* the list is rewritten */
			}
			__syncthreads(); /* the lists are rewritten by the next chunk or batch */
			if(r0 + ROWS >= R) break;
		}
	}
	if(nwords == 0) __syncthreads();
	const uint32_t fill = *L.fill;

	/* counting sort of the staged events by target tile */
	const uint32_t staged = min(fill, CAP);
	uint32_t carry = 0;
	for(uint32_t base = 0; base < W; base += THREADS) {
		const uint32_t p = base + tid;
		const uint32_t c = p < W ? cnt[p] : 0u;
		uint32_t total;
		const uint32_t pre = block_exclusive_scan<THREADS>(c, &total);
		if(p < W) {
			cur[p] = carry + pre;
			a.bin_table[(parity * a.tiles + tlo + p) * a.table_columns + col] = (c << 16) | (carry + pre);
		}
		carry += total;
	}
	__syncthreads();
	int2* out = a.bins + (parity * a.table_columns + col) * CAP;
	if(staged <= SORT_REGS * THREADS) {
		/* every thread holds its staged events in registers, then all write
		 * them back sorted into the stage, which is copied out contiguously */
		int2 e[SORT_REGS];
#pragma unroll
		for(unsigned u = 0; u < SORT_REGS; ++u) {
			const uint32_t i = u * THREADS + tid;
			e[u] = i < staged ? stage[i] : make_int2(-1, 0);
		}
		uint32_t pos[SORT_REGS];
#pragma unroll
		for(unsigned u = 0; u < SORT_REGS; ++u) {
			if(e[u].x >= 0) pos[u] = atomicAdd(&cur[uint32_t(e[u].x) / NEMO_TILE - tlo], 1u);
		}
		__syncthreads();
#pragma unroll
		for(unsigned u = 0; u < SORT_REGS; ++u) {
			if(e[u].x >= 0) stage[pos[u]] = make_int2(int(uint32_t(e[u].x) % NEMO_TILE), e[u].y);
		}
		__syncthreads();
		/* two events per 16-byte store (the stage and every bin region start
		 * 16-byte aligned), the odd last one alone; non-temporal, since the
		 * update reads them on other XCDs */
		typedef int v4i __attribute__((ext_vector_type(4)));
		const uint32_t pairs = carry / 2;
		const v4i* s4 = reinterpret_cast<const v4i*>(stage);
		v4i* o4 = reinterpret_cast<v4i*>(out);
		for(uint32_t i = tid; i < pairs; i += THREADS) __builtin_nontemporal_store(s4[i], &o4[i]);
		if((carry & 1) && tid == 0) out[carry - 1] = stage[carry - 1];
	} else {
		/* four staged events per thread at a time, so that their LDS
		 * atomics (which return the slot) overlap */
		for(uint32_t i0 = tid; i0 < staged; i0 += 4 * THREADS) {
			int2 e[4];
			uint32_t pos[4];
#pragma unroll
			for(int u = 0; u < 4; ++u) {
				const uint32_t i = i0 + u * THREADS;
				e[u] = i < staged ? stage[i] : make_int2(-1, 0);
			}
#pragma unroll
			for(int u = 0; u < 4; ++u) {
				if(e[u].x >= 0) pos[u] = atomicAdd(&cur[uint32_t(e[u].x) / NEMO_TILE - tlo], 1u);
			}
#pragma unroll
			for(int u = 0; u < 4; ++u) {
				if(e[u].x >= 0) out[pos[u]] = make_int2(int(uint32_t(e[u].x) % NEMO_TILE), e[u].y);
			}
		}
	}
	if(tid == 0 && fill) a.block_events[col] += fill;
}

/* ---------------------------------------------------------------- STDP */

/* An STDP block of the STDP-only launch: the targets among its bitmap words
 * that fired P steps before step r, and all their plastic incoming synapses
 * spread evenly over its threads (ILP loads in flight per thread).  The
 * update kernels do the same per tile when STDP runs inside them. */
template<unsigned THREADS>
__device__ inline void stdp_block(const nemo_propagate_args& a, uint64_t r, unsigned sb, unsigned char* lds)
{
	const nemo_hip_stdp& st = a.stdp;
	int32_t* s_fn = reinterpret_cast<int32_t*>(lds);
	uint32_t* s_rb = reinterpret_cast<uint32_t*>(lds + 128 * sizeof(int32_t));
	uint32_t* s_pos = s_rb + THREADS;
	const unsigned P = st.post_window;
	const unsigned tid = threadIdx.x;
	if(tid < 64) {
		s_fn[tid] = st.fn_pre[tid];
		s_fn[64 + tid] = st.fn_post[tid];
	}

	const uint64_t slot = (r - P) & PROPAGATE_RING_MASK;
	const size_t w0 = size_t(sb) * a.stdp_words;
	const size_t word = w0 + tid / 64;
	bool fired = false;
	if(tid / 64 < a.stdp_words && word < a.fired_words) {
		fired = (a.fired_bits[slot * a.fired_words + word] >> (tid & 63)) & 1u;
	}
	uint32_t nfired;
	const uint32_t idx = block_exclusive_scan<THREADS>(fired ? 1u : 0u, &nfired);
	uint32_t len = 0, rb = 0;
	if(fired) {
		const uint32_t n = uint32_t(w0 * 64 + tid);
		rb = st.rcm_ptr[n];
		len = st.rcm_ptr[n + 1] - rb;
	}
	uint32_t total;
	const uint32_t pos = block_exclusive_scan<THREADS>(len, &total);
	if(fired) {
		s_rb[idx] = rb;
		s_pos[idx] = pos;
	}
	if(tid == 0) s_pos[nfired] = total;
	__syncthreads();
	if(total == 0) return;

	const uint64_t* hist = a.hist + NEMO_HIST_INDEX(0, r, a.hist_pitch);
	for(uint32_t e0 = tid; e0 < total; e0 += ILP * THREADS) {
		uint32_t k[ILP];
		uint32_t sd[ILP];
		int32_t acc[ILP];
#pragma unroll
		for(int u = 0; u < ILP; ++u) k[u] = e0 + u * THREADS;
		unsigned lo[ILP];
		last_not_above_k<THREADS>(s_pos, nfired, k, lo);
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
		uint64_t h[ILP];
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			h[u] = 0;
			if(e0 + u * THREADS < total) h[u] = hist[sd[u] & 0x3ffffffu];
		}
#pragma unroll
		for(int u = 0; u < ILP; ++u) {
			if(e0 + u * THREADS < total) {
				const unsigned d = (sd[u] >> 26) + 1;
				const uint64_t preFiring = d >= 64 ? 0 : (h[u] >> d);
				const int32_t dw = stdp_wrap_add(
						stdp_update_region(preFiring & st.potentiation, P, st.pre_post, st.post_pre,
							s_fn, s_fn + 64),
						stdp_update_region(preFiring & st.depression, P, st.pre_post, st.post_pre,
							s_fn, s_fn + 64));
				if(dw != 0) {
					st.rcm_acc[k[u]] = stdp_wrap_add(acc[u], dw);
				}
			}
		}
	}
	if(tid == 0) atomicAdd(&st.examined[sb], (unsigned long long)total);
}

/* Bits [y, y+64) of the 128-bit firing record c | s << n (1 <= n <= 64,
 * y <= 64), where c is a neuron's history after step rl and s its history
 * after step rl - n: bit x of the record is firing at step rl - x, so this is
 * the history after step rl - y. */
__device__ inline uint64_t history_window(uint64_t c, uint64_t s, unsigned n, unsigned y)
{
	const uint64_t lo = c | (n < 64 ? s << n : 0);
	const uint64_t hi = n < 64 ? s >> (64 - n) : s;
	return y == 0 ? lo : y < 64 ? (lo >> y) | (hi << (64 - y)) : hi;
}

/* stdp_update_region of the arrivals that a region has before the spike
 * (after) and behind it (post): a side that the region has not, which most
 * regions have, is a branch that a wave does not take. */
__device__ inline int32_t stdp_update_sides(uint64_t arrivals, uint64_t pre_mask, uint64_t post_mask, unsigned post_window,
		const int32_t* s_fn)
{
	const unsigned NONE = ~0u;
	unsigned dt_pre = NONE, dt_post = NONE;
	if(pre_mask) {
		const uint64_t pre = arrivals & pre_mask;
		if(pre) dt_pre = unsigned(__builtin_ctzll(pre >> post_window));
	}
	if(post_mask) {
		const uint64_t post = arrivals & post_mask;
		if(post) dt_post = unsigned(__builtin_clzll(post << (64 - post_window)));
	}
	if(dt_pre < dt_post) return s_fn[dt_pre];
	if(dt_post < dt_pre) return s_fn[64 + dt_post];
	return 0;
}

/* The listed targets' synapses for all their steps, a wave per target: its
 * steps and row are then the wave's, in scalar registers, and no lane looks up
 * which target its synapse belongs to. */
template<unsigned THREADS, int SYN_ILP>
__device__ inline void stdp_batch_rows(const nemo_hip_stdp& st, const ulonglong2* rec, unsigned cur_slot, unsigned n,
		const int32_t* s_fn, const uint32_t* s_rb, const uint32_t* s_pos, const uint64_t* s_post, uint32_t nfired)
{
	const unsigned lane = threadIdx.x % 64;
	const unsigned P = st.post_window;
	for(unsigned idx = __builtin_amdgcn_readfirstlane(threadIdx.x / 64); idx < nfired; idx += THREADS / 64) {
		const uint32_t rb = __builtin_amdgcn_readfirstlane(s_rb[idx]);
		const uint32_t len = __builtin_amdgcn_readfirstlane(s_pos[idx + 1] - s_pos[idx]);
		const uint64_t steps = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(s_post[idx] >> 32)))) << 32
			| uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(s_post[idx])));
		const uint32_t* sds = st.rcm_sd + rb;
		int32_t* accs = st.rcm_acc + rb;
		for(uint32_t e0 = 0; e0 < len; e0 += SYN_ILP * 64) {
			uint32_t sd[SYN_ILP];
			int32_t acc[SYN_ILP];
#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				const uint32_t e = e0 + u * 64 + lane;
				sd[u] = e < len ? sds[e] : 0u;
				acc[u] = e < len ? accs[e] : 0;
			}
			uint64_t hc[SYN_ILP], hs[SYN_ILP];
#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				const ulonglong2 v = rec[sd[u] & 0x3ffffffu];
				hc[u] = cur_slot ? v.y : v.x;
				hs[u] = cur_slot ? v.x : v.y;
			}
#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				if(e0 + u * 64 >= len) break;
				const unsigned d = (sd[u] >> 26) + 1;
				int32_t dw = 0;
				for(uint64_t m = steps; m; m &= m - 1) {
					const uint64_t h = history_window(hc[u], hs[u], n, unsigned(__builtin_ctzll(m)));
					const uint64_t arrivals = d >= 64 ? 0 : (h >> d);
					dw = stdp_wrap_add(dw, stdp_wrap_add(
							stdp_update_sides(arrivals, st.potentiation & st.pre_post, st.potentiation & st.post_pre, P, s_fn),
							stdp_update_sides(arrivals, st.depression & st.pre_post, st.depression & st.post_pre, P, s_fn)));
				}
				const uint32_t e = e0 + u * 64 + lane;
				if(dw != 0 && e < len) accs[e] = stdp_wrap_add(acc[u], dw);
			}
		}
	}
}

/* The pending STDP accumulation (clock->stdp_first, stdp_count: 1..64
 * steps r0 .. rl) for the targets of block sb's bitmap words, from the two
 * history snapshots only: after rl (slot stdp_snaps % 2 of stdp_snap) and
 * after r0 - 1 (the other slot).  Together they hold every neuron's firing
 * over the 128 steps the n accumulations look at: a target fired at step
 * r - P when bit rl - r + P of its record is set, and a source's history
 * after step r is the window of its record at rl - r.  Each thread owns a
 * synapse for all the steps, so the accumulator is read and written once per
 * batch and no two threads touch it; the sum of 32-bit wrap-around additions
 * does not depend on their order, so the result equals n single-step
 * accumulations.  Nothing here reads the live history, so the batch may run
 * beside the steps that follow. */
template<unsigned THREADS, int SYN_ILP = STDP_BATCH_ILP>
__device__ inline void stdp_batch_block(const nemo_propagate_args& a, unsigned sb, unsigned char* lds)
{
	const uint64_t r0 = a.clock->stdp_first;
	const unsigned n = unsigned(a.clock->stdp_count);
	const unsigned cur_slot = unsigned(a.clock->stdp_snaps & 1);
	if(n == 0 || n > 64) return;
	const nemo_hip_stdp& st = a.stdp;
	int32_t* s_fn = reinterpret_cast<int32_t*>(lds);
	uint32_t* s_rb = reinterpret_cast<uint32_t*>(lds + 128 * sizeof(int32_t));
	uint32_t* s_pos = s_rb + THREADS;
	uint64_t* s_post = reinterpret_cast<uint64_t*>(s_pos + THREADS + 2);
	const unsigned P = st.post_window;
	const unsigned tid = threadIdx.x;
	if(tid < 64) {
		s_fn[tid] = st.fn_pre[tid];
		s_fn[64 + tid] = st.fn_post[tid];
	}
	const uint64_t rl = r0 + n - 1;
	/* the two snapshots, after rl and after r0 - 1: one 16-byte load per
	 * neuron */
	const ulonglong2* rec = reinterpret_cast<const ulonglong2*>(a.stdp_snap);
	auto split = [cur_slot](const ulonglong2 v, uint64_t& cur, uint64_t& old) {
		cur = cur_slot ? v.y : v.x;
		old = cur_slot ? v.x : v.y;
	};
	/* bit y: step rl - y is accumulated (in the batch, r >= P, not flushed) */
	uint64_t due = n >= 64 ? ~uint64_t(0) : (uint64_t(1) << n) - 1;
	if(rl < P) {
		due = 0;
	} else if(rl - P < 63) {
		due &= (uint64_t(2) << (rl - P)) - 1;
	}
	const uint64_t flushed = a.clock->stdp_flushed;
	if(flushed >= r0 && flushed <= rl) due &= ~(uint64_t(1) << (rl - flushed));

	/* the block's words, THREADS / 64 (one target per thread) at a time */
	unsigned long long examined_all = 0;
	for(unsigned wg = 0; wg < a.stdp_words; wg += THREADS / 64) {
		__syncthreads(); /* the previous group is done with the LDS lists */
		const size_t w0 = size_t(sb) * a.stdp_words + wg;
		const size_t word = w0 + tid / 64;
		uint64_t post = 0; /* bit y: the target fired at step rl - y - P */
		if(tid / 64 < min(THREADS / 64, a.stdp_words - wg) && word < a.fired_words) {
			const uint32_t tn = uint32_t(w0 * 64 + tid);
			uint64_t c, o;
			split(rec[tn], c, o);
			post = history_window(c, o, n, P) & due;
		}
		const bool fired = post != 0;
		uint32_t nfired;
		const uint32_t idx = block_exclusive_scan<THREADS>(fired ? 1u : 0u, &nfired);
		uint32_t len = 0, rb = 0;
		if(fired) {
			const uint32_t tn = uint32_t(w0 * 64 + tid);
			rb = st.rcm_ptr[tn];
			len = st.rcm_ptr[tn + 1] - rb;
		}
		uint32_t total;
		const uint32_t pos = block_exclusive_scan<THREADS>(len, &total);
		uint32_t examined;
		block_exclusive_scan<THREADS>(len * unsigned(__popcll(post)), &examined);
		examined_all += examined;
		if(fired) {
			s_rb[idx] = rb;
			s_pos[idx] = pos;
			s_post[idx] = post;
		}
		if(tid == 0) s_pos[nfired] = total;
		__syncthreads();
		if(total == 0) continue;

		if(a.stdp_rows && total >= STDP_WAVE_ROW * nfired) {
			stdp_batch_rows<THREADS, SYN_ILP>(st, rec, cur_slot, n, s_fn, s_rb, s_pos, s_post, nfired);
			continue;
		}
		for(uint32_t e0 = tid; e0 < total; e0 += SYN_ILP * THREADS) {
			uint32_t k[SYN_ILP];
			uint32_t sd[SYN_ILP];
			int32_t acc[SYN_ILP];
			uint64_t pm[SYN_ILP];
	#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) k[u] = e0 + u * THREADS;
			unsigned lo[SYN_ILP];
			last_not_above_k<THREADS>(s_pos, nfired, k, lo);
	#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				const uint32_t e = k[u];
				k[u] = 0;
				sd[u] = 0;
				acc[u] = 0;
				pm[u] = 0;
				if(e < total) {
					k[u] = s_rb[lo[u]] + (e - s_pos[lo[u]]);
					pm[u] = s_post[lo[u]];
					sd[u] = st.rcm_sd[k[u]];
					acc[u] = st.rcm_acc[k[u]];
				}
			}
			uint64_t hc[SYN_ILP], hs[SYN_ILP];
	#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				hc[u] = 0;
				hs[u] = 0;
				if(e0 + u * THREADS < total) {
					split(rec[sd[u] & 0x3ffffffu], hc[u], hs[u]);
				}
			}
	#pragma unroll
			for(int u = 0; u < SYN_ILP; ++u) {
				if(e0 + u * THREADS < total) {
					const unsigned d = (sd[u] >> 26) + 1;
					int32_t dw = 0;
					for(uint64_t m = pm[u]; m; m &= m - 1) {
						const unsigned y = unsigned(__builtin_ctzll(m));
						const uint64_t h = history_window(hc[u], hs[u], n, y);
						const uint64_t preFiring = d >= 64 ? 0 : (h >> d);
						dw = stdp_wrap_add(dw, stdp_wrap_add(
								stdp_update_region(preFiring & st.potentiation, P, st.pre_post, st.post_pre,
									s_fn, s_fn + 64),
								stdp_update_region(preFiring & st.depression, P, st.pre_post, st.post_pre,
									s_fn, s_fn + 64)));
					}
					if(dw != 0) {
						st.rcm_acc[k[u]] = stdp_wrap_add(acc[u], dw);
					}
				}
			}
		}
	}
	if(tid == 0) atomicAdd(&st.examined[sb], examined_all);
}

/* STDP accumulation of step t-1 by STDP block sb, unless it is not due */
template<unsigned THREADS>
__device__ inline void stdp_step(const nemo_propagate_args& a, uint64_t t, unsigned sb, unsigned char* lds)
{
	if(t == 0) return;
	const uint64_t r = t - 1;
	if(r == a.clock->stdp_flushed || r < a.stdp.post_window) return;
	stdp_block<THREADS>(a, r, sb, lds);
}


/* In an update launch of NEMO_COLAUNCH_BLOCK threads per block: run this
 * block as one of the propagate blocks the launch carries after the group's
 * tiles (nemo_hip_colaunch) and return true, or, in a block of the group's
 * own tiles, return false for its first NEMO_TILE threads (the tile's) and,
 * for the others, true (their waves then end; a block barrier waits only for
 * the waves still running) or, with GATHER_HELPERS, false: the kernel then
 * passes them to gather_input<NEMO_COLAUNCH_BLOCK>, which releases them.
 * Every update kernel of such a launch calls it first and returns when it
 * returns true. */
template<bool GATHER_HELPERS = false>
__device__ inline bool colaunched_block(const nemo_hip_step_buffers& b, const nemo_hip_neuron_group& g)
{
	static_assert(NEMO_COLAUNCH_BLOCK % 64 == 0 && NEMO_COLAUNCH_BLOCK >= NEMO_TILE, "whole waves beyond the tile");
	const unsigned tiles = (g.count + NEMO_TILE - 1) / NEMO_TILE;
	if(blockIdx.x < tiles) return !GATHER_HELPERS && threadIdx.x >= NEMO_TILE;
	extern __shared__ uint64_t colaunch_lds[];
	unsigned char* lds = reinterpret_cast<unsigned char*>(colaunch_lds);
	const unsigned k = blockIdx.x - tiles;
	const nemo_propagate_args& a = b.co.args;
	const uint64_t t = clock_base(a.clock) + a.step_offset;
	if(k < b.co.deliver_blocks) {
		deliver_block<NEMO_COLAUNCH_BLOCK, CARRIED_EVENT_ILP>(a, t, k, lds);
	} else {
		stdp_step<NEMO_COLAUNCH_BLOCK>(a, t - 1, k - b.co.deliver_blocks, lds);
	}
	return true;
}

} // namespace nemo_dev

#endif
