/*
 * Launch interface of the backend's own kernels (kernels.hip).  Plain C ABI:
 * device pointers, sizes and a stream; each returns the launch status.  These
 * replace the CUDA backend's launch wrappers (src/nemo/cuda/kernel.hpp:35-116).
 */
#ifndef NEMO_AMD_KERNELS_H
#define NEMO_AMD_KERNELS_H

#include <stddef.h>
#include <stdint.h>
#include <hip/hip_runtime_api.h>

#include "nemo_hip_plugin.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Longest supported synaptic delay (ms); the firing-history word is 64 bits. */
#define NEMO_MAX_DELAY 64
/* Threads per block of the backend's small kernels. */
#define NEMO_BLOCK 256
/* Threads per block of the propagate launches (delivery and STDP blocks):
 * one block per CU at a time does most of a step's delivery, so it gets
 * several waves per SIMD to hide LDS and memory latency. */
#ifndef NEMO_PROPAGATE_BLOCK
#define NEMO_PROPAGATE_BLOCK 512
#endif
/* Firing-bitmap words (64 targets each) an STDP block may cover: one target
 * per thread, or, in STDP batches, groups of that many in turn. */
#define NEMO_STDP_MAX_WORDS (NEMO_PROPAGATE_BLOCK / 64)
#define NEMO_STDP_BATCH_MAX_WORDS 64
/* Threads per STDP batch block, and the waves per SIMD its registers allow
 * (80 VGPRs): one wave per SIMD, which fits beside three blocks of an update
 * launch that carries delivery (NEMO_COLAUNCH_WAVES), so that a batch running
 * beside the steps does not take their blocks' places. */
#define NEMO_STDP_BATCH_BLOCK 256
#define NEMO_STDP_BATCH_WAVES 6
/* Default bitmap words per batch block: 261 blocks for 100k neurons, about
 * one per CU (100k x 1000 with STDP, us per step in one box: 4 words 23.2,
 * 5 words 22.4, 6 words 22.1, 7 words 22.2, 8 words 22.6) */
#define NEMO_STDP_BATCH_WORDS 6


/* A kernel's word to the host that what it wrote to pinned memory is there:
 * value into flag (pinned), by the last of its blocks; blocks (device memory,
 * 0 before and after) counts them.  The host sees it 7 us after a launch on an
 * idle stream, where hipStreamSynchronize returns after 13 and a polled
 * hipStreamQuery after 24. */
typedef struct nemo_host_signal {
	uint64_t* flag; /* NULL: no signal (where a kernel allows it) */
	uint64_t value;
	unsigned* blocks;
} nemo_host_signal;

/* dynamic LDS bytes a delivery block needs */
size_t nemo_propagate_lds_bytes(unsigned max_window, unsigned bin_capacity);
/* The pending STDP accumulation (clock->stdp_first, stdp_count) in one launch
 * of stdp_blocks blocks, from the two history snapshots.  It reads neither
 * the live history nor the bitmaps, so it may run beside later steps. */
hipError_t nemo_launch_stdp_batch(hipStream_t, const nemo_propagate_args*, unsigned stdp_blocks);
/* The same as a flush: afterwards nothing is pending and clock->stdp_flushed
 * is step base + offset (set by a kernel after the batch, so that no copy
 * from the host follows it) */
hipError_t nemo_launch_stdp_flush(hipStream_t, const nemo_propagate_args*, unsigned stdp_blocks, uint64_t offset);
/* A snapshot of the history after step base + offset (at most 64 steps after
 * the last one); the steps since the last snapshot become the pending
 * accumulation.  The pending batch must have run.  Then the clock's step
 * base moves on by advance (0: it stays). */
hipError_t nemo_launch_stdp_snapshot(hipStream_t, const nemo_propagate_args*, uint64_t offset, uint64_t advance);
/* dynamic LDS an update launch carrying propagate blocks needs (delivery
 * blocks when delivery is set, else STDP blocks only; the launch's update
 * blocks share the buffer) */
size_t nemo_colaunch_lds_bytes(unsigned max_window, unsigned bin_capacity, int delivery);
/* Static LDS of the propagate kernel (bytes). */
size_t nemo_propagate_static_lds(void);
/* Delivery (a->deliver_blocks blocks; none if 0) and STDP accumulation
 * (stdp_blocks blocks; none if 0): one launch with the STDP blocks after the
 * delivery blocks when fuse_stdp is set, else the STDP launch first.  start
 * and stop (may be NULL) are recorded at the start of the first kernel and
 * the end of the last. */
hipError_t nemo_launch_propagate(hipStream_t, const nemo_propagate_args*, unsigned stdp_blocks, int fuse_stdp,
		hipEvent_t start, hipEvent_t stop);

/* Both delivery sets of one step (a's blocks, then a2's; the same step,
 * clock, bin capacity, window and table) in one launch, with stdp_blocks STDP
 * blocks of a's arguments after them. */
hipError_t nemo_launch_propagate_sets(hipStream_t, const nemo_propagate_args* a, const nemo_propagate_args* a2,
		unsigned stdp_blocks, hipEvent_t start, hipEvent_t stop);

/* applyStdp (ConnectivityMatrix::applyStdp, ConnectivityMatrix.cpp:272-325 and
 * StdpProcess::updatedWeight, StdpProcess.cpp:128-138). */
typedef struct nemo_apply_args {
	const uint32_t* rcm_of;          /* per FCM synapse: its accumulator index (in tile, if any), or ~0 if static */
	int32_t* rcm_acc;
	int32_t* tile;                   /* accumulators by FCM synapse / NEMO_APPLY_TILE, or NULL */
	const uint32_t* rcm_tile;        /* with tile: per accumulator, its place there */
	int2* fcm;
	size_t count;                    /* plastic synapses */
	size_t fcm_count;                /* FCM synapses */
	int32_t reward;                  /* Q11.20 reward; 0 clears without adding */
	int32_t minE, maxE, minI, maxI;
	unsigned fbits;
} nemo_apply_args;

#define NEMO_APPLY_TILE (1u << 19)
hipError_t nemo_launch_apply_stdp(hipStream_t, const nemo_apply_args*);
/* rcm_of (fcm_count entries) and rcm_tile (count entries) for an applyStdp
 * with tiles of fcm_count entries in all; used: an entry per tile. */
hipError_t nemo_launch_assign_tiles(hipStream_t, const uint32_t* rcm_fwd, uint32_t* rcm_of, uint32_t* rcm_tile,
		uint32_t* used, size_t count, size_t fcm_count);
/* rcm_of (fcm_count entries): the accumulator index of every plastic
 * synapse, ~0 for the others, from rcm_fwd (count entries). */
hipError_t nemo_launch_invert_rcm(hipStream_t, const uint32_t* rcm_fwd, uint32_t* rcm_of, size_t count,
		size_t fcm_count);

/* Firing of step base_step + step_offset given from outside (one flag per
 * neuron in simulation order, or, flags NULL, a bit per device index, cleared
 * afterwards; dev_to_sim maps device index -> simulation index, ~0 for
 * padding): histories and the step's bitmap written as by an
 * update, and, with direct delivery, the events an update would deliver. */
hipError_t nemo_launch_external_fire(hipStream_t, const nemo_hip_step_buffers* b, const uint32_t* flags, uint32_t* bits,
		const uint32_t* dev_to_sim, unsigned tiles);
/* The ring of a directly delivered network set up from the firing of the
 * steps before t0 (its bitmaps) and the present weights: cleared, then the
 * events of every firing of the last D steps that arrive from t0 on, without
 * those that the update of step t0 delivers. */
hipError_t nemo_launch_direct_rebuild(hipStream_t, const nemo_hip_direct* r, size_t acc_pitch, const uint32_t* rowptr,
		unsigned D, const uint64_t* fired_bits, size_t fired_words, uint64_t t0);
/* Synaptic input of step base_step + step_offset gathered per tile (overflow
 * accumulators cleared; with direct delivery, the slot of the step before it
 * cleared, which no update has read) and written as floats in simulation
 * order. */
hipError_t nemo_launch_gather_currents(hipStream_t, const nemo_hip_step_buffers* b, const uint32_t* dev_to_sim,
		float* E, float* I, unsigned tiles, const nemo_host_signal* done);

/* Firing readout of the k steps from clock base + offset on (their
 * firing-bitmap ring slots, words words each) into pinned host memory: for
 * step t, slot t % NEMO_STEP_RING, counts[slot] the neurons fired and
 * list[slot * room ..] the first room of them in ascending device index, as
 * index's entries (NULL: device indices).  Then the flag is set to done.value
 * + base + offset. */
hipError_t nemo_launch_fired_readout(hipStream_t, const nemo_hip_clock* clock, uint64_t offset, unsigned k,
		const uint64_t* bits, size_t words, const uint32_t* index, uint32_t* counts, uint32_t* list, unsigned room,
		const nemo_host_signal* done);
/* *sum = the total of the n counters (sum in pinned host memory) */
hipError_t nemo_launch_sum_counters(hipStream_t, const unsigned long long* counters, size_t n, uint64_t* sum,
		const nemo_host_signal* done);

/* The stimulus of a step: bits set for the nf device indices fidx, ext[iidx[i]]
 * = ival[i] (distinct indices); the lists may be pinned host memory. */
hipError_t nemo_launch_stimulus(hipStream_t, uint32_t* bits, const uint32_t* fidx, size_t nf, float* ext,
		const uint32_t* iidx, const float* ival, size_t ni);
/* After the step: its firing bitmap copied to out (pinned host memory), and
 * the words of the firing stimulus cleared. */
hipError_t nemo_launch_step_readout(hipStream_t, const uint64_t* fired, uint64_t* out, size_t words, uint32_t* bits,
		const uint32_t* fidx, size_t nf, const nemo_host_signal* done);
/* out[i] = *src[i] (src and out pinned host memory) */
hipError_t nemo_launch_read_values(hipStream_t, const float* const* src, float* out, size_t n,
		const nemo_host_signal* done);
/* clock->base_step += steps */
hipError_t nemo_launch_advance_clock(hipStream_t, nemo_hip_clock* clock, uint64_t steps);

/* Device logf (fn 0), sinf (fn 1) or expf (fn 2) of n inputs (diagnostics). */
hipError_t nemo_launch_eval_math(hipStream_t, int fn, const float* in, float* out, size_t n);

#ifdef __cplusplus
}
#endif

#endif
