/*
 * Launch interface of the float-weight mode kernels (float_mode.hip): plain
 * C ABI, device pointers, sizes and a stream; each returns the launch status.
 */
#ifndef NEMO_AMD_FLOAT_MODE_H
#define NEMO_AMD_FLOAT_MODE_H

#include <stddef.h>
#include <stdint.h>
#include <hip/hip_runtime_api.h>

#ifdef __cplusplus
extern "C" {
#endif

/* One forward step t of the float-weight network (all N neurons). */
typedef struct nemo_float_step_args {
	unsigned n;                /* neurons */
	unsigned t;                /* step */
	const uint32_t* rcm_ptr;   /* n+1 offsets of each target's incoming synapses */
	const uint32_t* rcm_sd;    /* source | (delay-1) << 26 */
	const float* wr;           /* weights in reverse-matrix order */
	const float* pa;           /* Izhikevich a, b, c, d per neuron */
	const float* pb;
	const float* pc;
	const float* pd;
	const float* x;            /* [T][n] external current */
	float* S;                  /* [T][n] spikes (written at t when store) */
	float* V;                  /* [T][n] membrane potential after the step (store) */
	double* v;                 /* [n] state, updated */
	double* u;
	int store;                 /* write S[t], V[t] and the bitmap of step t */
	double* ckpt;              /* NULL, or [ceil(T/K)][2][n]: (v, u) before every K-th step */
	unsigned K;
	uint32_t* bits;            /* [T][pitch] spike bitmaps (read for t-d, written at t when store) */
	unsigned pitch;            /* words per step, nemo_float_bitmap_pitch(n) or more, a multiple of 4 */
	unsigned dmax;             /* longest delay */
	int stage;                 /* stage the last dmax bitmaps in LDS; needs nemo_float_stage_bytes
	                              of at most NEMO_FLOAT_STAGE_MAX */
	const uint32_t* slice_ptr; /* with stage, or NULL: [ceil(n / 8) + 1] offsets of eight targets'
	                              synapses, in lines of 64 x 4, and the synapses in that order,
	                              as wr is then: source | (dmax - delay) << 26 */
	const uint32_t* slice_sd;
} nemo_float_step_args;

/* The static workspace of the allocation-free forward: a file-scope device
 * array of NEMO_FLOAT_SCRATCH_BYTES, one per device (each device holds it
 * until the process ends).  Its address on the current device, looked up
 * once per device (with hipGetSymbolAddress, the only valid device address
 * of the array in host code); devices numbered below
 * NEMO_FLOAT_SCRATCH_DEVICES. */
#define NEMO_FLOAT_SCRATCH_BYTES (64u << 20)
#define NEMO_FLOAT_SCRATCH_DEVICES 64
hipError_t nemo_float_scratch(void** ptr, size_t* bytes);

/* Largest LDS stage of spike bitmaps a forward block takes. */
#define NEMO_FLOAT_STAGE_MAX 49152
unsigned nemo_float_bitmap_pitch(unsigned n);
size_t nemo_float_stage_bytes(unsigned n, unsigned dmax);

/* Replay of forward steps t0..t1-1 from the state before t0 and the
 * recorded spikes (as firing histories): each step's entry state and input,
 * equal to the forward's. */
typedef struct nemo_float_replay_args {
	unsigned n;
	unsigned t0, t1;
	unsigned dmax;             /* longest delay, at most 64 */
	const uint32_t* rcm_ptr;
	const uint32_t* rcm_sd;
	const float* wr;
	const float* pa;
	const float* pb;
	const float* pc;
	const float* pd;
	const float* x;            /* [T][n] */
	const uint64_t* hist;      /* [hist_rows][n] from nemo_launch_pack_history */
	unsigned hist_rows;
	const double* v0;          /* [n] state before t0 */
	const double* u0;
	double* seg_v;             /* [t1 - t0][n] entry state and input of each step */
	double* seg_u;
	double* seg_I;
	const uint32_t* slice_ptr; /* as nemo_float_step_args, or NULL; needs n of at most */
	const uint32_t* slice_sd;  /* NEMO_FLOAT_REPLAY_MAX and dmax below 58 */
} nemo_float_replay_args;
#define NEMO_FLOAT_REPLAY_MAX 20480u

hipError_t nemo_launch_float_replay(hipStream_t, const nemo_float_replay_args*);
/* rows of the firing histories of a T-step run */
unsigned nemo_float_history_rows(unsigned T);
/* hist[r][j], bit k: neuron j fired at step 64 (r - 1) + k (S [T][n]); row 0
 * and steps from T on are zero */
hipError_t nemo_launch_pack_history(hipStream_t, uint64_t* hist, unsigned rows, const float* S, unsigned n,
		unsigned T);
/* One backward step t (in decreasing t) of the adjoint. */
typedef struct nemo_float_back_args {
	unsigned n;
	unsigned t;
	unsigned T;                /* steps of the forward run */
	unsigned ring;             /* slots of LI (max delay + 1) */
	const uint32_t* fcm_ptr;   /* n+1 offsets of each source's synapses */
	const uint32_t* fcm_td;    /* target | (delay-1) << 26 */
	const float* wf;           /* weights in forward-matrix order */
	const float* pa;
	const float* pb;
	const float* pc;
	const float* pd;
	const float* S;            /* [T][n] forward spikes */
	const float* gS;           /* [T][n] dL/dS, or NULL */
	const float* gV;           /* [T][n] dL/dV, or NULL */
	unsigned t0;               /* first step of the recorded segment */
	const double* seg_v;       /* recorded entry state and input of the segment */
	const double* seg_u;
	const double* seg_I;
	double* LV;                /* [n] dL/dv of the state after step t; becomes the one before */
	double* LU;
	double* LI;                /* [ring][n] dL/dI of recent steps */
	float* gw;                 /* [synapses] dL/dw in forward-matrix order, accumulated */
	float* ga;                 /* [n] accumulated */
	float* gb;
	float* gd;
	float* gx;                 /* [T][n] dL/dx, or NULL */
} nemo_float_back_args;

/* The same for networks of up to NEMO_FLOAT_PUSH_MAX neurons whose input
 * adjoints of one step fit in LDS. */
#define NEMO_FLOAT_PUSH_MAX 65536
#define NEMO_FLOAT_PUSH_LDS (160u << 10)
/* What a lane of a slice passes: synapses of a neuron of the block with one
 * delay (0: none) */
typedef struct nemo_float_row {
	uint16_t neuron, delay;
} nemo_float_row;
typedef struct nemo_float_push_args {
	unsigned n;
	unsigned t;
	unsigned T;
	unsigned t0;               /* as nemo_float_back_args */
	unsigned dmax;             /* longest delay */
	unsigned tile;             /* neurons per block; (pitch + 2 + tile) doubles fit NEMO_FLOAT_PUSH_LDS */
	unsigned pitch;            /* nemo_float_push_pitch(n) */
	unsigned lanes;            /* per row: 1, 2, 4, 8, 16 or 32 */
	unsigned slices;           /* per block, of 64 / lanes rows */
	const uint32_t* slice_ptr; /* [blocks * slices + 1] offsets of their synapses, in lines of 64 x 4 */
	const nemo_float_row* rows;  /* [blocks * slices][64] the row of each lane */
	const uint16_t* row_target; /* [lines][64][4], pitch where there is no synapse */
	const float* row_w;        /* weights in that order */
	float* row_gw;             /* dL/dw in that order, accumulated */
	const float* pa;
	const float* pb;
	const float* S;
	const float* gS;
	const float* gV;
	const double* seg_v;
	const double* seg_u;
	const double* seg_I;
	double* LV;
	double* LU;
	double* LI;                /* [2][pitch] dL/dI of this step and the next */
	double* ring;              /* [dmax][n] spike adjoints of the steps before */
	float* ga;
	float* gb;
	float* gd;
	float* gx;
} nemo_float_push_args;

unsigned nemo_float_push_pitch(unsigned n);
/* allows the LDS of the staged kernels on the current device; once before
 * their launches */
hipError_t nemo_float_staged_attributes();
hipError_t nemo_launch_float_push_step(hipStream_t, const nemo_float_push_args*);

hipError_t nemo_launch_float_forward_step(hipStream_t, const nemo_float_step_args*);
hipError_t nemo_launch_float_backward_step(hipStream_t, const nemo_float_back_args*);

/* wr[k] = w[user[k]] in the slices' order, 0 where that is no synapse; lines:
 * of the longest slice */
hipError_t nemo_launch_float_slice_weights(hipStream_t, float* wr, const float* w, const uint32_t* user,
		const uint32_t* slice_ptr, unsigned slices, unsigned lines, size_t synapses);

/* The synapses' places in the slices (slice_sd zero and slice_user all ones
 * before). */
typedef struct nemo_float_slice_args {
	unsigned n, dmax;
	size_t synapses;
	const uint32_t* rcm_ptr;
	const uint32_t* rcm_sd;
	const uint32_t* rcm_user;
	const uint32_t* slice_ptr;
	uint32_t* slice_sd;
	uint32_t* slice_user;
} nemo_float_slice_args;
hipError_t nemo_launch_float_fill_slices(hipStream_t, const nemo_float_slice_args*);

/* The synapses' places in the rows of the backward (row_user all ones and
 * row_target the pitch before). */
typedef struct nemo_float_rows_args {
	unsigned n, dmax, lanes;
	const uint32_t* fcm_ptr;
	const uint32_t* fcm_td;
	const uint32_t* row_at;    /* [n * dmax] */
	uint32_t* row_user;
	uint16_t* row_target;
} nemo_float_rows_args;
hipError_t nemo_launch_float_fill_rows(hipStream_t, const nemo_float_rows_args*);

/* wr[k] = w[wr_user[k]] for the first wr_entries; v, u = v0, u0 */
typedef struct nemo_float_begin_forward_args {
	size_t n, synapses, wr_entries;
	const float* w;
	const uint32_t* wr_user;
	float* wr;
	const float* v0;
	const float* u0;
	double* v;
	double* u;
} nemo_float_begin_forward_args;
hipError_t nemo_launch_float_begin_forward(hipStream_t, const nemo_float_begin_forward_args*);

/* wr[k] = w[wr_user[k]]; row_w[k] = w[row_user[k]] (0 where row_user is no
 * synapse) and row_gw zero for the entries, gw zero without any; the rest zero */
typedef struct nemo_float_begin_backward_args {
	size_t n, synapses, wr_entries, entries, li; /* li: doubles of LI */
	const float* w;
	const uint32_t* wr_user;
	float* wr;
	const uint32_t* row_user;
	float* row_w;
	float* row_gw;
	double* LI;
	double* LV;
	double* LU;
	float* gw;
	float* ga;
	float* gb;
	float* gd;
} nemo_float_begin_backward_args;
hipError_t nemo_launch_float_begin_backward(hipStream_t, const nemo_float_begin_backward_args*);
/* gw[row_user[k]] = row_gw[k] for the entries that are synapses; gv0, gu0 = LV, LU as
 * floats, each unless NULL */
typedef struct nemo_float_end_backward_args {
	size_t n, synapses, entries;
	const uint32_t* row_user;
	const float* row_gw;
	float* gw;
	const double* LV;
	const double* LU;
	float* gv0;
	float* gu0;
} nemo_float_end_backward_args;
hipError_t nemo_launch_float_end_backward(hipStream_t, const nemo_float_end_backward_args*);

#ifdef __cplusplus
}
#endif

#endif
