/*
 * Float-weight mode and its adjoint: the Izhikevich network with FP32
 * weights and FP32 current sums, differentiable through a surrogate of the
 * spike threshold.  No counterpart in the reference (its plain mode is the
 * fixed-point one, src/nemo/cpu/Simulation.cpp:259-308 and
 * src/nemo/cpu/plugins/Izhikevich.cpp:14-98, whose neuron step this mode
 * keeps).
 *
 * Model, per 1 ms step t and neuron j (weights in float; their sum, the
 * state v, u and all adjoint quantities in double):
 *   I    = x[t][j] + sum over synapses (i -> j, delay d, weight w) of w * S[t-d][i]
 *   4 substeps k (h = 0.25), each only while the neuron has not crossed 30 mV
 *   in an earlier substep (mask m_k):
 *     v <- v + h (0.04 v^2 + 5 v + 140 - u + I)
 *     u <- u + h a (b v - u)                                (new v)
 *   S[t][j] = H(v - 30);  v <- v + S (c - v);  u <- u + S d;  V[t][j] = v
 * Backward: reverse-mode through the same expression, with the masks m_k and
 * the spike value in the reset held constant (the reset is not
 * differentiated through the threshold), and dH/dv replaced by the
 * fast-sigmoid surrogate 1 / (1 + 10 |v - 30|)^2 where S feeds the synapses
 * and the loss.
 *
 * Layout: neurons 0..N-1; the forward matrix holds each source's synapses
 * (all delays) contiguously, fcm_td = target | (delay-1) << 26; the reverse
 * matrix holds each target's incoming synapses, rcm_sd = source | (delay-1)
 * << 26.  Weights are gathered per call into both orders.  S, V, x and the
 * gradients are [T][N] row-major float.
 *
 * A group of lanes per neuron: they stride over the neuron's synapses, a
 * fixed butterfly sums them (so results do not depend on scheduling), the
 * group's first lane does the neuron arithmetic.  The forward step tests a
 * synapse's spike in a bitmap of recent steps ([T][pitch] words, bit j of
 * step t set when neuron j fired), which each block stages in LDS when the
 * last dmax steps' bitmaps are small.  Networks whose spikes and adjoints fit
 * in LDS have their synapses a second time, in the order in which the waves
 * of the staged kernels read them (forward_sliced_kernel,
 * replay_sliced_kernel, backward_push_kernel); the others, and those that
 * this order would fill with empty places, take the general kernels.
 */
#include <hip/hip_runtime.h>

#include <mutex>

#include "float_mode.h"

namespace {

/* Backward: LANES lanes per neuron, BLOCK threads per block. */
constexpr unsigned BLOCK = 256;
#ifndef NEMO_FLOAT_LANES
#define NEMO_FLOAT_LANES 32
#endif
constexpr unsigned LANES = NEMO_FLOAT_LANES;
constexpr unsigned GROUPS = BLOCK / LANES;
static_assert(LANES >= 8 && LANES <= 64 && (LANES & (LANES - 1)) == 0, "LANES: a power of two, 8..64");
/* Forward: FLANES lanes per neuron and 32 neurons per block, so that a
 * block's spikes make one word of the spike bitmap. */
#ifndef NEMO_FLOAT_FWD_LANES
#define NEMO_FLOAT_FWD_LANES 32
#endif
constexpr unsigned FLANES = NEMO_FLOAT_FWD_LANES;
constexpr unsigned FGROUPS = 32;
constexpr unsigned FBLOCK = FGROUPS * FLANES;
static_assert(FLANES >= 8 && FLANES <= 32 && (FLANES & (FLANES - 1)) == 0, "FLANES: a power of two, 8..32");
constexpr unsigned PUSH_BLOCK = 1024;
constexpr uint32_t IDX_MASK = 0x3ffffffu;
constexpr double H = 0.25;
/* synapses in flight per lane */
template<unsigned L> constexpr unsigned unroll_for() { return L >= 16 ? 256 / L : 16; }

/* x of the partner lane under a DPP control (one 32-bit half at a time):
 * quad_perm [1,0,3,2] pairs lanes 4k+0/1 and 4k+2/3, [2,3,0,1] pairs 4k+0/2
 * and 4k+1/3, row_half_mirror pairs i and 7-i in each 8, row_mirror pairs i
 * and 15-i in each 16. */
template<int CTRL>
__device__ inline double dpp_partner(double x)
{
	const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
	const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
	return __hiloint2double(hi, lo);
}
constexpr int DPP_QUAD_1032 = 0xb1;
constexpr int DPP_QUAD_2301 = 0x4e;
constexpr int DPP_ROW_HALF_MIRROR = 0x141;
constexpr int DPP_ROW_MIRROR = 0x140;

/* Sum over groups of L consecutive lanes (L a power of two up to 64), the
 * same fixed pairing in every call: within quads, eights and rows of 16 by
 * DPP, across rows by shuffles.  The first lane of a group (the one that
 * reads it) always adds in the same order, so a sum is reproducible bit for
 * bit. */
template<unsigned L>
__device__ inline double group_sum(double x)
{
	static_assert(L >= 1 && L <= 64 && (L & (L - 1)) == 0, "L: a power of two up to 64");
	if(L > 1) x += dpp_partner<DPP_QUAD_1032>(x);
	if(L > 2) x += dpp_partner<DPP_QUAD_2301>(x);
	if(L > 4) x += dpp_partner<DPP_ROW_HALF_MIRROR>(x);
	if(L > 8) x += dpp_partner<DPP_ROW_MIRROR>(x);
	if(L > 16) x += __shfl_xor(x, 16);
	if(L > 32) x += __shfl_xor(x, 32);
	return x;
}

__device__ inline double surrogate(double v)
{
	const double z = 1.0 + 10.0 * fabs(v - 30.0);
	return 1.0 / (z * z);
}

/* One step of the neuron from (v, u) with input I: four substeps while
 * v < 30, then the reset; returns the spike.  The forward and the replay
 * share it, so that the replay reproduces the forward's state exactly. */
__device__ inline bool neuron_step(double& v, double& u, double I, double A, double B, float C, float D)
{
	bool m = true;
#pragma unroll
	for(int k = 0; k < 4; ++k) {
		if(m) {
			v = v + H * (0.04 * v * v + 5.0 * v + 140.0 - u + I);
			u = u + H * A * (B * v - u);
			m = v < 30.0;
		}
	}
	const bool s = v >= 30.0;
	if(s) {
		v = double(C);
		u = u + double(D);
	}
	return s;
}

/* Spike test of synapse (source src, delay d) at step t: bit src of the
 * bitmap of step t - d, from the block's staged rows (row d-1 holds step
 * t-d) or from global memory. */
template<bool STAGED>
__device__ inline bool spiked(const nemo_float_step_args& a, const uint32_t* stage, unsigned t, unsigned d, uint32_t src)
{
	const uint32_t w = STAGED ? stage[(d - 1) * a.pitch + (src >> 5)] : a.bits[size_t(t - d) * a.pitch + (src >> 5)];
	return (w >> (src & 31)) & 1u;
}

/* One forward step for networks beyond the sliced form. */
template<bool STAGED>
__global__ void __launch_bounds__(FBLOCK)
forward_step_kernel(nemo_float_step_args a)
{
	constexpr unsigned UNROLL = unroll_for<FLANES>();
	extern __shared__ uint4 stage4[];
	__shared__ uint32_t fired;
	const unsigned t = a.t;
	const size_t n = a.n;
	const unsigned g = threadIdx.x / FLANES;
	const unsigned j = blockIdx.x * FGROUPS + g;
	const unsigned lane = threadIdx.x % FLANES;
	const bool live = j < n;
	uint32_t beg = 0, end = 0;
	float xj = 0.0f, C = 0.0f, Dd = 0.0f;
	double v0 = 0.0, u0 = 0.0, A = 0.0, B = 0.0;
	if(live) {
		/* the neuron's own operands, loaded before the staging and the
		 * synapses so that their latency overlaps */
		beg = a.rcm_ptr[j];
		end = a.rcm_ptr[j + 1];
		xj = a.x[size_t(t) * n + j];
		v0 = a.v[j];
		u0 = a.u[j];
		A = a.pa[j];
		B = a.pb[j];
		C = a.pc[j];
		Dd = a.pd[j];
	}
	/* UNROLL synapses per lane in flight; the sum runs in ascending synapse
	 * order per lane.  The first batch is issued before the staging so that
	 * both are in flight together. */
	uint32_t sd[UNROLL];
	float w[UNROLL];
	uint32_t k0 = beg + lane;
#pragma unroll
	for(unsigned q = 0; q < UNROLL; ++q) {
		const uint32_t k = k0 + FLANES * q;
		sd[q] = k < end ? a.rcm_sd[k] : 0u;
		w[q] = k < end ? a.wr[k] : 0.0f;
	}
	if(STAGED) {
		/* bitmaps of steps t-1 .. t-min(dmax, t), pitch a multiple of 4 words */
		const unsigned q4 = a.pitch / 4;
		const unsigned total = min(a.dmax, t) * q4;
		for(unsigned e = threadIdx.x; e < total; e += FBLOCK) {
			const unsigned r = e / q4;
			stage4[e] = reinterpret_cast<const uint4*>(a.bits + size_t(t - 1 - r) * a.pitch)[e - r * q4];
		}
	}
	if(threadIdx.x == 0) fired = 0;
	__syncthreads();
	const uint32_t* stage = reinterpret_cast<const uint32_t*>(stage4);

	bool s = false;
	if(live) {
		double acc = 0.0;
		while(k0 < end) {
#pragma unroll
			for(unsigned q = 0; q < UNROLL; ++q) {
				const unsigned d = (sd[q] >> 26) + 1;
				if(k0 + FLANES * q < end && t >= d && spiked<STAGED>(a, stage, t, d, sd[q] & IDX_MASK))
					acc += double(w[q]);
			}
			k0 += FLANES * UNROLL;
#pragma unroll
			for(unsigned q = 0; q < UNROLL; ++q) {
				const uint32_t k = k0 + FLANES * q;
				sd[q] = k < end ? a.rcm_sd[k] : 0u;
				w[q] = k < end ? a.wr[k] : 0.0f;
			}
		}
		acc = group_sum<FLANES>(acc);
		if(lane == 0) {
			const double I = acc + double(xj);
			if(a.ckpt && t % a.K == 0) {
				a.ckpt[size_t(t / a.K) * 2 * n + j] = v0;
				a.ckpt[size_t(t / a.K) * 2 * n + n + j] = u0;
			}
			double v = v0, u = u0;
			s = neuron_step(v, u, I, A, B, C, Dd);
			a.v[j] = v;
			a.u[j] = u;
			if(a.store) {
				a.S[size_t(t) * n + j] = s ? 1.0f : 0.0f;
				a.V[size_t(t) * n + j] = float(v);
			}
		}
	}
	if(a.store) {
		/* the block's 32 neurons are word blockIdx.x of step t's bitmap */
		if(s) atomicOr(&fired, 1u << g);
		__syncthreads();
		if(threadIdx.x == 0) a.bits[size_t(t) * a.pitch + blockIdx.x] = fired;
	}
}

/* Sixteen bytes per lane from src to the wave's place dst in LDS (lane l's at
 * dst + 16 l), without passing a register; staged() waits for the lanes' own. */
__device__ inline void stage16(void* dst, const void* src)
{
	__builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(src),
			(__attribute__((address_space(3))) void*)(dst), 16, 0, 0);
}

__device__ inline void staged()
{
	__builtin_amdgcn_s_waitcnt(0x0f70); /* vmcnt(0) */
}

/* The synapses of eight targets as a wave reads them (a slice): eight lanes per
 * target, four synapses per lane and line, of which lane l takes those at
 * 32 q + 4 l .. + 3 of its target's, a line per q up to the longest target's;
 * the places beyond a target's synapses have weight 0.  Lane l's j-th sum is
 * then that of lane 4 l + j of the 32 that forward_step_kernel gives a target,
 * and the sums over lanes pair the same values: a spike bit adds the weight or
 * +0, which leaves a sum as it is, so the input is forward_step_kernel's bit
 * for bit.
 *
 * The synapse's upper bits hold dmax - delay, its row in the staged bitmaps. */
constexpr unsigned SLICE = 8;
constexpr unsigned QUADS = 8; /* lines in flight: 256 synapses per target */

__device__ inline double slice_sum(const double (&acc)[4])
{
	return group_sum<8>((acc[0] + acc[1]) + (acc[2] + acc[3]));
}

/* w where bit (bit & 31) of word is set, +0 where not */
__device__ inline double masked(float w, uint32_t word, uint32_t bit)
{
	return double(__int_as_float(__float_as_int(w) & __builtin_amdgcn_sbfe(int(word), bit, 1)));
}

/* One forward step, a wave per slice and 32 neurons per block: the loads are
 * 16 bytes per lane from addresses that only the slice's number decides, a
 * synapse's spike test and sum are eight instructions without a branch, and a
 * wave's spikes are a byte of the bitmap that it writes by itself.
 *
 * 10 000 neurons x 200: forward_step_kernel takes 7.6 us a step, of which its
 * instructions are 3 us, this 5.7; 1000 x 100: 5.2 and 4.2, a chain of launch,
 * loads and the neuron's doubles. */
__global__ void __launch_bounds__(BLOCK)
forward_sliced_kernel(nemo_float_step_args a)
{
	extern __shared__ uint4 stage4[];
	const unsigned t = a.t;
	const size_t n = a.n;
	const unsigned lane = threadIdx.x % 64;
	const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
	const unsigned slice = blockIdx.x * (BLOCK / 64) + wave;
	const size_t j = size_t(slice) * SLICE + lane / SLICE;
	const bool neuron = lane % SLICE == 0 && j < n;
	/* bitmaps of steps t-dmax .. t-1, those before the first zero */
	const unsigned have = min(a.dmax, t);
	const unsigned none = (a.dmax - have) * (a.pitch / 4);
	const uint4* rows = reinterpret_cast<const uint4*>(a.bits + size_t(t - have) * a.pitch);
	for(unsigned e = threadIdx.x; e < have * (a.pitch / 4); e += BLOCK) stage16(stage4 + none + (e - lane), rows + e);
	for(unsigned e = threadIdx.x; e < none; e += BLOCK) stage4[e] = make_uint4(0, 0, 0, 0);

	uint32_t base = 0, end = 0;
	if(size_t(slice) * SLICE < n) {
		base = a.slice_ptr[slice];
		end = a.slice_ptr[slice + 1];
	}
	const uint4* sds = reinterpret_cast<const uint4*>(a.slice_sd) + lane;
	const float4* ws = reinterpret_cast<const float4*>(a.wr) + lane;
	uint4 sd[QUADS];
	float4 w[QUADS];
	auto load = [&](uint32_t line) {
#pragma unroll
		for(unsigned q = 0; q < QUADS; ++q) {
			if(line + q >= end) break;
			sd[q] = sds[size_t(line + q) * 64];
			w[q] = ws[size_t(line + q) * 64];
		}
	};
	float xj = 0.0f, C = 0.0f, Dd = 0.0f, A = 0.0f, B = 0.0f;
	double v = 0.0, u = 0.0;
	if(neuron) {
		xj = a.x[size_t(t) * n + j];
		v = a.v[j];
		u = a.u[j];
		A = a.pa[j];
		B = a.pb[j];
		C = a.pc[j];
		Dd = a.pd[j];
	}
	load(base);
	staged();
	__syncthreads();

	const uint32_t* stage = reinterpret_cast<const uint32_t*>(stage4);
	auto word = [&](uint32_t sd) { return stage[__umul24(sd >> 26, a.pitch) + ((sd & IDX_MASK) >> 5)]; };
	double acc[4] = {};
	for(uint32_t line = base; line < end; line += QUADS) {
		if(line != base) load(line);
#pragma unroll
		for(unsigned q = 0; q < QUADS; ++q) {
			if(line + q >= end) break;
			acc[0] += masked(w[q].x, word(sd[q].x), sd[q].x);
			acc[1] += masked(w[q].y, word(sd[q].y), sd[q].y);
			acc[2] += masked(w[q].z, word(sd[q].z), sd[q].z);
			acc[3] += masked(w[q].w, word(sd[q].w), sd[q].w);
		}
	}
	const double sum = slice_sum(acc);
	bool s = false;
	if(neuron) {
		if(a.ckpt && t % a.K == 0) {
			a.ckpt[size_t(t / a.K) * 2 * n + j] = v;
			a.ckpt[size_t(t / a.K) * 2 * n + n + j] = u;
		}
		s = neuron_step(v, u, sum + double(xj), A, B, C, Dd);
		a.v[j] = v;
		a.u[j] = u;
		if(a.store) {
			a.S[size_t(t) * n + j] = s ? 1.0f : 0.0f;
			a.V[size_t(t) * n + j] = float(v);
		}
	}
	if(a.store) {
		/* bits 0, 8, .. 56 to the bits of a byte */
		const uint64_t fired = __ballot(s);
		const unsigned byte = unsigned((fired * 0x0102040810204080ULL) >> 56);
		if(lane == 0) reinterpret_cast<uint8_t*>(a.bits + size_t(t) * a.pitch)[slice] = uint8_t(byte);
	}
}

/* A neuron's step recomputed from its entry state and input, for its adjoint. */
struct StepTrace {
	double v[5], u[5]; /* before and after each substep */
	bool active[4];
	double A, B;
};

__device__ inline StepTrace trace_step(double v, double u, double I, double A, double B)
{
	StepTrace s;
	s.A = A;
	s.B = B;
	s.v[0] = v;
	s.u[0] = u;
	bool m = true;
#pragma unroll
	for(int k = 0; k < 4; ++k) {
		s.active[k] = m;
		if(m) {
			s.v[k + 1] = s.v[k] + H * (0.04 * s.v[k] * s.v[k] + 5.0 * s.v[k] + 140.0 - s.u[k] + I);
			s.u[k + 1] = s.u[k] + H * A * (B * s.v[k + 1] - s.u[k]);
			m = s.v[k + 1] < 30.0;
		} else {
			s.v[k + 1] = s.v[k];
			s.u[k + 1] = s.u[k];
		}
	}
	return s;
}

/* Adjoints of a step: of the state before it, of its input, and its terms of
 * the parameters' gradients. */
struct StepAdjoint {
	double Lv, Lu, lI, ga, gb, gd;
};

/* From those of the state after the step (lv, lu) and of its spike (lS). */
__device__ inline StepAdjoint adjoint_step(const StepTrace& f, double lv, double lu, double lS, double slope)
{
	const double s = f.v[4] >= 30.0 ? 1.0 : 0.0;
	StepAdjoint g;
	/* reset v' = v4 + s (c - v4), u' = u4 + s d with s constant; the spike
	 * s = H(v4 - 30) reaches v4 through the surrogate */
	g.gd = lu * s;
	g.Lv = lv * (1.0 - s) + lS * slope;
	g.Lu = lu;
	/* substeps in reverse; a masked substep is the identity */
	g.lI = 0.0;
	g.ga = 0.0;
	g.gb = 0.0;
#pragma unroll
	for(int k = 3; k >= 0; --k) {
		if(!f.active[k]) continue;
		const double total = g.Lv + g.Lu * H * f.A * f.B;
		g.ga += g.Lu * H * (f.B * f.v[k + 1] - f.u[k]);
		g.gb += g.Lu * H * f.A * f.v[k + 1];
		const double nLu = g.Lu * (1.0 - H * f.A) - total * H;
		g.Lv = total * (1.0 + H * (0.08 * f.v[k] + 5.0));
		g.Lu = nLu;
		g.lI += total * H;
	}
	return g;
}

/* One backward step for networks beyond the staged form: the spike adjoint
 * of a neuron is gathered over its synapses from the ring of recent input
 * adjoints in memory. */
__global__ void __launch_bounds__(BLOCK)
backward_step_kernel(nemo_float_back_args a)
{
	const unsigned i = blockIdx.x * GROUPS + threadIdx.x / LANES;
	const unsigned lane = threadIdx.x % LANES;
	if(i >= a.n) return;
	const unsigned tau = a.t;
	const size_t n = a.n;
	const unsigned R = a.ring;
	const uint32_t beg = a.fcm_ptr[i], end = a.fcm_ptr[i + 1];
	const size_t r = size_t(tau) * n + i;
	const bool fired = a.S[r] != 0.0f;
	/* the neuron's own operands, loaded before the synapses so that their
	 * latency overlaps the gathers' */
	const size_t sq = size_t(tau - a.t0) * n + i;
	const float gSr = a.gS ? a.gS[r] : 0.0f;
	const float gVr = a.gV ? a.gV[r] : 0.0f;
	const double LVi = a.LV[i], LUi = a.LU[i];
	const double I = a.seg_I[sq];
	const double sv = a.seg_v[sq], su = a.seg_u[sq];
	const double A = a.pa[i], B = a.pb[i];
	const float ga0 = a.ga[i], gb0 = a.gb[i], gd0 = a.gd[i];

	/* adjoint of this step's spike from the steps it reaches (transposed
	 * delivery), and the weight gradient of the synapses it drove; UNROLL
	 * synapses per lane in flight, summed in ascending synapse order */
	/* 4 in flight per lane keeps the kernel at 7 waves per SIMD; 8 would
	 * need more registers than 5 waves allow */
	constexpr unsigned UNROLL = 4;
	const unsigned tm = tau % R; /* slot of step tau + d: tm + d, less R once past it (d < R) */
	double acc = 0.0;
	for(uint32_t k0 = beg + lane; k0 < end; k0 += LANES * UNROLL) {
		uint32_t td[UNROLL];
		float w[UNROLL], g[UNROLL];
#pragma unroll
		for(unsigned q = 0; q < UNROLL; ++q) {
			const uint32_t k = k0 + LANES * q;
			td[q] = k < end ? a.fcm_td[k] : 0u;
			w[q] = k < end ? a.wf[k] : 0.0f;
			g[q] = k < end && fired ? a.gw[k] : 0.0f;
		}
		bool live[UNROLL];
		double l[UNROLL];
#pragma unroll
		for(unsigned q = 0; q < UNROLL; ++q) {
			const unsigned d = (td[q] >> 26) + 1;
			live[q] = k0 + LANES * q < end && tau + d < a.T;
			const unsigned slot = tm + d >= R ? tm + d - R : tm + d;
			l[q] = live[q] ? a.LI[size_t(slot) * n + (td[q] & IDX_MASK)] : 0.0;
		}
#pragma unroll
		for(unsigned q = 0; q < UNROLL; ++q) {
			if(!live[q]) continue;
			acc += double(w[q]) * l[q];
			if(fired) a.gw[k0 + LANES * q] = float(double(g[q]) + l[q]);
		}
	}
	acc = group_sum<LANES>(acc);
	if(lane != 0) return;

	const StepTrace f = trace_step(sv, su, I, A, B);
	const StepAdjoint g = adjoint_step(f, LVi + double(gVr), LUi, double(gSr) + acc, surrogate(f.v[4]));
	a.LV[i] = g.Lv;
	a.LU[i] = g.Lu;
	a.LI[size_t(tau % R) * n + i] = g.lI;
	if(a.gx) a.gx[r] = float(g.lI);
	a.ga[i] = ga0 + float(g.ga);
	a.gb[i] = gb0 + float(g.gb);
	a.gd[i] = gd0 + float(g.gd);
}

/* One backward step with the input adjoints of one step in LDS.  A block owns
 * tile neurons and their synapses, sorted by delay: rows of (neuron, delay).
 * The adjoints of step t + 1, complete since the last launch, are staged whole
 * (8 bytes per neuron), and each row adds its weighted sum of them to the
 * spike adjoint of its neuron at step t + 1 - delay, which a ring of dmax
 * steps collects; delay 1 completes step t, whose adjoint the block's last
 * threads then form.  L lanes per row sum in a fixed order, and a spike
 * adjoint receives its delays in descending order: the sums are reproducible
 * bit for bit.
 *
 * A wave passes a slice of 64 / L rows: the block's rows are sorted by length
 * and a slice's synapses stored as its lanes read them, four per lane and
 * line, up to the longest row; the places left have weight 0 and the adjoint
 * of a neuron that does not exist, 0.  (With each row stored by itself a load
 * touched as many cache lines as rows, and the steps took no less than the
 * general form's.)  The gradients of the weights of fired neurons are in that order
 * too, and wait for a load of their own: they come last, beside the neurons.
 *
 * The general form above gathers every synapse's adjoint from memory, 2e6
 * cache lines a step at 10 000 neurons x 200, which bounds it (14.2 us a
 * step); here a synapse costs the 6 bytes of its weight and target, in order,
 * and an LDS read: 6.7 us there (1000 x 100: 5.4 against 4.4, where the chain
 * of launch, loads, two barriers and the neuron's doubles is the whole step). */
template<unsigned L>
__global__ void __launch_bounds__(PUSH_BLOCK)
backward_push_kernel(nemo_float_push_args a)
{
	constexpr unsigned LINES = 4; /* in flight, four synapses per lane each */
	extern __shared__ double2 push_lds[];
	double* li = reinterpret_cast<double*>(push_lds); /* [pitch] of step t + 1, and a zero */
	double* spike = li + a.pitch + 2;                 /* [tile] of step t */
	const unsigned threads = blockDim.x;
	const unsigned tau = a.t;
	const size_t n = a.n;
	const unsigned D = a.dmax;
	const unsigned first = blockIdx.x * a.tile;
	const unsigned count = min(a.tile, unsigned(n) - first);
	const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
	const unsigned lane = threadIdx.x % 64;
	/* the last step has no adjoints after it */
	const unsigned slices = tau + 1 < a.T ? a.slices : 0;

	const ushort4* targets = reinterpret_cast<const ushort4*>(a.row_target) + lane;
	const float4* weights = reinterpret_cast<const float4*>(a.row_w) + lane;
	float4* grads = reinterpret_cast<float4*>(a.row_gw) + lane;
	ushort4 target[LINES];
	float4 w[LINES];
	uint32_t base = 0, end = 0; /* lines of the slice */
	nemo_float_row row = {};
	double* slot = nullptr;
	double before = 0.0;
	bool fired = false;
	auto load = [&](uint32_t line) {
#pragma unroll
		for(unsigned q = 0; q < LINES; ++q) {
			if(line + q >= end) break;
			target[q] = targets[size_t(line + q) * 64];
			w[q] = weights[size_t(line + q) * 64];
		}
	};
	auto begin_slice = [&](unsigned s) {
		const size_t at = size_t(blockIdx.x) * a.slices + s;
		base = a.slice_ptr[at];
		end = a.slice_ptr[at + 1];
		row = a.rows[at * 64 + lane];
		load(base);
		const unsigned d = row.delay;
		slot = nullptr;
		fired = false;
		/* delay 0: no row; a step before the first receives nothing */
		if(d == 0 || d > tau + 1) return;
		const unsigned step = tau + 1 - d;
		const size_t source = first + row.neuron;
		slot = a.ring + size_t(step % D) * n + source;
		before = d == D ? 0.0 : *slot;
		fired = a.S[size_t(step) * n + source] != 0.0f;
	};
	/* the gradients of the weights of fired neurons; the places without a
	 * synapse collect zeros */
	auto drove = [&]() {
		if(!fired) return;
		for(uint32_t line = base; line < end; line += LINES) {
			if(line != base || end - base > LINES) load(line);
			float4 g[LINES];
#pragma unroll
			for(unsigned q = 0; q < LINES; ++q)
				if(line + q < end) g[q] = grads[size_t(line + q) * 64];
#pragma unroll
			for(unsigned q = 0; q < LINES; ++q) {
				if(line + q >= end) break;
				g[q].x = float(double(g[q].x) + li[target[q].x]);
				g[q].y = float(double(g[q].y) + li[target[q].y]);
				g[q].z = float(double(g[q].z) + li[target[q].z]);
				g[q].w = float(double(g[q].w) + li[target[q].w]);
				grads[size_t(line + q) * 64] = g[q];
			}
		}
	};

	/* the block's last threads take its neurons: their waves have the fewest slices */
	const unsigned nl = threads - 1 - threadIdx.x;
	const bool neuron = nl < count;
	const size_t i = first + nl;
	const size_t at = size_t(tau) * n + i;
	double LVi = 0.0, LUi = 0.0, I = 0.0, sv = 0.0, su = 0.0;
	float gSr = 0.0f, gVr = 0.0f, A = 0.0f, B = 0.0f, ga0 = 0.0f, gb0 = 0.0f, gd0 = 0.0f;
	if(slices) {
		const double2* next = reinterpret_cast<const double2*>(a.LI + size_t((tau + 1) & 1) * a.pitch);
		for(unsigned e = threadIdx.x; e < a.pitch / 2; e += threads) stage16(push_lds + (e - lane), next + e);
		if(threadIdx.x == 0) li[a.pitch] = 0.0;
	}
	if(neuron) {
		const size_t sq = size_t(tau - a.t0) * n + i;
		sv = a.seg_v[sq];
		su = a.seg_u[sq];
		I = a.seg_I[sq];
		A = a.pa[i];
		B = a.pb[i];
		LVi = a.LV[i];
		LUi = a.LU[i];
		if(a.gS) gSr = a.gS[at];
		if(a.gV) gVr = a.gV[at];
		ga0 = a.ga[i];
		gb0 = a.gb[i];
		gd0 = a.gd[i];
	}
	if(wave < slices) begin_slice(wave);
	staged();
	__syncthreads();
	for(unsigned s = wave; s < slices; s += threads / 64) {
		double acc[4] = {};
		for(uint32_t line = base; line < end; line += LINES) {
			if(line != base) load(line);
#pragma unroll
			for(unsigned q = 0; q < LINES; ++q) {
				if(line + q >= end) break;
				acc[0] = __builtin_fma(double(w[q].x), li[target[q].x], acc[0]);
				acc[1] = __builtin_fma(double(w[q].y), li[target[q].y], acc[1]);
				acc[2] = __builtin_fma(double(w[q].z), li[target[q].z], acc[2]);
				acc[3] = __builtin_fma(double(w[q].w), li[target[q].w], acc[3]);
			}
		}
		const double sum = before + group_sum<L>((acc[0] + acc[1]) + (acc[2] + acc[3]));
		if(lane % L == 0 && slot) {
			if(row.delay == 1) spike[row.neuron] = sum;
			else *slot = sum;
		}
		if(s + threads / 64 < slices) {
			drove();
			begin_slice(s + threads / 64);
		}
	}
	__syncthreads();
	if(neuron) {
		const StepTrace f = trace_step(sv, su, I, A, B);
		const StepAdjoint g = adjoint_step(f, LVi + double(gVr), LUi, double(gSr) + (slices ? spike[nl] : 0.0),
				surrogate(f.v[4]));
		a.LV[i] = g.Lv;
		a.LU[i] = g.Lu;
		a.LI[size_t(tau & 1) * a.pitch + i] = g.lI;
		if(a.gx) a.gx[at] = float(g.lI);
		a.ga[i] = ga0 + float(g.ga);
		a.gb[i] = gb0 + float(g.gb);
		a.gd[i] = gd0 + float(g.gd);
	}
	if(wave < slices) drove();
}

/* Firing histories for the replay: hist[r][j] bit k set when neuron j
 * fired at step 64 (r - 1) + k; row 0 (steps -64..-1) and steps from T on
 * are zero. */
__global__ void __launch_bounds__(BLOCK)
pack_history_kernel(uint64_t* hist, unsigned rows, const float* S, unsigned n, unsigned T)
{
	const unsigned j = blockIdx.x * BLOCK + threadIdx.x;
	const unsigned r = blockIdx.y;
	if(j >= n || r >= rows) return;
	uint64_t word = 0;
	if(r > 0) {
		const unsigned t0 = 64 * (r - 1);
		/* 16 loads in flight */
#pragma unroll
		for(unsigned k0 = 0; k0 < 64; k0 += 16) {
			float s[16];
#pragma unroll
			for(unsigned k = 0; k < 16; ++k) s[k] = S[size_t(min(t0 + k0 + k, T - 1)) * n + j];
#pragma unroll
			for(unsigned k = 0; k < 16; ++k)
				if(t0 + k0 + k < T && s[k] != 0.0f) word |= uint64_t(1) << (k0 + k);
		}
	}
	hist[size_t(r) * n + j] = word;
}

/* Steps t0..t1-1 of the forward in one launch, from the state before t0 and
 * the recorded spikes: each step's entry state and input are recorded.  The
 * synaptic sums are those of forward_step_kernel, operation for operation
 * (same lanes per neuron, same synapse-to-lane assignment and order, same
 * butterfly), so the replayed state equals the forward's.  CH steps at a
 * time: each synapse's spikes over the CH steps come from at most two
 * history words. */
constexpr unsigned CH = 16;

__global__ void __launch_bounds__(BLOCK)
replay_kernel(nemo_float_replay_args a)
{
	constexpr unsigned UNROLL = 4;
	constexpr unsigned RGROUPS = BLOCK / FLANES;
	static_assert(CH <= FLANES, "lane c holds the input of step c of a chunk");
	const unsigned j = blockIdx.x * RGROUPS + threadIdx.x / FLANES;
	const unsigned lane = threadIdx.x % FLANES;
	if(j >= a.n) return;
	const size_t n = a.n;
	const uint32_t beg = a.rcm_ptr[j], end = a.rcm_ptr[j + 1];
	const double A = a.pa[j], B = a.pb[j];
	const float C = a.pc[j], Dd = a.pd[j];
	double v = a.v0[j], u = a.u0[j];
	for(unsigned c0 = a.t0; c0 < a.t1; c0 += CH) {
		const unsigned steps = min(CH, a.t1 - c0);
		const float xl = lane < steps ? a.x[size_t(c0 + lane) * n + j] : 0.0f;
		double acc[CH];
#pragma unroll
		for(unsigned q = 0; q < CH; ++q) acc[q] = 0.0;
		for(uint32_t k0 = beg + lane; k0 < end; k0 += FLANES * UNROLL) {
			uint32_t sd[UNROLL];
			float w[UNROLL];
#pragma unroll
			for(unsigned q = 0; q < UNROLL; ++q) {
				const uint32_t k = k0 + FLANES * q;
				sd[q] = k < end ? a.rcm_sd[k] : 0u;
				w[q] = k < end ? a.wr[k] : 0.0f;
			}
			/* the source's spikes at steps c0-d .. c0-d+CH-1: history bits
			 * from p = c0 - d + 64 (d <= 64, so p >= 0) */
			uint64_t lo[UNROLL], hi[UNROLL];
#pragma unroll
			for(unsigned q = 0; q < UNROLL; ++q) {
				const bool valid = k0 + FLANES * q < end;
				const unsigned p = c0 + 64 - ((sd[q] >> 26) + 1);
				const size_t row = size_t(p >> 6) * n + (sd[q] & IDX_MASK);
				lo[q] = valid ? a.hist[row] : 0;
				hi[q] = valid && (p & 63) + CH > 64 ? a.hist[row + n] : 0;
			}
#pragma unroll
			for(unsigned q = 0; q < UNROLL; ++q) {
				const unsigned o = (c0 + 64 - ((sd[q] >> 26) + 1)) & 63;
				const uint64_t win = o ? (lo[q] >> o) | (hi[q] << (64 - o)) : lo[q];
#pragma unroll
				for(unsigned c = 0; c < CH; ++c)
					if((win >> c) & 1) acc[c] += double(w[q]);
			}
		}
#pragma unroll
		for(unsigned c = 0; c < CH; ++c) {
			const double tot = group_sum<FLANES>(acc[c]);
			const float xc = __shfl(xl, c, FLANES);
			if(lane == 0 && c < steps) {
				const double I = tot + double(xc);
				const size_t rec = size_t(c0 + c - a.t0) * n + j;
				a.seg_v[rec] = v;
				a.seg_u[rec] = u;
				a.seg_I[rec] = I;
				neuron_step(v, u, I, A, B, C, Dd);
			}
		}
	}
}

/* The same for sliced networks of up to NEMO_FLOAT_REPLAY_MAX neurons and
 * delays below 58: the sources' spikes over 65 - dmax steps and the dmax
 * before them are staged as 64-bit windows.  The inputs do not depend on the
 * state, so the block's waves share its slices' steps, REPLAY_CH at a time and
 * summed in the order of forward_step_kernel; then a thread per neuron passes
 * the steps.
 *
 * The general form reads a window per synapse and 16 steps from memory, 8e6
 * gathers per 50 steps at 10 000 neurons x 200 (82 us).  With a wave per
 * slice that passes sums and state in turn this form took 71 us: 313 blocks
 * of four waves leave some compute units two, and the state's chain waits
 * alone.  Now 44 us, and 14 instead of 16 for 25 steps of 1000 x 100. */
constexpr unsigned REPLAY_CH = 8;
constexpr unsigned REPLAY_BLOCK = 1024;

__global__ void __launch_bounds__(REPLAY_BLOCK)
replay_sliced_kernel(nemo_float_replay_args a, unsigned slices)
{
	constexpr unsigned LINES = 4;
	extern __shared__ uint64_t window[]; /* [n] bit b: fired at step c0 - dmax + b */
	const size_t n = a.n;
	const unsigned threads = blockDim.x;
	const unsigned lane = threadIdx.x % 64;
	const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
	const unsigned shares = threads / 64 / slices; /* of a slice's steps */
	const unsigned share = wave / slices;
	const unsigned slice = blockIdx.x * slices + wave % slices;
	const size_t j = size_t(slice) * SLICE + lane / SLICE;
	const unsigned l = lane % SLICE;
	uint32_t base = 0, end = 0;
	if(size_t(slice) * SLICE < n) {
		base = a.slice_ptr[slice];
		end = a.slice_ptr[slice + 1];
	}
	const uint4* sds = reinterpret_cast<const uint4*>(a.slice_sd) + lane;
	const float4* ws = reinterpret_cast<const float4*>(a.wr) + lane;
	const unsigned span = 65 - a.dmax;
	for(unsigned c0 = a.t0; c0 < a.t1; c0 += span) {
		/* history bits from p = c0 - dmax + 64 */
		const unsigned p = c0 + 64 - a.dmax;
		const uint64_t* lo = a.hist + size_t(p >> 6) * n;
		const unsigned o = p & 63;
		if(c0 != a.t0) __syncthreads();
#pragma unroll 4
		for(unsigned e = threadIdx.x; e < n; e += threads)
			window[e] = o ? (lo[e] >> o) | (lo[n + e] << (64 - o)) : lo[e];
		__syncthreads();
		const unsigned c1 = min(a.t1, c0 + span);
		for(unsigned c = c0 + share * REPLAY_CH; c < c1; c += shares * REPLAY_CH) {
			const bool mine = j < n && c + l < c1;
			const float xl = mine ? a.x[size_t(c + l) * n + j] : 0.0f;
			double acc[REPLAY_CH][4] = {};
			for(uint32_t line = base; line < end; line += LINES) {
				uint4 sd[LINES];
				float4 w[LINES];
#pragma unroll
				for(unsigned q = 0; q < LINES; ++q) {
					if(line + q >= end) break;
					sd[q] = sds[size_t(line + q) * 64];
					w[q] = ws[size_t(line + q) * 64];
				}
#pragma unroll
				for(unsigned q = 0; q < LINES; ++q) {
					if(line + q >= end) break;
					const uint32_t src[4] = {sd[q].x, sd[q].y, sd[q].z, sd[q].w};
					const float wq[4] = {w[q].x, w[q].y, w[q].z, w[q].w};
#pragma unroll
					for(unsigned i = 0; i < 4; ++i) {
						/* bit k: fired at step c + k - delay */
						const uint32_t bits = uint32_t(window[src[i] & IDX_MASK] >> ((src[i] >> 26) + (c - c0)));
#pragma unroll
						for(unsigned k = 0; k < REPLAY_CH; ++k) acc[k][i] += masked(wq[i], bits, k);
					}
				}
			}
			/* lane l of the target has the input of step c + l */
			double I = 0.0;
#pragma unroll
			for(unsigned k = 0; k < REPLAY_CH; ++k) {
				const double sum = slice_sum(acc[k]);
				if(l == k) I = sum;
			}
			if(mine) a.seg_I[size_t(c + l - a.t0) * n + j] = I + double(xl);
		}
	}
	__syncthreads();
	/* the block's inputs are in memory, visible to it */
	const size_t i = size_t(blockIdx.x) * slices * SLICE + threadIdx.x;
	if(threadIdx.x >= slices * SLICE || i >= n) return;
	const float C = a.pc[i], Dd = a.pd[i];
	const double A = a.pa[i], B = a.pb[i];
	double v = a.v0[i], u = a.u0[i];
	const unsigned steps = a.t1 - a.t0;
	double next[REPLAY_CH];
#pragma unroll
	for(unsigned k = 0; k < REPLAY_CH; ++k) next[k] = k < steps ? a.seg_I[size_t(k) * n + i] : 0.0;
	for(unsigned c = 0; c < steps; c += REPLAY_CH) {
		double I[REPLAY_CH];
#pragma unroll
		for(unsigned k = 0; k < REPLAY_CH; ++k) {
			I[k] = next[k];
			const unsigned s = min(c + REPLAY_CH + k, steps - 1);
			next[k] = a.seg_I[size_t(s) * n + i];
		}
#pragma unroll
		for(unsigned k = 0; k < REPLAY_CH; ++k) {
			if(c + k >= steps) break;
			const size_t rec = size_t(c + k) * n + i;
			a.seg_v[rec] = v;
			a.seg_u[rec] = u;
			neuron_step(v, u, I[k], A, B, C, Dd);
		}
	}
}

/* 0 for a place without a synapse */
__device__ inline float weight_of(const float* w, uint32_t user, size_t synapses)
{
	return user < synapses ? w[user] : 0.0f;
}

/* The weights in the slices' order, a line of a slice per 64 lanes.  The grid
 * passes the first lines of all slices, then the second ones, and so on: a
 * target's synapses are in source order, so what is read at one time are the
 * weights of some neighbouring sources, which the L2 caches hold (1.1 of 8 MB
 * at 10 000 neurons x 200).  Read target by target, every weight is a cache
 * line from memory: 23.5 us there, 15.8 so. */
__global__ void __launch_bounds__(BLOCK)
slice_weights_kernel(float4* wr, const float* w, const uint4* user, const uint32_t* slice_ptr, unsigned slices,
		size_t synapses)
{
	const unsigned slice = blockIdx.x * (BLOCK / 64) + threadIdx.x / 64;
	if(slice >= slices) return;
	const uint32_t line = slice_ptr[slice] + blockIdx.y;
	if(line >= slice_ptr[slice + 1]) return;
	const size_t at = size_t(line) * 64 + threadIdx.x % 64;
	const uint4 u = user[at];
	wr[at] = make_float4(weight_of(w, u.x, synapses), weight_of(w, u.y, synapses), weight_of(w, u.z, synapses),
			weight_of(w, u.w, synapses));
}

/* A synapse's place in the slices of forward_sliced_kernel, one thread per
 * synapse of the reverse matrix. */
__global__ void __launch_bounds__(BLOCK)
fill_slices_kernel(nemo_float_slice_args a)
{
	const size_t k = size_t(blockIdx.x) * BLOCK + threadIdx.x;
	if(k >= a.synapses) return;
	/* the target: the last one whose synapses do not begin after k */
	unsigned lo = 0, hi = a.n;
	while(hi - lo > 1) {
		const unsigned mid = lo + (hi - lo) / 2;
		if(a.rcm_ptr[mid] <= k) lo = mid;
		else hi = mid;
	}
	const uint32_t e = uint32_t(k - a.rcm_ptr[lo]);
	const size_t at = (size_t(a.slice_ptr[lo / SLICE]) + e / 32) * 256 + lo % SLICE * 32 + e % 32;
	const uint32_t packed = a.rcm_sd[k];
	a.slice_sd[at] = (packed & IDX_MASK) | (a.dmax - 1 - (packed >> 26)) << 26;
	a.slice_user[at] = a.rcm_user[k];
}

/* A neuron's synapses to their places in the rows of backward_push_kernel, a
 * thread per neuron in network order; row_at is the first place of each row. */
constexpr unsigned FILL_BLOCK = 64;

__global__ void __launch_bounds__(FILL_BLOCK)
fill_rows_kernel(nemo_float_rows_args a)
{
	__shared__ uint32_t used[64][FILL_BLOCK]; /* of the row of each delay */
	const size_t i = size_t(blockIdx.x) * FILL_BLOCK + threadIdx.x;
	if(i >= a.n) return;
	for(unsigned d = 0; d < a.dmax; ++d) used[d][threadIdx.x] = 0;
	for(uint32_t p = a.fcm_ptr[i]; p < a.fcm_ptr[i + 1]; ++p) {
		const uint32_t td = a.fcm_td[p];
		const unsigned d = td >> 26;
		const uint32_t e = used[d][threadIdx.x]++;
		const size_t at = a.row_at[i * a.dmax + d] + size_t(e / (4 * a.lanes)) * 256 + e % (4 * a.lanes);
		a.row_user[at] = p;
		a.row_target[at] = uint16_t(td & IDX_MASK);
	}
}

/* What a forward begins with: the weights in reverse order (unless they are
 * in slices), and the state in double. */
__global__ void __launch_bounds__(BLOCK)
begin_forward_kernel(nemo_float_begin_forward_args a)
{
	const size_t k = size_t(blockIdx.x) * BLOCK + threadIdx.x;
	if(k < a.wr_entries) a.wr[k] = weight_of(a.w, a.wr_user[k], a.synapses);
	if(k < a.n) {
		a.v[k] = double(a.v0[k]);
		a.u[k] = double(a.u0[k]);
	}
}

/* What a backward begins with: the weights in its orders, and its sums at
 * zero. */
__global__ void __launch_bounds__(BLOCK)
begin_backward_kernel(nemo_float_begin_backward_args a)
{
	const size_t k = size_t(blockIdx.x) * BLOCK + threadIdx.x;
	if(k < a.wr_entries) a.wr[k] = weight_of(a.w, a.wr_user[k], a.synapses);
	if(k < a.synapses && !a.entries) a.gw[k] = 0.0f;
	if(k < a.entries) {
		a.row_w[k] = weight_of(a.w, a.row_user[k], a.synapses);
		a.row_gw[k] = 0.0f;
	}
	if(k < a.li) a.LI[k] = 0.0;
	if(k < a.n) {
		a.LV[k] = 0.0;
		a.LU[k] = 0.0;
		a.ga[k] = 0.0f;
		a.gb[k] = 0.0f;
		a.gd[k] = 0.0f;
	}
}

/* What a backward ends with: the weights' gradients back in network order,
 * and the state's adjoints before the first step as floats. */
__global__ void __launch_bounds__(BLOCK)
end_backward_kernel(nemo_float_end_backward_args a)
{
	const size_t k = size_t(blockIdx.x) * BLOCK + threadIdx.x;
	if(k < a.entries) {
		const uint32_t u = a.row_user[k];
		if(u < a.synapses) a.gw[u] = a.row_gw[k];
	}
	if(k < a.n) {
		if(a.gv0) a.gv0[k] = float(a.LV[k]);
		if(a.gu0) a.gu0[k] = float(a.LU[k]);
	}
}

inline unsigned blocks_for(size_t n)
{
	return unsigned((n + BLOCK - 1) / BLOCK);
}

} // namespace

/* The workspace of the allocation-free forward (see nemo_float_scratch).
 * Host code never passes its name to a kernel: the name is a host-side
 * stand-in, and the device address comes from hipGetSymbolAddress. */
static __device__ __align__(256) unsigned char scratch[NEMO_FLOAT_SCRATCH_BYTES];

extern "C" {

hipError_t nemo_float_scratch(void** ptr, size_t* bytes)
{
	static std::mutex lock;
	static void* addr[NEMO_FLOAT_SCRATCH_DEVICES] = {};
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if(e != hipSuccess) return e;
	if(dev < 0 || dev >= NEMO_FLOAT_SCRATCH_DEVICES) return hipErrorInvalidDevice;
	std::lock_guard<std::mutex> held(lock);
	if(!addr[dev]) {
		void* p = nullptr;
		e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
		if(e != hipSuccess) return e;
		if(!p) return hipErrorInvalidSymbol;
		addr[dev] = p;
	}
	*ptr = addr[dev];
	*bytes = sizeof(scratch);
	return hipSuccess;
}

hipError_t nemo_launch_float_forward_step(hipStream_t st, const nemo_float_step_args* a)
{
	if(a->n == 0) return hipSuccess;
	if(a->ckpt && a->K == 0) return hipErrorInvalidValue;
	if(!a->bits || a->pitch % 4 || a->pitch < nemo_float_bitmap_pitch(a->n) || a->dmax == 0)
		return hipErrorInvalidValue;
	const dim3 grid(unsigned((a->n + FGROUPS - 1) / FGROUPS));
	if(a->slice_ptr) {
		const size_t lds = nemo_float_stage_bytes(a->n, a->dmax);
		if(!a->stage || lds > NEMO_FLOAT_STAGE_MAX) return hipErrorInvalidValue;
		static_assert(FGROUPS == BLOCK / 64 * SLICE, "a word of the bitmap per block");
		hipLaunchKernelGGL(forward_sliced_kernel, grid, dim3(BLOCK), lds, st, *a);
	} else if(a->stage) {
		const size_t lds = nemo_float_stage_bytes(a->n, a->dmax);
		if(lds > NEMO_FLOAT_STAGE_MAX) return hipErrorInvalidValue;
		hipLaunchKernelGGL(forward_step_kernel<true>, grid, dim3(FBLOCK), lds, st, *a);
	} else {
		hipLaunchKernelGGL(forward_step_kernel<false>, grid, dim3(FBLOCK), 0, st, *a);
	}
	return hipGetLastError();
}

unsigned nemo_float_bitmap_pitch(unsigned n)
{
	return ((n + 31) / 32 + 3) / 4 * 4;
}

size_t nemo_float_stage_bytes(unsigned n, unsigned dmax)
{
	return size_t(dmax) * nemo_float_bitmap_pitch(n) * sizeof(uint32_t);
}

hipError_t nemo_launch_pack_history(hipStream_t st, uint64_t* hist, unsigned rows, const float* S, unsigned n,
		unsigned T)
{
	if(n == 0 || rows == 0) return hipSuccess;
	if(rows < nemo_float_history_rows(T)) return hipErrorInvalidValue;
	hipLaunchKernelGGL(pack_history_kernel, dim3(blocks_for(n), rows), dim3(BLOCK), 0, st, hist, rows, S, n, T);
	return hipGetLastError();
}

unsigned nemo_float_history_rows(unsigned T)
{
	return (T + 63) / 64 + 2;
}

hipError_t nemo_launch_float_replay(hipStream_t st, const nemo_float_replay_args* a)
{
	if(a->n == 0 || a->t1 <= a->t0) return hipSuccess;
	if(!a->hist || a->hist_rows < nemo_float_history_rows(a->t1) || a->dmax == 0 || a->dmax > 64)
		return hipErrorInvalidValue;
	if(a->slice_ptr) {
		if(a->n > NEMO_FLOAT_REPLAY_MAX || a->dmax + REPLAY_CH > 65) return hipErrorInvalidValue;
		/* a block per compute unit, as each stages all the windows, and up to
		 * 16 waves in it */
		const unsigned all = (a->n + SLICE - 1) / SLICE;
		const unsigned slices = (all + 255) / 256;
		const unsigned most = REPLAY_BLOCK / 64 / slices;
		const unsigned parts = (a->t1 - a->t0 + REPLAY_CH - 1) / REPLAY_CH;
		const unsigned threads = slices * (parts < most ? parts : most) * 64;
		hipLaunchKernelGGL(replay_sliced_kernel, dim3((all + slices - 1) / slices), dim3(threads),
				size_t(a->n) * sizeof(uint64_t), st, *a, slices);
		return hipGetLastError();
	}
	constexpr unsigned RGROUPS = BLOCK / FLANES;
	hipLaunchKernelGGL(replay_kernel, dim3(unsigned((a->n + RGROUPS - 1) / RGROUPS)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_backward_step(hipStream_t st, const nemo_float_back_args* a)
{
	if(a->n == 0) return hipSuccess;
	if(a->ring == 0 || a->t >= a->T || a->t < a->t0) return hipErrorInvalidValue;
	hipLaunchKernelGGL(backward_step_kernel, dim3(unsigned((a->n + GROUPS - 1) / GROUPS)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_push_step(hipStream_t st, const nemo_float_push_args* a)
{
	if(a->n == 0) return hipSuccess;
	if(a->t >= a->T || a->t < a->t0 || a->dmax == 0 || a->n > NEMO_FLOAT_PUSH_MAX || a->tile == 0
			|| a->tile > PUSH_BLOCK || a->pitch != nemo_float_push_pitch(a->n))
		return hipErrorInvalidValue;
	const size_t lds = (size_t(a->pitch) + 2 + a->tile) * sizeof(double);
	if(lds > NEMO_FLOAT_PUSH_LDS) return hipErrorInvalidValue;
	const dim3 grid((a->n + a->tile - 1) / a->tile);
	/* a wave per slice, and one for the neurons where there is room */
	unsigned threads = (a->slices + 1) * 64;
	if(threads < BLOCK) threads = BLOCK;
	if(threads < a->tile) threads = (a->tile + 63) / 64 * 64;
	if(threads > PUSH_BLOCK) threads = PUSH_BLOCK;
	void (*kernel)(nemo_float_push_args) = nullptr;
	switch(a->lanes) {
	case 1: kernel = backward_push_kernel<1>; break;
	case 2: kernel = backward_push_kernel<2>; break;
	case 4: kernel = backward_push_kernel<4>; break;
	case 8: kernel = backward_push_kernel<8>; break;
	case 16: kernel = backward_push_kernel<16>; break;
	case 32: kernel = backward_push_kernel<32>; break;
	default: return hipErrorInvalidValue;
	}
	hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, st, *a);
	return hipGetLastError();
}

unsigned nemo_float_push_pitch(unsigned n)
{
	return (n + 1) / 2 * 2;
}

hipError_t nemo_float_staged_attributes()
{
	const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(replay_sliced_kernel),
			hipFuncAttributeMaxDynamicSharedMemorySize, NEMO_FLOAT_REPLAY_MAX * sizeof(uint64_t));
	if(e != hipSuccess) return e;
	for(auto kernel : {backward_push_kernel<1>, backward_push_kernel<2>, backward_push_kernel<4>, backward_push_kernel<8>,
			backward_push_kernel<16>, backward_push_kernel<32>}) {
		const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
				hipFuncAttributeMaxDynamicSharedMemorySize, NEMO_FLOAT_PUSH_LDS);
		if(e != hipSuccess) return e;
	}
	return hipSuccess;
}

hipError_t nemo_launch_float_slice_weights(hipStream_t st, float* wr, const float* w, const uint32_t* user,
		const uint32_t* slice_ptr, unsigned slices, unsigned lines, size_t synapses)
{
	if(slices == 0 || lines == 0) return hipSuccess;
	if(lines > 65535) return hipErrorInvalidValue;
	hipLaunchKernelGGL(slice_weights_kernel, dim3((slices + BLOCK / 64 - 1) / (BLOCK / 64), lines), dim3(BLOCK), 0, st,
			reinterpret_cast<float4*>(wr), w, reinterpret_cast<const uint4*>(user), slice_ptr, slices, synapses);
	return hipGetLastError();
}

hipError_t nemo_launch_float_fill_slices(hipStream_t st, const nemo_float_slice_args* a)
{
	if(a->synapses == 0) return hipSuccess;
	hipLaunchKernelGGL(fill_slices_kernel, dim3(blocks_for(a->synapses)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_fill_rows(hipStream_t st, const nemo_float_rows_args* a)
{
	if(a->n == 0) return hipSuccess;
	if(a->dmax > 64 || a->lanes == 0) return hipErrorInvalidValue;
	hipLaunchKernelGGL(fill_rows_kernel, dim3((a->n + FILL_BLOCK - 1) / FILL_BLOCK), dim3(FILL_BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_begin_forward(hipStream_t st, const nemo_float_begin_forward_args* a)
{
	const size_t n = a->wr_entries > a->n ? a->wr_entries : a->n;
	if(n == 0) return hipSuccess;
	hipLaunchKernelGGL(begin_forward_kernel, dim3(blocks_for(n)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_begin_backward(hipStream_t st, const nemo_float_begin_backward_args* a)
{
	size_t n = a->synapses > a->n ? a->synapses : a->n;
	if(a->li > n) n = a->li;
	if(a->entries > n) n = a->entries;
	if(a->wr_entries > n) n = a->wr_entries;
	if(n == 0) return hipSuccess;
	hipLaunchKernelGGL(begin_backward_kernel, dim3(blocks_for(n)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

hipError_t nemo_launch_float_end_backward(hipStream_t st, const nemo_float_end_backward_args* a)
{
	const size_t n = a->entries > a->n ? a->entries : a->n;
	if(n == 0) return hipSuccess;
	hipLaunchKernelGGL(end_backward_kernel, dim3(blocks_for(n)), dim3(BLOCK), 0, st, *a);
	return hipGetLastError();
}

} // extern "C"
