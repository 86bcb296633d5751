/*
 * Kuramoto oscillator plugin (libKuramoto.so), bit-exact with
 * src/nemo/cpu/plugins/Kuramoto.cpp:14-159; built with NEMO_KURAMOTO_LAG
 * defined (plugins/KuramotoLag.hip) it is libKuramotoLag.so, bit-exact with
 * src/nemo/cpu/plugins/KuramotoLag.cpp:15-138: a third parameter alpha is
 * subtracted inside every sine, sin(theta_k - theta - alpha).
 *
 * Parameters (plugins/Kuramoto.h): omega, the phase advance per unit time,
 * and Cmean, the coupling normalisation (1 when not positive).  State: the
 * phase theta, with a history of H = 32 slots (Kuramoto.ini): the update
 * at cycle c reads slot c % H and writes slot (c + 1) % H.  Per step, one
 * RK4 step of h = 0.05 of
 *   dtheta/dt = omega + sum_k w_k sin(theta_k(c - (d_k - 1)) - theta) / Cmean
 * over the oscillator's incoming synapses k (source phase d_k - 1 cycles
 * back), summed in the order of the reverse matrix; the new phase is
 * fmodf(theta, float(2 pi)), plus 2 pi in double when theta < 0.
 * Oscillators never fire and read no synaptic current.  A synapse whose
 * delay reads the history slot the step writes (delay 32 or 64) sees what
 * the CPU backend's neuron-by-neuron loop sees: the source's new phase when
 * the source's index is lower, its old phase otherwise; the backend then
 * orders the updates in passes (nemo_hip_neuron_group.levels).
 *
 * The sine is glibc's sinf restated (glibc_math.h), which this library
 * evaluates for |x| < 120; a larger argument sets NEMO_HIP_STATUS_SINF_RANGE
 * and the host reports it.
 */
#include <hip/hip_ext.h>

#include "../plugin_device.h"

namespace {

enum { PARAM_FREQUENCY = 0, PARAM_CMEAN = 1, PARAM_ALPHA = 2 };

#ifdef NEMO_KURAMOTO_LAG
constexpr bool LAG = true;
#else
constexpr bool LAG = false;
#endif

/* 2.0f * M_PI is evaluated in double (Kuramoto.cpp:124) */
constexpr double TWO_PI = 2.0 * 3.14159265358979323846;

/* the phase stored after a step: fmodf(phase, float(2 pi)) + (2 pi if
 * phase < 0), the sum in double (Kuramoto.cpp:124, 153) */
__device__ inline float wrap_phase(float phase)
{
	const float r = nemo_math::fmodf_exact(phase, float(TWO_PI));
	return float(double(r) + (phase < 0.0f ? TWO_PI : 0.0));
}

/* The coupling term of synapse k, w sin(source phase - target phase), and its
 * operands that do not depend on the target's phase.  With `levelled`, a
 * source read at slot (cycle + 1) % H -- the slot this step writes -- is the
 * source's new phase when its index is below nl (the CPU backend updated it
 * earlier in its loop) and its old phase, kept in scratch, otherwise. */
__device__ inline float source_phase(const nemo_hip_neuron_group& g, uint32_t sd, unsigned nl, uint32_t cycle,
		bool levelled)
{
	const unsigned H = g.history;
	const uint32_t slot = (cycle - (sd >> 26)) % H; /* delay - 1 cycles back */
	const unsigned src = (sd & 0x3ffffffu) - g.start;
	return levelled && slot == (cycle + 1) % H && src >= nl ? g.scratch[src] : g.state[size_t(slot) * g.pitch + src];
}

__device__ inline float coupling(float w, float sourcePhase, float targetPhase, float alpha, bool* range)
{
	const float x = LAG ? sourcePhase - targetPhase - alpha : sourcePhase - targetPhase;
	*range = *range || __builtin_fabsf(x) >= 120.0f;
	return w * nemo_math::sinf_exact(x);
}

/* sum + the first n terms of the group's L lanes, one after another in lane
 * order, the same value in every lane.  A quad and a row of 16 add all their
 * lanes' terms by DPP broadcasts (quad_perm [q,q,q,q], row_newbcast:q), one
 * instruction a term; a wave reads the first n lanes (n uniform).  Terms past
 * the synapses are +0, which changes no sum that started from +0 (such a sum
 * is never -0). */
template<int CTRL>
__device__ inline float dpp_term(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

template<unsigned L>
__device__ inline float ordered_sum(float sum, float term, uint32_t n)
{
	static_assert(L == 4 || L == 16 || L == 64, "a quad, a row of 16 lanes or a wave");
	if constexpr(L == 4) {
		sum += dpp_term<0x00>(term);
		sum += dpp_term<0x55>(term);
		sum += dpp_term<0xaa>(term);
		sum += dpp_term<0xff>(term);
	} else if constexpr(L == 16) {
		sum += dpp_term<0x150>(term);
		sum += dpp_term<0x151>(term);
		sum += dpp_term<0x152>(term);
		sum += dpp_term<0x153>(term);
		sum += dpp_term<0x154>(term);
		sum += dpp_term<0x155>(term);
		sum += dpp_term<0x156>(term);
		sum += dpp_term<0x157>(term);
		sum += dpp_term<0x158>(term);
		sum += dpp_term<0x159>(term);
		sum += dpp_term<0x15a>(term);
		sum += dpp_term<0x15b>(term);
		sum += dpp_term<0x15c>(term);
		sum += dpp_term<0x15d>(term);
		sum += dpp_term<0x15e>(term);
		sum += dpp_term<0x15f>(term);
	} else {
		for(uint32_t i0 = 0; i0 < n; i0 += 16) {
#pragma unroll
			for(uint32_t i = 0; i < 16; ++i) {
				sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(term), int(i0 + i)));
			}
		}
	}
	return sum;
}

/* One RK4 step of oscillator nl at cycle `cycle` (Kuramoto.cpp:100-126) by a
 * group of L lanes, each a synapse of every L: the new phase, in every lane.
 * *range is set in lanes whose sine argument left (-120, 120).
 *
 * The sines of a sum are independent and take about 130 instructions each;
 * only the additions have to follow one another in reverse-matrix order
 * (sumN, Kuramoto.cpp:22-34).  One thread per oscillator took 204 us a step
 * for 1000 oscillators of 100 synapses: 16 waves on the whole chip, each a
 * chain of 400 sines.  The first KEEP synapses of a lane are loaded once for
 * the four sums. */
template<unsigned L>
__device__ inline float kuramoto_phase(const nemo_hip_neuron_group& g, const nemo_hip_step_buffers& b, unsigned nl,
		unsigned lane, uint32_t cycle, bool levelled, bool* range)
{
	constexpr uint32_t KEEP = 4;
	const size_t P = g.pitch;
	const unsigned ng = g.start + nl;
	const uint32_t r0 = b.rcm_all.ptr[ng], r1 = b.rcm_all.ptr[ng + 1];
	const float f = g.param[PARAM_FREQUENCY * P + nl];
	const float cm = g.param[PARAM_CMEAN * P + nl];
	const float Cmean = cm > 0 ? cm : 1;
	const float alpha = LAG ? g.param[PARAM_ALPHA * P + nl] : 0.0f;
	const float h = 0.05f;
	const float target = g.state[size_t(cycle % g.history) * P + nl];
	uint32_t sd[KEEP];
	float w[KEEP], phase[KEEP];
#pragma unroll
	for(uint32_t c = 0; c < KEEP; ++c) {
		const uint32_t k = r0 + c * L + lane;
		sd[c] = k < r1 ? b.rcm_all.source_delay[k] : 0u;
		w[c] = k < r1 ? b.rcm_all.weight[k] : 0.0f;
	}
#pragma unroll
	for(uint32_t c = 0; c < KEEP; ++c) {
		phase[c] = r0 + c * L + lane < r1 ? source_phase(g, sd[c], nl, cycle, levelled) : 0.0f;
	}
	auto sumN = [&](float targetPhase) {
		float sum = 0.0f;
#pragma unroll
		for(uint32_t c = 0; c < KEEP; ++c) {
			const uint32_t k = r0 + c * L;
			if(k >= r1) break; /* uniform in the group */
			const float term = k + lane < r1 ? coupling(w[c], phase[c], targetPhase, alpha, range) : 0.0f;
			sum = ordered_sum<L>(sum, term, min(L, r1 - k));
		}
		for(uint32_t k = r0 + KEEP * L; k < r1; k += L) {
			float term = 0.0f;
			if(k + lane < r1) {
				const float p = source_phase(g, b.rcm_all.source_delay[k + lane], nl, cycle, levelled);
				term = coupling(b.rcm_all.weight[k + lane], p, targetPhase, alpha, range);
			}
			sum = ordered_sum<L>(sum, term, min(L, r1 - k));
		}
		return sum;
	};
	const float k0 = f + (sumN(target) / Cmean);
	const float k1 = f + (sumN(target + k0 * 0.5f * h) / Cmean);
	const float k2 = f + (sumN(target + k1 * 0.5f * h) / Cmean);
	const float k3 = f + (sumN(target + k2 * h) / Cmean);
	return wrap_phase(target + h * (k0 + 2 * k1 + 2 * k2 + k3) / 6.0f);
}

__device__ inline uint32_t cycle_of(const nemo_hip_step_buffers& b)
{
	/* the reference's cycle is a 32-bit unsigned (H divides 2^32) */
	return uint32_t(nemo_dev::current_step(b) - b.clock->cycle_origin);
}

/* The step of the oscillator of this thread's group of L lanes, groups
 * counted from 0 over the launch's phase blocks (in passes: over the pass's
 * oscillators, group_local indices in order). */
template<unsigned L>
__device__ inline void kuramoto_group(const nemo_hip_neuron_group& g, const nemo_hip_step_buffers& b, unsigned nl,
		bool levelled)
{
	const uint32_t cycle = cycle_of(b);
	const unsigned lane = threadIdx.x % L;
	bool range = false;
	const float phase = kuramoto_phase<L>(g, b, nl, lane, cycle, levelled, &range);
	if(lane == 0) g.state[size_t((cycle + 1) % g.history) * g.pitch + nl] = phase;
	if(range) atomicOr(b.status, NEMO_HIP_STATUS_SINF_RANGE);
}

/* The first oscillator of the wave is a scalar when a wave works on one. */
template<unsigned L>
__device__ inline unsigned group_index(unsigned block)
{
	const unsigned t = threadIdx.x / L;
	const unsigned i = block * (blockDim.x / L) + t;
	return L == 64 ? unsigned(__builtin_amdgcn_readfirstlane(int(i))) : i;
}

/* One launch per step: the tiles' (empty) firing records, any propagate
 * blocks, then the oscillators, a group of L lanes each. */
template<bool CO, unsigned L>
__global__ void NEMO_UPDATE_BOUNDS(CO)
kuramoto_update(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	const unsigned before = (g.count + NEMO_UPDATE_BLOCK - 1) / NEMO_UPDATE_BLOCK + b.co.deliver_blocks
		+ b.co.stdp_blocks + b.direct.late_blocks;
	if(blockIdx.x >= before) {
		const unsigned nl = group_index<L>(blockIdx.x - before);
		if(nl < g.count) kuramoto_group<L>(g, b, nl, false);
		return;
	}
	if(CO && nemo_dev::colaunched_block(b, g)) return;
	nemo_dev::UpdateLds& U = nemo_dev::update_lds<CO>();
	if(!CO && b.direct.ring && nemo_dev::direct_block(b, g, U)) return;
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	const bool valid = nl < g.count;
	const unsigned ng = g.start + nl;
	const uint64_t hist = nemo_dev::load_history(b, ng, valid);
	nemo_dev::record_firing(b, ng, valid, false, hist); /* nothing to push */
	nemo_dev::stdp_tile(b, U, ng, valid, hist);
}

/* Update passes (nemo_hip_neuron_group.levels): first the old contents of
 * the slot the step writes into scratch, then pass by pass the passes'
 * oscillators, then the tiles' firing records. */
__global__ void __launch_bounds__(NEMO_UPDATE_BLOCK)
kuramoto_keep_next(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	if(nl < g.count) g.scratch[nl] = g.state[size_t((cycle_of(b) + 1) % g.history) * g.pitch + nl];
}

template<unsigned L>
__global__ void __launch_bounds__(NEMO_UPDATE_BLOCK)
kuramoto_pass(nemo_hip_neuron_group g, nemo_hip_step_buffers b, uint32_t first, uint32_t count)
{
	const unsigned i = group_index<L>(blockIdx.x);
	if(i < count) kuramoto_group<L>(g, b, g.level_idx[first + i], true);
}

template<bool CO>
__global__ void NEMO_UPDATE_BOUNDS(CO)
kuramoto_record(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	if(CO && nemo_dev::colaunched_block(b, g)) return;
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<CO>();
	if(!CO && b.direct.ring && nemo_dev::direct_block(b, g, L)) return;
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	const bool valid = nl < g.count;
	const unsigned ng = g.start + nl;
	const uint64_t hist = nemo_dev::load_history(b, ng, valid);
	nemo_dev::record_firing(b, ng, valid, false, hist);
	nemo_dev::stdp_tile(b, L, ng, valid, hist);
}

/* Kuramoto.cpp:137-159: the history before the first cycle, each
 * oscillator run backwards one omega per slot without coupling, from slot 0
 * into slots H-1, H-2, ..., 1 */
__global__ void __launch_bounds__(NEMO_UPDATE_BLOCK)
kuramoto_init(nemo_hip_neuron_group g)
{
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	if(nl >= g.count) return;
	const size_t P = g.pitch;
	const unsigned H = g.history;
	const float f = g.param[PARAM_FREQUENCY * P + nl];
	for(unsigned t = 0; t + 1 < H; ++t) {
		const uint32_t current = 0u - t;
		const uint32_t previous = 0u - (t + 1u);
		const float phase = g.state[size_t(current % H) * P + nl] - f;
		g.state[size_t(previous % H) * P + nl] = wrap_phase(phase);
	}
}

} // namespace

/* Lanes per oscillator of a launch over n oscillators of the group: a wave
 * each while the chip has few of them, where the length of one oscillator's
 * step counts; rows of 16 beyond, whose additions take one instruction a term
 * instead of two; quads when there are many of few synapses.  Measured (us a
 * step; one thread an oscillator, as before / row of 16 / wave, at in-degree
 * 30, 100, 300): 1000 oscillators 65, 202, 583 / 8.3, 19.2, 47.8 / 7.6, 13.1,
 * 27.8; 2000: 68, 210, 603 / 8.3, 19.6, 48.6 / 7.8, 13.7, 28.4; 4000: 69, 214,
 * 614 / 8.3, 20.0, 48.9 / 9.9, 20.5, 46.2; 16000: 72, 224, 866 / 11.8, 29.8,
 * 89.8 / 24.6, 56, 143.  64000 of in-degree 4: thread 15.4, quad 14.9, row 18.2;
 * 16000: 13.7, 8.4, 8.2. */
constexpr unsigned WAVE_MAX = 2048;
constexpr unsigned QUAD_MIN = 32768;
constexpr unsigned QUAD_DEGREE = 8;

static unsigned lanes_for(const nemo_hip_neuron_group* g, unsigned n)
{
	if(n <= WAVE_MAX) return 64;
	return n >= QUAD_MIN && g->incoming <= uint64_t(QUAD_DEGREE) * g->count ? 4 : 16;
}

template<unsigned L>
static hipError_t launch_update(hipStream_t stream, const nemo_hip_neuron_group* g, const nemo_hip_step_buffers* b)
{
	/* the group's tiles and the blocks the launch carries, then the
	 * oscillators */
	const unsigned before = nemo_dev::update_blocks(g, b);
	if(b->co.deliver_blocks || b->co.stdp_blocks) {
		const unsigned per = NEMO_COLAUNCH_BLOCK / L;
		hipExtLaunchKernelGGL((kuramoto_update<true, L>), dim3(before + (g->count + per - 1) / per),
				dim3(NEMO_COLAUNCH_BLOCK), b->co.lds_bytes, stream, b->time_start, b->time_stop, 0, *g, *b);
	} else {
		const unsigned per = NEMO_UPDATE_BLOCK / L;
		hipExtLaunchKernelGGL((kuramoto_update<false, L>), dim3(before + (g->count + per - 1) / per),
				dim3(NEMO_UPDATE_BLOCK), b->co.lds_bytes, stream, b->time_start, b->time_stop, 0, *g, *b);
	}
	return hipGetLastError();
}

template<unsigned L>
static hipError_t launch_pass(hipStream_t stream, const nemo_hip_neuron_group* g, const nemo_hip_step_buffers* b,
		uint32_t first, uint32_t count)
{
	const unsigned per = NEMO_UPDATE_BLOCK / L;
	hipLaunchKernelGGL(kuramoto_pass<L>, dim3((count + per - 1) / per), dim3(NEMO_UPDATE_BLOCK), 0, stream, *g, *b, first,
			count);
	return hipGetLastError();
}

extern "C" hipError_t
hip_update_neurons(hipStream_t stream, const nemo_hip_neuron_group* g, const nemo_hip_step_buffers* b)
{
	if(g->count == 0) return hipSuccess;
	if(!b->rcm_all.ptr || !b->status || g->history < 1) return hipErrorInvalidValue;
	if(!g->level_ptr) {
		const unsigned L = lanes_for(g, g->count);
		return L == 64 ? launch_update<64>(stream, g, b) : L == 16 ? launch_update<16>(stream, g, b)
			: launch_update<4>(stream, g, b);
	}
	if(!g->scratch || !g->level_idx || g->levels < 1) return hipErrorInvalidValue;
	const unsigned tiles = (g->count + NEMO_UPDATE_BLOCK - 1) / NEMO_UPDATE_BLOCK;
	const unsigned blocks = nemo_dev::update_blocks(g, b);
	const bool co = b->co.deliver_blocks || b->co.stdp_blocks;
	hipExtLaunchKernelGGL(kuramoto_keep_next, dim3(tiles), dim3(NEMO_UPDATE_BLOCK), 0, stream, b->time_start,
			nullptr, 0, *g, *b);
	hipError_t e = hipGetLastError();
	for(unsigned l = 0; l < g->levels && e == hipSuccess; ++l) {
		const uint32_t first = g->level_ptr[l], count = g->level_ptr[l + 1] - first;
		if(count == 0) continue;
		const unsigned L = lanes_for(g, count);
		e = L == 64 ? launch_pass<64>(stream, g, b, first, count) : L == 16 ? launch_pass<16>(stream, g, b, first, count)
			: launch_pass<4>(stream, g, b, first, count);
	}
	if(e != hipSuccess) return e;
	if(co) {
		hipExtLaunchKernelGGL(kuramoto_record<true>, dim3(blocks), dim3(NEMO_COLAUNCH_BLOCK), b->co.lds_bytes, stream,
				nullptr, b->time_stop, 0, *g, *b);
	} else {
		hipExtLaunchKernelGGL(kuramoto_record<false>, dim3(blocks), dim3(NEMO_UPDATE_BLOCK), b->co.lds_bytes, stream,
				nullptr, b->time_stop, 0, *g, *b);
	}
	return hipGetLastError();
}

extern "C" hipError_t
hip_init_neurons(hipStream_t stream, const nemo_hip_neuron_group* g, const nemo_hip_step_buffers*)
{
	if(g->count == 0 || g->history < 2) return hipSuccess;
	hipLaunchKernelGGL(kuramoto_init, dim3((g->count + NEMO_UPDATE_BLOCK - 1) / NEMO_UPDATE_BLOCK),
			dim3(NEMO_UPDATE_BLOCK), 0, stream, *g);
	return hipGetLastError();
}
