/*
 * Hodgkin-Huxley neuron plugin (libHH.so).
 *
 * Bit-exact with src/nemo/cpu/plugins/HH.cpp:14-138: 999 Euler substeps
 * ((int)(1/0.001f)) of the classic HH equations with glibc-exact expf; the
 * neuron fires on the first downturn of v (change < -1e-9) once the timer
 * cycle is >= 10.  State v, n, m, h, dir (HH.ini: 5 state variables, no
 * parameters).  Per-type arrays are indexed within the type (see QIF).
 *
 * A step is three launches when the group has its four scratch planes
 * (HH.ini [hip] scratch-planes=4): the tiles' input gather (one thread per
 * neuron, as every model), the substeps with sixteen lanes per neuron in
 * one-wave blocks -- six lanes evaluate the six rate functions (each an
 * expf), three advance the gates and five form the terms of the current -- and
 * the tiles' firing record.  One wave of a tile block otherwise spends each
 * substep on six exponentials for its 64 neurons, one wave per SIMD on a few
 * CUs; the split spreads the same arithmetic, operation for operation, over
 * sixteen times as many waves.  Without scratch planes the single launch runs.
 */
#include <hip/hip_ext.h>

#include "../plugin_device.h"

namespace {

using nemo_math::expf_exact;

/* HH.cpp:26-39 */
constexpr float DT = 0.001f;
constexpr float G_NA = 120.0f;
constexpr float G_K = 36.0f;
constexpr float G_L = 0.3f;
constexpr float E_NA = 115.0f - 65.0f;
constexpr float E_K = -12.0f - 65.0f;
constexpr float E_L = 10.6f - 65.0f;
constexpr float C_M = 1.0f;
constexpr float REV_E = 0.0f;
constexpr float REV_I = -70.0f;

/* scratch planes of the split step */
enum { SCR_E = 0, SCR_I = 1, SCR_X = 2, SCR_FIRED = 3 };
constexpr unsigned LANES = 16;     /* per neuron in the substep launch: one DPP row */
constexpr unsigned SUB_BLOCK = 64; /* one wave: four neurons */

/* The value of lane Q of this lane's row of 16 (DPP row_share). */
template<int Q>
__device__ inline float row_lane(float v)
{
	return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + Q, 0xf, 0xf, true));
}

/* The gating and membrane update of one substep from the six rates (HH.cpp:44-62). */
__device__ inline void hh_substep(float& v, float& n, float& m, float& h, float& dir, bool& fired, uint64_t cycle,
		float Excit, float Inhib, float Exter, float alphan, float alpham, float alphah, float betan,
		float betam, float betah)
{
	const float I = (Excit * (REV_E - v)) + (Inhib * ((REV_I - v) / -1)) + Exter;
	m = m + DT * (alpham * (1.0f - m) - betam * m);
	n = n + DT * (alphan * (1.0f - n) - betan * n);
	h = h + DT * (alphah * (1.0f - h) - betah * h);
	const float Ik = G_NA * (m * m * m) * h * (v - E_NA) + G_K * (n * n * n * n) * (v - E_K) + G_L * (v - E_L);
	const float newv = v + DT * (-Ik + I) / C_M;
	const float new_dir = (newv - v);
	const float change = (dir < 0) | (newv < -45) ? 0 : new_dir;
	dir = new_dir;
	if(!fired && cycle >= 10) fired = double(change) < -0.000000001;
	v = newv;
}

/* Single launch: gather, substeps and firing record per tile. */
/* CO: the launch may carry propagate blocks after the tiles (compiled
 * out otherwise, which leaves the update far fewer registers) */
template<bool CO>
__global__ void NEMO_UPDATE_BOUNDS(CO)
hh_update(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	if(CO && nemo_dev::colaunched_block<true>(b, g)) return;
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<CO>();
	if(!CO && b.direct.ring && nemo_dev::direct_block(b, g, L)) return;
	if(!nemo_dev::gather_input<CO ? NEMO_COLAUNCH_BLOCK : NEMO_TILE>(b, g, L)) return; /* helpers end here */
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	const bool valid = nl < g.count;
	const unsigned nn = g.start + nl;
	const uint64_t hist = nemo_dev::load_history(b, nn, valid);
	bool fired = false;

	if(valid) {
		const size_t P = g.pitch;
		float* s = g.state;
		float v = s[0 * P + nl];
		float n = s[1 * P + nl];
		float m = s[2 * P + nl];
		float h = s[3 * P + nl];
		float dir = s[4 * P + nl];
		float Excit, Inhib;
		nemo_dev::take_current(b, L.input, nn, Excit, Inhib);
		const float Exter = nemo_dev::take_external(b, nn);
		const uint64_t cycle = nemo_dev::current_step(b) - b.clock->cycle_origin;
		const int inc_max = (int)(1 / DT);
		for(int t = 0; t < inc_max; ++t) {
			const float alphan = (0.1f - 0.01f * (v + 65.0f)) / (expf_exact(1.0f - 0.1f * (v + 65.0f)) - 1.0f);
			const float alpham = (2.5f - 0.1f * (v + 65.0f)) / (expf_exact(2.5f - 0.1f * (v + 65.0f)) - 1.0f);
			const float alphah = 0.07f * expf_exact(-(v + 65.0f) / 20.0f);
			const float betan = 0.125f * expf_exact(-(v + 65.0f) / 80.0f);
			const float betam = 4.0f * expf_exact(-(v + 65.0f) / 18.0f);
			const float betah = 1.0f / (expf_exact(3.0f - 0.1f * (v + 65.0f)) + 1.0f);
			hh_substep(v, n, m, h, dir, fired, cycle, Excit, Inhib, Exter, alphan, alpham, alphah, betan, betam, betah);
		}
		fired = fired || nemo_dev::stimulated(b, nn);
		s[0 * P + nl] = v;
		s[1 * P + nl] = n;
		s[2 * P + nl] = m;
		s[3 * P + nl] = h;
		s[4 * P + nl] = dir;
	}
	nemo_dev::record_firing<CO>(b, L, nn, valid, fired, hist);
	nemo_dev::stdp_tile(b, L, nn, valid, hist);
}

/* Split step, launch 1: the tiles' synaptic and external input. */
/* CO: the launch may carry propagate blocks after the tiles (compiled
 * out otherwise, which leaves the update far fewer registers) */
template<bool CO>
__global__ void NEMO_UPDATE_BOUNDS(CO)
hh_input(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	if(CO && nemo_dev::colaunched_block<true>(b, g)) return;
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<CO>();
	if(!CO && b.direct.ring && nemo_dev::direct_block(b, g, L)) return;
	if(!nemo_dev::gather_input<CO ? NEMO_COLAUNCH_BLOCK : NEMO_TILE>(b, g, L)) return; /* helpers end here */
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	if(nl < g.count) {
		const unsigned nn = g.start + nl;
		const size_t P = g.pitch;
		float Excit, Inhib;
		nemo_dev::take_current(b, L.input, nn, Excit, Inhib);
		g.scratch[SCR_E * P + nl] = Excit;
		g.scratch[SCR_I * P + nl] = Inhib;
		g.scratch[SCR_X * P + nl] = nemo_dev::take_external(b, nn);
	}
}

/* lane i + N of the row for lane i (DPP row_shl) */
template<int N>
__device__ inline float row_up(float x)
{
	return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x100 + N, 0xf, 0xf, true));
}

/* Lane i + 1 of the row for the lanes of the row's first four, old for the
 * others. */
__device__ inline float row_up_first_bank(float old, float x)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), 0x101, 0xf, 0x1, false));
}

/* n / d, correctly rounded, where no intermediate value leaves the normal
 * range: the reciprocal refined once, the quotient twice (both with exact
 * FMA residuals).  The first quotient is taken from the unrefined reciprocal,
 * which the second refinement absorbs (the one before it leaves 2^-20 ulp
 * beside the rounding, and the last is exact for any faithful quotient). */
__device__ inline float div_normal(float n, float d)
{
	const float r0 = __builtin_amdgcn_rcpf(d);
	const float q0 = n * r0;
	const float e = __builtin_fmaf(-d, r0, 1.0f);
	const float s0 = __builtin_fmaf(-d, q0, n);
	const float r = __builtin_fmaf(e, r0, r0);
	const float q1 = __builtin_fmaf(s0, r, q0);
	const float s1 = __builtin_fmaf(-d, q1, n);
	return __builtin_fmaf(s1, r, q1);
}

/* The lanes of a neuron's row in the substep launch.  M, H and N hold the
 * gates m, h and n and evaluate their alphas, the lanes eight up their betas.
 * The sodium term is formed at M (with the h of the lane above), the
 * potassium term at N, the parts of the current that no gate scales at LEAK,
 * INH and EXC. */
enum { M = 0, H = 1, LEAK = 2, N = 4, INH = 5, EXC = 6, BETA = 8 };

struct HHLane {
	/* the exponent is a0 - a1 y + k y, with y = v + 65: a0 - 0.1 y
	 * (k = 0), or -y / c as a product with 1 / c in two floats */
	float a0, a1, k;
	/* the rate is (c0 - c1 y) / (e + e0), or fac e */
	float c0, c1, e0, fac;
	bool quotient;
	/* the current's terms: conductance (factor of h at M) and reversal potential */
	float G, E;
	bool power4;
	float divisor; /* of the exponent, for the general path */
};

__device__ inline HHLane hh_lane(unsigned q, float Excit, float Inhib)
{
	HHLane L;
	const bool alpham = q == M, alphah = q == H, alphan = q == N, betam = q == BETA + M, betan = q == BETA + N;
	L.quotient = !(alphah || betam || betan); /* alphan, alpham; betah, and the lanes without a rate */
	L.divisor = alphah ? 20.0f : betan ? 80.0f : betam ? 18.0f : 1.0f;
	const float c = L.divisor;
	const float inv = 1.0f / c;
	L.a0 = alphan ? 1.0f : alpham ? 2.5f : L.quotient ? 3.0f : 0.0f;
	L.a1 = L.quotient ? 0.1f : float(1.0 / double(c) - double(inv));
	L.k = L.quotient ? 0.0f : -inv;
	L.c0 = alphan ? 0.1f : alpham ? 2.5f : 1.0f;
	L.c1 = alphan ? 0.01f : alpham ? 0.1f : 0.0f;
	L.e0 = alphan || alpham ? -1.0f : 1.0f;
	L.fac = alphah ? 0.07f : betan ? 0.125f : 4.0f;
	L.G = q == M ? G_NA : q == LEAK ? G_L : q == INH ? Inhib : q == EXC ? -Excit : G_K;
	L.E = q == M ? E_NA : q == LEAK ? E_L : q == INH ? REV_I : q == EXC ? REV_E : E_K;
	L.power4 = q == N;
	return L;
}

/* The state of a row in its substeps: v, dir and turn the same in every lane. */
struct HHRow {
	float v;     /* potential */
	float x;     /* gate of the lane */
	float dir;   /* last change of v */
	float turn;  /* lowest change of v that may count as a downturn */
	float times; /* last factor of the gates' product: h at M, G_K elsewhere */
};

/* The lane's gate from its rate (HH.cpp:55-57), and the current it scales
 * (HH.cpp:58-59): G m^3 h (v - E) at M, n^4 G (v - E) at N; then v.  A DPP
 * move waits two instructions for its operand: fill(0), fill(1) and fill(2)
 * are work that may stand there. */
template<class Fill>
__device__ inline float hh_advance(const HHLane& L, HHRow& s, float rate, float rest, float drive, float part, float I,
		Fill fill)
{
	s.x = s.x + DT * (rate * rest - row_up<BETA>(rate) * s.x);
	s.times = row_up_first_bank(s.times, s.x);
	const float term = (((s.x * s.x * s.x) * (L.power4 ? s.x : G_NA)) * s.times) * drive;
	__builtin_amdgcn_sched_barrier(0);
	fill(0);
	__builtin_amdgcn_sched_barrier(0);
	const float sodium = row_lane<M>(term);
	__builtin_amdgcn_sched_barrier(0);
	fill(1);
	__builtin_amdgcn_sched_barrier(0);
	const float gated = sodium + row_lane<N>(term);
	__builtin_amdgcn_sched_barrier(0);
	fill(2);
	__builtin_amdgcn_sched_barrier(0);
	const float Ik = gated + row_lane<LEAK>(part);
	return s.v + DT * (-Ik + I) / C_M;
}

/* The current that no gate scales (HH.cpp:54; its factors with two signs
 * moved). */
__device__ inline float hh_input_current(float part, float Exter)
{
	return (row_lane<EXC>(part) + row_lane<INH>(part)) + Exter;
}

/* COUNT substeps without the special cases: they hold while |v + 65| is at
 * most FAST_Y, of which top is the highest seen, and where a quotient by 0
 * (at v = -55 and -40) leaves a NaN for a true infinity, v becomes NaN.  What
 * the potential does not wait for is done while the table entry of the
 * exponential travels, or in the waits of hh_advance.
 *
 * A change of v is noted as a downturn one substep later: it counts unless
 * the change before it was negative or v is below -45.  The latter as v's
 * difference from the float below -45, which at or above -45 is far below
 * -1e-9 and under -45 not negative. */
constexpr float FAST_Y = 256.0f;

template<int COUNT>
__device__ inline float hh_fast_substeps(const HHLane& L, const uint64_t* s_exp, float Exter, HHRow& s)
{
	float top = 0.0f;
	float before = -1.0f; /* the change before dir; the first dir is not counted */
	constexpr float under = -45.0f - 0x1p-18f;
	auto note = [&](float counted, float low) { s.turn = __builtin_fminf(s.turn, __builtin_fmaxf(counted, low)); };
#pragma unroll 37
	for(int i = 0; i < COUNT; ++i) {
		const float y = s.v + 65.0f;
		const nemo_math::ExpfParts p =
				nemo_math::expf_main_begin(__builtin_fmaf(L.k, y, L.a0 - L.a1 * y), s_exp);
		__builtin_amdgcn_sched_barrier(0);
		const double exp_poly = nemo_math::expf_main_poly(p);
		const float poly = L.c0 - L.c1 * y;
		const float drive = s.v - L.E;
		const float part = L.G * drive;
		const float I = hh_input_current(part, Exter);
		const float rest = 1.0f - s.x;
		__builtin_amdgcn_sched_barrier(0);
		const float e = nemo_math::expf_main_end(p, exp_poly);
		float quotient = div_normal(poly, e + L.e0);
		asm("" : "+v"(quotient)); /* one instruction stream for all lanes */
		float low, counted;
		const float newv = hh_advance(L, s, L.quotient ? quotient : L.fac * e, rest, drive, part, I, [&](int k) {
			if(k == 0) {
				top = __builtin_fmaxf(top, __builtin_fabsf(y));
				low = under - s.v;
			} else if(k == 1) {
				counted = before < 0 ? 0.0f : s.dir;
				before = s.dir;
			} else {
				note(counted, low);
			}
		});
		s.dir = newv - s.v;
		s.v = newv;
	}
	note(before < 0 ? 0.0f : s.dir, under - s.v);
	return top;
}

/* One substep in general form, whatever the values. */
__device__ inline void hh_substep_any(const HHLane& L, const uint64_t* s_exp, float Exter, HHRow& s)
{
	const float y = s.v + 65.0f;
	const float arg = L.quotient ? L.a0 - L.a1 * y : nemo_math::div_by_const(-y, L.divisor, -L.k);
	const float e = nemo_math::expf_exact_tab(arg, s_exp);
	/* without c1, the quotient's numerator is 1 whatever y */
	const float poly = L.c1 == 0.0f ? 1.0f : L.c0 - L.c1 * y;
	const float rate = L.quotient ? poly / (e + L.e0) : L.fac * e;
	const float drive = s.v - L.E;
	const float part = L.G * drive;
	const float newv = hh_advance(L, s, rate, 1.0f - s.x, drive, part, hh_input_current(part, Exter),
			[](int) {});
	const float change = newv - s.v;
	const float counted = s.dir < 0 || newv < -45 ? 0.0f : change;
	if(counted < s.turn) s.turn = counted;
	s.dir = change;
	s.v = newv;
}

/* Split step, launch 2: the substeps, LANES lanes per neuron.  The rates are
 * evaluated side by side, each lane with constants of its own in one stream
 * of instructions; the gates and the terms of the current likewise (HHLane),
 * and DPP moves hand on what another lane needs.  Every value goes through
 * the operations of the single launch in their order, so it has its bits.
 *
 * The substeps are one dependent chain on a wave alone on its SIMD, which
 * issues an instruction every four cycles at best, so the number of
 * instructions of a substep counts, whichever lanes they serve, and the
 * latencies that nothing independent fills.  So BLOCK substeps at a time run
 * without the special cases of the exponential and of the division and
 * without branches; top, the highest |v + 65| that they saw, and a v that has
 * become NaN, which it stays, tell where that was not right, and then the
 * block is done again in general form.  A v that was NaN before makes the
 * same NaNs either way: a neuron whose potential once met the 0 / 0 at -55 or
 * -40 is one of those for good.
 *
 * 400 neurons: 252 us before the gates, the current's terms and the firing
 * test were spread over lanes and shortened (117 instructions a substep, of
 * which the gates and currents ran redundantly in every lane), 126 us now (70
 * instructions, 290 cycles; 130 with the loop unrolled by 3 and without the
 * fills). */
__global__ void __launch_bounds__(SUB_BLOCK)
hh_substeps(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	__shared__ uint64_t s_exp[32 * nemo_math::EXPF_REPEATS];
	for(unsigned i = threadIdx.x; i < 32 * nemo_math::EXPF_REPEATS; i += SUB_BLOCK)
		s_exp[i] = nemo_math::expf_table(i);
	__syncthreads();
	const unsigned t = blockIdx.x * SUB_BLOCK + threadIdx.x;
	const unsigned nl = t / LANES;
	const unsigned q = t % LANES;
	if(nl >= g.count) return; /* whole groups of LANES lanes */
	const size_t P = g.pitch;
	float* s = g.state;
	const unsigned gate = q == N ? 1 : q == M ? 2 : 3; /* n, m, h */
	HHRow row = {s[0 * P + nl], s[gate * P + nl], s[4 * P + nl], 0.0f, G_K};
	const float Excit = g.scratch[SCR_E * P + nl];
	const float Inhib = g.scratch[SCR_I * P + nl];
	const float Exter = g.scratch[SCR_X * P + nl];
	const uint64_t cycle = nemo_dev::current_step(b) - b.clock->cycle_origin;
	const HHLane L = hh_lane(q, Excit, Inhib);
	constexpr int inc_max = (int)(1 / DT);
	constexpr int BLOCK = 111;
	static_assert(inc_max % BLOCK == 0, "blocks of substeps");
	for(int it = 0; it < inc_max; it += BLOCK) {
		const HHRow start = row;
		const float top = hh_fast_substeps<BLOCK>(L, s_exp, Exter, row);
		if(__ballot(!(top <= FAST_Y) || (row.v != row.v && start.v == start.v))) {
			row = start;
#pragma unroll 1
			for(int i = 0; i < BLOCK; ++i) hh_substep_any(L, s_exp, Exter, row);
		}
	}
	if(q == M) {
		s[0 * P + nl] = row.v;
		s[4 * P + nl] = row.dir;
		/* in double the threshold lies between this float and the one below */
		g.scratch[SCR_FIRED * P + nl] = cycle >= 10 && row.turn < -0.000000001f ? 1.0f : 0.0f;
	}
	if(q == M || q == H || q == N) s[gate * P + nl] = row.x;
}

/* Split step, launch 3: the tiles' firing record (and per-tile STDP). */
__global__ void __launch_bounds__(NEMO_UPDATE_BLOCK)
hh_record(nemo_hip_neuron_group g, nemo_hip_step_buffers b)
{
	nemo_dev::UpdateLds& L = nemo_dev::update_lds<false>();
	const unsigned nl = blockIdx.x * NEMO_UPDATE_BLOCK + threadIdx.x;
	const bool valid = nl < g.count;
	const unsigned nn = g.start + nl;
	const uint64_t hist = nemo_dev::load_history(b, nn, valid);
	nemo_dev::begin_push(b, L, nn);
	bool fired = false;
	if(valid) fired = g.scratch[SCR_FIRED * g.pitch + nl] != 0.0f || nemo_dev::stimulated(b, nn);
	nemo_dev::record_firing<false>(b, L, nn, valid, fired, hist);
	nemo_dev::stdp_tile(b, L, nn, valid, hist);
}

} // namespace

extern "C" hipError_t
hip_update_neurons(hipStream_t stream, const nemo_hip_neuron_group* g, const nemo_hip_step_buffers* b)
{
	if(g->count == 0) return hipSuccess;
	const unsigned tiles = (g->count + NEMO_UPDATE_BLOCK - 1) / NEMO_UPDATE_BLOCK;
	const unsigned blocks = nemo_dev::update_blocks(g, b);
	if(!g->scratch) {
		if(b->co.deliver_blocks || b->co.stdp_blocks) {
			hipExtLaunchKernelGGL(hh_update<true>, dim3(blocks), dim3(NEMO_COLAUNCH_BLOCK), b->co.lds_bytes, stream,
					b->time_start, b->time_stop, 0, *g, *b);
		} else {
			hipExtLaunchKernelGGL(hh_update<false>, dim3(blocks), dim3(NEMO_UPDATE_BLOCK), b->co.lds_bytes, stream,
					b->time_start, b->time_stop, 0, *g, *b);
		}
		return hipGetLastError();
	}
	if(b->co.deliver_blocks || b->co.stdp_blocks) {
		hipExtLaunchKernelGGL(hh_input<true>, dim3(blocks), dim3(NEMO_COLAUNCH_BLOCK), b->co.lds_bytes, stream,
				b->time_start, nullptr, 0, *g, *b);
	} else {
		hipExtLaunchKernelGGL(hh_input<false>, dim3(blocks), dim3(NEMO_UPDATE_BLOCK), b->co.lds_bytes, stream,
				b->time_start, nullptr, 0, *g, *b);
	}
	hipError_t e = hipGetLastError();
	if(e != hipSuccess) return e;
	const unsigned sub = unsigned((size_t(g->count) * LANES + SUB_BLOCK - 1) / SUB_BLOCK);
	hipLaunchKernelGGL(hh_substeps, dim3(sub), dim3(SUB_BLOCK), 0, stream, *g, *b);
	e = hipGetLastError();
	if(e != hipSuccess) return e;
	hipExtLaunchKernelGGL(hh_record, dim3(tiles), dim3(NEMO_UPDATE_BLOCK), 0, stream, nullptr, b->time_stop, 0, *g,
			*b);
	return hipGetLastError();
}

extern "C" hipError_t
hip_init_neurons(hipStream_t, const nemo_hip_neuron_group*, const nemo_hip_step_buffers*)
{
	return hipSuccess; /* src/nemo/cpu/plugins/default_init.c:3-21: nothing to do */
}
