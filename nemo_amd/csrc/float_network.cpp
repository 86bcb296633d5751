/*
 * Host side of the float-weight mode: connectivity in forward (network)
 * order and reverse (by target) order, and the forward / checkpointed
 * adjoint step loops over the kernels of float_mode.hip.
 */
#include "backend.hpp"
#include "float_mode.h"

#include <algorithm>
#include <cstdlib>
#include <string>
#include <vector>

namespace nemo_hip {

FloatNetwork::FloatNetwork(const Network& net, int device) : m_device(device < 0 ? 0 : device)
{
	HIP_CHECK(hipSetDevice(m_device));
	unsigned types = 0;
	const Network::Group* grp = nullptr;
	for(unsigned t = 0; t < net.types.size(); ++t) {
		if(net.groups[t].gidx.empty()) continue;
		++types;
		grp = &net.groups[t];
		if(net.types[t].name != "Izhikevich") {
			throw Error(NEMO_API_UNSUPPORTED, "the float-weight mode supports Izhikevich neurons only");
		}
	}
	if(types != 1) {
		throw Error(NEMO_INVALID_INPUT, "the float-weight mode needs one neuron type");
	}
	m_n = grp->gidx.size();
	if(m_n >= (size_t(1) << 26)) throw Error(NEMO_API_UNSUPPORTED, "too many neurons for the float-weight mode");
	std::vector<char> seen(m_n, 0);
	for(unsigned g : grp->gidx) {
		if(g >= m_n || seen[g]) {
			throw Error(NEMO_INVALID_INPUT, "the float-weight mode needs neuron indices 0..N-1");
		}
		seen[g] = 1;
	}
	m_s = net.synapseCount;
	if(m_s >= (size_t(1) << 32)) throw Error(NEMO_API_UNSUPPORTED, "too many synapses for the float-weight mode");
	m_D = std::max(1u, net.maxDelay);

	/* NEMO_HIP_FLOAT_STAGE=0 stages nothing in LDS */
	const char* env = std::getenv("NEMO_HIP_FLOAT_STAGE");
	const bool mayStage = !env || std::string(env) != "0";
	/* the backward's staged form, where a step's input adjoints fit in LDS
	 * (20 398 neurons): 256 blocks share the neurons, one per compute unit,
	 * since each stages all the adjoints */
	m_tile = unsigned((m_n + 255) / 256);
	m_pushPitch = nemo_float_push_pitch(unsigned(m_n));
	m_push = mayStage && (size_t(m_pushPitch) + 2 + m_tile) * sizeof(double) <= NEMO_FLOAT_PUSH_LDS;
	std::vector<uint32_t> rowLen(m_push ? m_n * m_D : 0, 0); /* synapses by (source, delay) */

	/* forward order = network order: sources ascending, insertion order */
	std::vector<uint32_t> fptr(m_n + 1, 0), ftd(std::max<size_t>(1, m_s)), tgtOf(std::max<size_t>(1, m_s));
	std::vector<uint32_t> incoming(m_n + 1, 0);
	size_t k = 0;
	for(auto& kv : net.fcm) {
		const Network::Axon& ax = kv.second;
		if(kv.first >= m_n) {
			throw Error(NEMO_INVALID_INPUT, "Invalid synapse source neuron " + std::to_string(kv.first));
		}
		fptr[kv.first + 1] = uint32_t(ax.target.size());
		for(size_t i = 0; i < ax.target.size(); ++i, ++k) {
			const uint32_t tgt = ax.target[i];
			if(tgt >= m_n) throw Error(NEMO_INVALID_INPUT, "Invalid synapse target neuron " + std::to_string(tgt));
			ftd[k] = tgt | (uint32_t(ax.delay[i] - 1) << 26);
			if(!rowLen.empty()) rowLen[kv.first * size_t(m_D) + ax.delay[i] - 1] += 1;
			tgtOf[k] = tgt;
			incoming[tgt + 1] += 1;
		}
	}
	for(size_t i = 0; i < m_n; ++i) fptr[i + 1] += fptr[i];
	/* reverse order: by target, then network order */
	for(size_t i = 0; i < m_n; ++i) incoming[i + 1] += incoming[i];
	std::vector<uint32_t> cursor(incoming.begin(), incoming.end() - 1);
	std::vector<uint32_t> rsd(std::max<size_t>(1, m_s)), ruser(std::max<size_t>(1, m_s));
	k = 0;
	for(auto& kv : net.fcm) {
		const Network::Axon& ax = kv.second;
		for(size_t i = 0; i < ax.target.size(); ++i, ++k) {
			const uint32_t pos = cursor[tgtOf[k]]++;
			rsd[pos] = kv.first | (uint32_t(ax.delay[i] - 1) << 26);
			ruser[pos] = uint32_t(k);
		}
	}
	auto upload = [](DeviceArray<uint32_t>& d, const std::vector<uint32_t>& h) {
		d.allocate(h.size());
		HIP_CHECK(hipMemcpy(d.ptr, h.data(), d.bytes(), hipMemcpyHostToDevice));
	};
	upload(m_fcmPtr, fptr);
	upload(m_fcmTd, ftd);
	PushRows push;
	if(m_push) {
		push = pushRows(rowLen);
		m_push = !push.ptr.empty();
	}
	if(m_push) {
		upload(m_rowSlices, push.ptr);
		m_rows.allocate(push.rows.size());
		HIP_CHECK(hipMemcpy(m_rows.ptr, push.rows.data(), m_rows.bytes(), hipMemcpyHostToDevice));
		const size_t entries = std::max<size_t>(1, push.ptr.back()) * 256;
		m_rowUser.allocate(entries);
		m_rowTarget.allocate(entries);
		m_rowW.allocate(entries);
		m_rowGw.allocate(entries);
		HIP_CHECK(hipMemset(m_rowUser.ptr, 0xff, m_rowUser.bytes()));
		HIP_CHECK(hipMemsetD16(reinterpret_cast<hipDeviceptr_t>(m_rowTarget.ptr), uint16_t(m_pushPitch), entries));
		DeviceArray<uint32_t> rowAt;
		upload(rowAt, push.at);
		nemo_float_rows_args fill = {};
		fill.n = unsigned(m_n);
		fill.dmax = m_D;
		fill.lanes = m_pushLanes;
		fill.fcm_ptr = m_fcmPtr.ptr;
		fill.fcm_td = m_fcmTd.ptr;
		fill.row_at = rowAt.ptr;
		fill.row_user = m_rowUser.ptr;
		fill.row_target = m_rowTarget.ptr;
		HIP_CHECK(nemo_launch_float_fill_rows(nullptr, &fill));
		HIP_CHECK(hipStreamSynchronize(nullptr));
		m_fcmPtr.release();
		m_fcmTd.release();
		m_LI.allocate(2 * size_t(m_pushPitch) + size_t(m_D) * m_n);
	} else {
		m_LI.allocate(size_t(m_D + 1) * m_n);
	}
	upload(m_rcmPtr, incoming);
	upload(m_rcmSd, rsd);
	upload(m_rcmUser, ruser);
	m_v.allocate(m_n);
	m_u.allocate(m_n);
	m_LV.allocate(m_n);
	m_LU.allocate(m_n);
	m_pitch = nemo_float_bitmap_pitch(unsigned(m_n));
	/* stage the recent spike bitmaps in LDS when they fit and cost fewer
	 * cache lines than a block's (32 neurons') spike gathers would */
	const size_t stage = nemo_float_stage_bytes(unsigned(m_n), m_D);
	m_stage = mayStage && stage <= NEMO_FLOAT_STAGE_MAX && stage / 64 <= 32 * (m_s / std::max<size_t>(1, m_n));
	/* the sliced form reads the staged bitmaps; where it cannot be, or where
	 * its weights do not fit a workspace that the plain order fits, the sums
	 * are the same */
	if(m_stage) {
		const std::vector<uint32_t> slices = pullSlices(incoming);
		if(!slices.empty()) {
			upload(m_slicePtr, slices);
			const size_t entries = std::max<size_t>(1, slices.back()) * 256;
			m_sliceSd.allocate(entries);
			m_sliceUser.allocate(entries);
			HIP_CHECK(hipMemset(m_sliceSd.ptr, 0, m_sliceSd.bytes()));
			HIP_CHECK(hipMemset(m_sliceUser.ptr, 0xff, m_sliceUser.bytes()));
			nemo_float_slice_args fill = {};
			fill.n = unsigned(m_n);
			fill.dmax = m_D;
			fill.synapses = m_s;
			fill.rcm_ptr = m_rcmPtr.ptr;
			fill.rcm_sd = m_rcmSd.ptr;
			fill.rcm_user = m_rcmUser.ptr;
			fill.slice_ptr = m_slicePtr.ptr;
			fill.slice_sd = m_sliceSd.ptr;
			fill.slice_user = m_sliceUser.ptr;
			HIP_CHECK(nemo_launch_float_fill_slices(nullptr, &fill));
			HIP_CHECK(hipStreamSynchronize(nullptr));
		}
	}
	HIP_CHECK(nemo_float_staged_attributes());
	m_wr.allocate(std::max(std::max<size_t>(1, m_s), m_sliceUser.n));
}

/* The slices of backward_push_kernel: a block's rows of (source, delay), longest
 * first.  rowLen holds each row's synapses. */
FloatNetwork::PushRows FloatNetwork::pushRows(const std::vector<uint32_t>& rowLen)
{
	/* as many lanes per row as leave a wave for the neurons, and four
	 * synapses or more per lane on average: 100 training steps of 10 000 x 200
	 * (rows of 20, two lanes) take 1327 us, with one lane 1430, with four
	 * 1424; 50 steps of 1000 x 100 (rows of 10, two lanes) 441, 493 and 443 */
	const size_t rowsPerBlock = size_t(m_tile) * m_D;
	const size_t perRow = m_s / std::max<size_t>(1, m_n * m_D);
	m_pushLanes = 1;
	while(m_pushLanes < 32 && rowsPerBlock * m_pushLanes * 2 <= 960 && m_pushLanes * 8 <= perRow) m_pushLanes *= 2;
	const unsigned L = m_pushLanes;
	const unsigned groups = 64 / L;
	m_slices = unsigned((rowsPerBlock + groups - 1) / groups);
	const size_t blocks = (m_n + m_tile - 1) / m_tile;

	PushRows out;
	out.ptr.assign(blocks * m_slices + 1, 0);
	out.rows.assign(blocks * m_slices * 64, nemo_float_row{0, 0});
	out.at.assign(m_n * m_D, 0);
	std::vector<uint32_t> order, bins;
	for(size_t b = 0; b < blocks; ++b) {
		const size_t first = b * m_tile;
		const size_t rows = std::min<size_t>(m_tile, m_n - first) * m_D;
		const uint32_t* len = rowLen.data() + first * m_D;
		const uint32_t longestRow = *std::max_element(len, len + rows);
		bins.assign(longestRow + 2, 0);
		for(size_t r = 0; r < rows; ++r) bins[longestRow - len[r] + 1] += 1;
		for(size_t k = 0; k + 1 < bins.size(); ++k) bins[k + 1] += bins[k];
		order.resize(rows);
		for(size_t r = 0; r < rows; ++r) order[bins[longestRow - len[r]]++] = uint32_t(r);
		for(unsigned s = 0; s < m_slices; ++s) {
			const size_t slice = b * m_slices + s;
			const size_t r0 = size_t(s) * groups;
			const size_t longest = r0 < rows ? len[order[r0]] : 0;
			const size_t base = out.ptr[slice];
			const size_t next = base + (longest + 4 * L - 1) / (4 * L);
			/* rows far longer than most would fill slices with nothing */
			if(next * 256 > 2 * m_s + 256 * (slice + 1) || next * 256 > UINT32_MAX) return PushRows();
			out.ptr[slice + 1] = uint32_t(next);
			for(size_t g = 0; g < groups && r0 + g < rows; ++g) {
				const uint32_t r = order[r0 + g];
				for(unsigned l = 0; l < L; ++l)
					out.rows[slice * 64 + g * L + l] = {uint16_t(r / m_D), uint16_t(r % m_D + 1)};
				out.at[first * m_D + r] = uint32_t(base * 256 + g * L * 4);
			}
		}
	}
	return out;
}

/* The slices of forward_sliced_kernel, or nothing. */
std::vector<uint32_t> FloatNetwork::pullSlices(const std::vector<uint32_t>& ptr)
{
	const size_t slices = (m_n + 7) / 8;
	std::vector<uint32_t> out(slices + 1, 0);
	m_sliceLines = 0;
	for(size_t s = 0; s < slices; ++s) {
		uint32_t longest = 0;
		for(size_t j = 8 * s; j < std::min(m_n, 8 * s + 8); ++j) longest = std::max(longest, ptr[j + 1] - ptr[j]);
		const uint32_t lines = longest / 32 + (longest % 32 != 0);
		/* targets far beyond their neighbours would fill slices with nothing */
		if((size_t(out[s]) + lines) * 256 > 2 * m_s + 256 * (s + 1) || lines > 65535) return {};
		out[s + 1] = out[s] + lines;
		m_sliceLines = std::max(m_sliceLines, lines);
	}
	return out;
}

void FloatNetwork::sliceWeights(hipStream_t st, float* wr, const float* w)
{
	HIP_CHECK(nemo_launch_float_slice_weights(st, wr, w, m_sliceUser.ptr, m_slicePtr.ptr, unsigned(m_slicePtr.n - 1),
			m_sliceLines, m_s));
}

void FloatNetwork::prepare(unsigned T, unsigned K)
{
	if(T == 0) throw Error(NEMO_INVALID_INPUT, "the float-weight mode needs at least one step");
	if(K == 0) throw Error(NEMO_INVALID_INPUT, "checkpoint interval must be positive");
	HIP_CHECK(hipSetDevice(m_device));
	const unsigned k = std::min(K, T);
	if(k > m_segK) {
		m_seg.allocate(3 * size_t(k) * m_n);
		m_segK = k;
	}
	if(T > m_bitsT) {
		m_bits.allocate(size_t(T) * m_pitch);
		m_bitsT = T;
	}
}

void FloatNetwork::forward(hipStream_t st, unsigned T, unsigned K, const float* w, const float* a,
		const float* b, const float* c, const float* d, const float* v0, const float* u0, const float* x,
		float* S, float* V, double* ckpt)
{
	prepare(T, K);
	ForwardWorkspace ws;
	ws.sliced = m_sliceUser.n != 0;
	ws.wr = m_wr.ptr;
	ws.v = m_v.ptr;
	ws.u = m_u.ptr;
	ws.bits = m_bits.ptr;
	forwardWith(ws, st, T, K, w, a, b, c, d, v0, u0, x, S, V, ckpt);
}

/* The forward on the device's static workspace: the kernels and arguments of
 * forward(), with the workspace carved from the file-scope array of
 * float_mode.hip instead of this object's allocations, so that nothing is
 * allocated (the array's address is looked up on the device's first call).
 * Calls on one device share the array, so they must not overlap. */
void FloatNetwork::forwardStatic(hipStream_t st, unsigned T, unsigned K, const float* w, const float* a,
		const float* b, const float* c, const float* d, const float* v0, const float* u0, const float* x,
		float* S, float* V, double* ckpt)
{
	if(T == 0) throw Error(NEMO_INVALID_INPUT, "the float-weight mode needs at least one step");
	if(K == 0) throw Error(NEMO_INVALID_INPUT, "checkpoint interval must be positive");
	HIP_CHECK(hipSetDevice(m_device));
	void* base = nullptr;
	size_t cap = 0;
	HIP_CHECK(nemo_float_scratch(&base, &cap));
	const bool sliced = m_sliceUser.n && forwardWorkspaceBytes(T, true) <= cap;
	const size_t need = forwardWorkspaceBytes(T, sliced);
	if(need > cap) {
		throw Error(NEMO_INVALID_INPUT, "the allocation-free forward of " + std::to_string(T) + " steps needs "
				+ std::to_string(need) + " bytes of workspace; its static workspace holds " + std::to_string(cap));
	}
	forwardWith(carveWorkspace(base, T, sliced), st, T, K, w, a, b, c, d, v0, u0, x, S, V, ckpt);
}

/* Bytes of the forward's workspace for T steps, each part 256-byte aligned:
 * weights in reverse order (4 B per synapse), v and u in double (16 B per
 * neuron) and the spike bitmaps of every step. */
size_t FloatNetwork::forwardWorkspaceBytes(unsigned T, bool sliced) const
{
	auto up = [](size_t x) { return (x + 255) / 256 * 256; };
	return up((sliced ? m_sliceUser.n : std::max<size_t>(1, m_s)) * sizeof(float)) + 2 * up(m_n * sizeof(double))
		+ up(size_t(T) * m_pitch * sizeof(uint32_t));
}

FloatNetwork::ForwardWorkspace FloatNetwork::carveWorkspace(void* base, unsigned T, bool sliced) const
{
	auto up = [](size_t x) { return (x + 255) / 256 * 256; };
	unsigned char* p = static_cast<unsigned char*>(base);
	ForwardWorkspace ws;
	ws.sliced = sliced;
	ws.wr = reinterpret_cast<float*>(p);
	p += up((sliced ? m_sliceUser.n : std::max<size_t>(1, m_s)) * sizeof(float));
	ws.v = reinterpret_cast<double*>(p);
	p += up(m_n * sizeof(double));
	ws.u = reinterpret_cast<double*>(p);
	p += up(m_n * sizeof(double));
	ws.bits = reinterpret_cast<uint32_t*>(p);
	(void) T;
	return ws;
}

/* The forward's kernels on a given workspace; launches only (nothing is
 * allocated, freed or waited for), so it may be captured in a graph. */
void FloatNetwork::forwardWith(const ForwardWorkspace& ws, hipStream_t st, unsigned T, unsigned K, const float* w,
		const float* a, const float* b, const float* c, const float* d, const float* v0, const float* u0,
		const float* x, float* S, float* V, double* ckpt)
{
	if(T == 0) throw Error(NEMO_INVALID_INPUT, "the float-weight mode needs at least one step");
	if(K == 0) throw Error(NEMO_INVALID_INPUT, "checkpoint interval must be positive");
	HIP_CHECK(hipSetDevice(m_device));
	nemo_float_begin_forward_args begin = {};
	begin.n = m_n;
	begin.synapses = m_s;
	begin.w = w;
	begin.wr_entries = ws.sliced ? 0 : m_s;
	begin.wr_user = m_rcmUser.ptr;
	begin.wr = ws.wr;
	begin.v0 = v0;
	begin.u0 = u0;
	begin.v = ws.v;
	begin.u = ws.u;
	HIP_CHECK(nemo_launch_float_begin_forward(st, &begin));
	if(ws.sliced) sliceWeights(st, ws.wr, w);
	nemo_float_step_args f = {};
	f.n = unsigned(m_n);
	f.rcm_ptr = m_rcmPtr.ptr;
	f.rcm_sd = m_rcmSd.ptr;
	f.wr = ws.wr;
	f.pa = a;
	f.pb = b;
	f.pc = c;
	f.pd = d;
	f.x = x;
	f.S = S;
	f.V = V;
	f.v = ws.v;
	f.u = ws.u;
	f.store = 1;
	f.ckpt = ckpt;
	f.K = K;
	f.bits = ws.bits;
	f.pitch = m_pitch;
	f.dmax = m_D;
	f.stage = m_stage;
	f.slice_ptr = ws.sliced ? m_slicePtr.ptr : nullptr;
	f.slice_sd = m_sliceSd.ptr;
	for(unsigned t = 0; t < T; ++t) {
		f.t = t;
		HIP_CHECK(nemo_launch_float_forward_step(st, &f));
	}
}

/* Segments of K steps in reverse: replay the segment's forward steps from its
 * checkpoint (one launch), recording entry state and input, then run its
 * adjoint steps backwards. */
void FloatNetwork::backward(hipStream_t st, unsigned T, unsigned K, const float* w, const float* a,
		const float* b, const float* c, const float* d, const float* x, const float* S, const double* ckpt,
		const float* gS, const float* gV, float* gw, float* ga, float* gb, float* gd, float* gx,
		float* gv0, float* gu0)
{
	prepare(T, K);
	nemo_float_begin_backward_args begin = {};
	begin.n = m_n;
	begin.synapses = m_s;
	begin.li = m_LI.n;
	begin.w = w;
	const bool sliced = m_sliceUser.n && m_n <= NEMO_FLOAT_REPLAY_MAX && m_D < 58;
	begin.wr_entries = sliced ? 0 : m_s;
	begin.wr_user = m_rcmUser.ptr;
	begin.wr = m_wr.ptr;
	begin.row_user = m_rowUser.ptr;
	begin.entries = m_push ? m_rowUser.n : 0;
	begin.row_w = m_rowW.ptr;
	begin.row_gw = m_rowGw.ptr;
	begin.LI = m_LI.ptr;
	begin.LV = m_LV.ptr;
	begin.LU = m_LU.ptr;
	begin.gw = gw;
	begin.ga = ga;
	begin.gb = gb;
	begin.gd = gd;
	HIP_CHECK(nemo_launch_float_begin_backward(st, &begin));
	if(sliced) sliceWeights(st, m_wr.ptr, w);
	const unsigned Kseg = std::min(K, T);
	const size_t segPlane = size_t(Kseg) * m_n;

	/* the replay reads the recorded spikes as firing histories */
	const unsigned rows = nemo_float_history_rows(T);
	if(size_t(rows) * m_n > m_hist.n) m_hist.allocate(size_t(rows) * m_n);
	HIP_CHECK(nemo_launch_pack_history(st, m_hist.ptr, rows, S, unsigned(m_n), T));
	nemo_float_replay_args f = {};
	f.n = unsigned(m_n);
	f.dmax = m_D;
	f.rcm_ptr = m_rcmPtr.ptr;
	f.rcm_sd = m_rcmSd.ptr;
	f.wr = m_wr.ptr;
	f.pa = a;
	f.pb = b;
	f.pc = c;
	f.pd = d;
	f.x = x;
	f.hist = m_hist.ptr;
	f.hist_rows = rows;
	f.seg_v = m_seg.ptr;
	f.seg_u = m_seg.ptr + segPlane;
	f.seg_I = m_seg.ptr + 2 * segPlane;
	f.slice_ptr = sliced ? m_slicePtr.ptr : nullptr;
	f.slice_sd = m_sliceSd.ptr;

	nemo_float_push_args p = {};
	nemo_float_back_args g = {};
	if(m_push) {
		p.n = unsigned(m_n);
		p.T = T;
		p.dmax = m_D;
		p.tile = m_tile;
		p.pitch = m_pushPitch;
		p.lanes = m_pushLanes;
		p.slices = m_slices;
		p.slice_ptr = m_rowSlices.ptr;
		p.rows = m_rows.ptr;
		p.row_target = m_rowTarget.ptr;
		p.row_w = m_rowW.ptr;
		p.row_gw = m_rowGw.ptr;
		p.pa = a;
		p.pb = b;
		p.S = S;
		p.gS = gS;
		p.gV = gV;
		p.seg_v = f.seg_v;
		p.seg_u = f.seg_u;
		p.seg_I = f.seg_I;
		p.LV = m_LV.ptr;
		p.LU = m_LU.ptr;
		p.LI = m_LI.ptr;
		p.ring = m_LI.ptr + 2 * size_t(m_pushPitch);
		p.ga = ga;
		p.gb = gb;
		p.gd = gd;
		p.gx = gx;
	} else {
		g.n = unsigned(m_n);
		g.T = T;
		g.ring = m_D + 1;
		g.fcm_ptr = m_fcmPtr.ptr;
		g.fcm_td = m_fcmTd.ptr;
		g.wf = w;
		g.pa = a;
		g.pb = b;
		g.S = S;
		g.gS = gS;
		g.gV = gV;
		g.seg_v = f.seg_v;
		g.seg_u = f.seg_u;
		g.seg_I = f.seg_I;
		g.LV = m_LV.ptr;
		g.LU = m_LU.ptr;
		g.LI = m_LI.ptr;
		g.gw = gw;
		g.ga = ga;
		g.gb = gb;
		g.gd = gd;
		g.gx = gx;
	}

	const unsigned segments = (T + K - 1) / K;
	for(unsigned s = segments; s-- > 0;) {
		const unsigned t0 = s * K;
		const unsigned t1 = std::min(T, t0 + K);
		f.t0 = t0;
		f.t1 = t1;
		f.v0 = ckpt + size_t(s) * 2 * m_n;
		f.u0 = ckpt + size_t(s) * 2 * m_n + m_n;
		HIP_CHECK(nemo_launch_float_replay(st, &f));
		p.t0 = g.t0 = t0;
		for(unsigned t = t1; t-- > t0;) {
			p.t = g.t = t;
			if(m_push) HIP_CHECK(nemo_launch_float_push_step(st, &p));
			else HIP_CHECK(nemo_launch_float_backward_step(st, &g));
		}
	}
	nemo_float_end_backward_args done = {};
	done.n = m_n;
	done.synapses = m_s;
	done.entries = m_push ? m_rowUser.n : 0;
	done.row_user = m_rowUser.ptr;
	done.row_gw = m_rowGw.ptr;
	done.gw = gw;
	done.LV = m_LV.ptr;
	done.LU = m_LU.ptr;
	done.gv0 = gv0;
	done.gu0 = gu0;
	HIP_CHECK(nemo_launch_float_end_backward(st, &done));
}

} // namespace nemo_hip
