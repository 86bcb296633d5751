"""Kernels and dispatch branches chosen by size, each against the oracle at
the sizes where they change: through the C ABI, bit for bit."""
import math

import numpy as np
import pytest

import nemo_amd
from nemo_amd import generators as gen
import oracle_api as oa

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu(require_gpu):
    pass


def same_f32(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


# ------------------------------------------------- Kuramoto lane groups
def oscillators(api, n, degrees, dmax, seed):
    """n oscillators; oscillator i has degrees[i % len(degrees)] incoming
    synapses from random sources, added source by source."""
    rng = np.random.default_rng(seed)
    deg = np.resize(np.asarray(degrees), n)
    tgt = np.repeat(np.arange(n, dtype=np.uint32), deg)
    src = rng.integers(0, n, tgt.size, dtype=np.uint32)
    delay = rng.integers(1, dmax + 1, tgt.size, dtype=np.uint32)
    w = (rng.random(tgt.size, dtype=np.float32) * 2 - 1).astype(np.float32)
    order = np.argsort(src, kind="stable")
    net = api.Network()
    t = net.add_neuron_type("Kuramoto")
    net.add_neuron(t, np.arange(n, dtype=np.uint32), rng.random(n, dtype=np.float32), np.float32(30.0),
                   (rng.random(n) * 2 * math.pi).astype(np.float32))
    net.add_synapse(src[order], tgt[order], delay[order], w[order], np.zeros(tgt.size, np.uint8))
    return api.Simulation(net, api.Configuration())


@pytest.mark.parametrize("n,degrees,dmax", [
    (1, (1,), 1),
    (67, (0, 1, 2, 63, 64, 65, 255, 256, 257, 300), 20),   # a wave per oscillator, around its kept synapses
    (67, (5, 64, 270), 32),                                # ... in update passes
    (2048, (0, 3, 17), 20),                                # the largest launch of waves
    (2049, (0, 1, 15, 16, 17, 63, 64, 65, 80), 20),        # rows of 16, around their kept synapses
    (6000, (2, 16), 33),                                   # ... in update passes of both widths
    (32767, (2, 3), 20),                                   # the largest launch of rows at a small in-degree
    (32768, (0, 1, 3, 4, 5, 16, 17), 20),                  # quads, around their kept synapses
    (40000, (2, 3), 32),                                   # ... in update passes
])
def test_kuramoto_lane_groups_match_oracle(n, degrees, dmax):
    """Phases equal the oracle's after every one of 12 steps: the sums run in
    the reference's order whatever the lanes per oscillator."""
    ref, hip = (oscillators(api, n, degrees, dmax, seed=n + dmax) for api in (oa, nemo_amd))
    for t in range(12):
        assert ref.step() == hip.step() == []
        assert same_f32(ref.neuron_states(0), hip.neuron_states(0)), t


# --------------------------------------------------- direct delivery
def stdp(conf):
    pre, post = gen.stdp_exp_function(0.1, -0.12, 20.0, 20)
    conf.set_stdp_function(pre, post, 0.0, 10.0, 0.0, -10.0)
    return conf


def pair(spec, with_stdp):
    sims = []
    for api in (oa, nemo_amd):
        net = api.Network()
        spec.load(net)
        conf = api.Configuration()
        sims.append(api.Simulation(net, stdp(conf) if with_stdp else conf))
    return sims


@pytest.mark.parametrize("binned", [False, True])
@pytest.mark.parametrize("n,m,dmax", [
    (1, 3, 1),        # a ring of two slots, self synapses
    (255, 40, 1),
    (257, 60, 31),    # 32 slots, every delay of them used
    (700, 30, 32),    # 64 slots
    (513, 300, 43),   # rows of one neuron longer than a block's threads
    (600, 400, 1),    # more pieces of rows than a block lists at a time
    (1500, 40, 6),    # more fired rows than a delivery block lists at a time
])
def test_small_network_delivery_matches_oracle(n, m, dmax, binned):
    """Rasters, events, potentials and learned weights against the oracle over
    runs, single steps, a step in which every neuron fires (each block delivers
    thousands of events), applyStdp with events under way, and a shape set and
    left in between."""
    spec = gen.random_izhikevich(n, m, dmax=dmax, seed=n + dmax, stdp=True)
    ref, hip = pair(spec, True)
    if binned:
        hip.launch_shape = hip.launch_shape

    def advance(steps):
        before = ref.delivered_events()
        want = [ref.step() for _ in range(steps)]
        counts, fired, events = hip.run(steps)
        assert counts.tolist() == [len(f) for f in want]
        assert fired.tolist() == [i for f in want for i in f]
        assert events == ref.delivered_events() - before

    everyone = list(range(n))
    advance(70)
    assert ref.step(everyone) == hip.step(everyone)
    advance(3)
    for sim in (ref, hip):
        sim.apply_stdp(1.0)
    advance(dmax + 5)
    if not binned:
        hip.launch_shape = hip.launch_shape  # the binned delivery from here on, with events under way
    for _ in range(3):
        assert ref.step(everyone) == hip.step(everyone)
    advance(66)
    ref.apply_stdp(-0.5)
    hip.apply_stdp(-0.5)
    assert np.array_equal(ref.fixed_weights(spec.synapse_count), hip.fixed_weights())
    for var in (0, 1):
        assert same_f32(ref.neuron_states(var), hip.neuron_states(var))


def test_maximum_delay_and_propagate_with_steps_in_between():
    """Delays up to 64 (a ring of 128 slots), and Brian's propagate before,
    between and after steps: its events stay under way for the steps, and the
    input of a step it passed over is not left for a later one."""
    spec = gen.random_izhikevich(600, 80, dmax=64, seed=9)
    ref, hip = pair(spec, False)
    rng = np.random.default_rng(2)
    for block in range(4):
        for _ in range(5 if block else 150):
            f = sorted(rng.choice(600, 40, replace=False).tolist())
            (er, ir), (eh, ih) = ref.propagate(f), hip.propagate(f)
            assert same_f32(er, eh) and same_f32(ir, ih)
        for _ in range(7):
            assert ref.step() == hip.step()
        want = [ref.step() for _ in range(130)]
        counts, fired, _ = hip.run(130)
        assert counts.tolist() == [len(f) for f in want]
        assert fired.tolist() == [i for f in want for i in f]


# ------------------------------------------------------- firing readout
def sources_and_neurons(n, first, seed, order):
    """n Poisson sources firing with rate 1 per ms (every step) or, past
    4090, now and then, and 300 Izhikevich neurons, in either type order."""
    rate = np.where(np.arange(n) < 4090, np.float32(1.0), np.float32(0.01)).astype(np.float32)
    po = gen.NetworkSpec(blocks=[gen.NeuronBlock("PoissonSource", np.arange(first, first + n, dtype=np.uint32), [rate])])
    iz = gen.random_izhikevich(300, 40, dmax=8, seed=seed, first_index=first + n)
    return gen.merge(*((po, iz) if order else (iz, po)))


@pytest.mark.parametrize("sizes", [(4000,), (4095,), (4200,), (9000,), (2500, 4090, 3000)])
def test_readout_of_steps_around_its_room(sizes):
    """Steps that fire fewer and more neurons than the readout has room for,
    over several graphs, against the oracle: a single network and a batch
    whose networks list their types in different orders."""
    specs = [sources_and_neurons(n, 7, 30 + k, k % 2) for k, n in enumerate(sizes)]
    refs, nets = [], []
    for spec in specs:
        for api, out in ((oa, refs), (nemo_amd, nets)):
            net = api.Network()
            spec.load(net)
            out.append(oa.Simulation(net, oa.Configuration()) if api is oa else net)
    steps = 131
    conf = nemo_amd.Configuration()
    if len(nets) == 1:
        counts, fired, _ = nemo_amd.Simulation(nets[0], conf).run(steps)
        got = [(counts, fired)]
    else:
        batch = nemo_amd.Batch(nets, conf)
        counts, fired, _ = batch.run(steps)
        got = batch.split(counts, fired)
    for ref, (c, f) in zip(refs, got):
        want = [ref.step() for _ in range(steps)]
        assert c.tolist() == [len(x) for x in want]
        assert f.tolist() == [i for x in want for i in x]


# ------------------------------------------------- Hodgkin-Huxley substeps
def hh_cells(api, v, gates, dirs):
    net = api.Network()
    t = net.add_neuron_type("HH")
    n = len(v)
    net.add_neuron(t, np.arange(n, dtype=np.uint32), np.asarray(v, np.float32), *[np.asarray(g, np.float32) for g in gates],
                   np.asarray(dirs, np.float32))
    return api.Simulation(net, api.Configuration())


# y = v + 65: the quotients of alphan and alpham are by 0 at y = 10 and 25;
# the substeps without special cases are for |y| <= 256
HH_POTENTIALS = [-65.0, -55.0, -40.0, -45.0, -45.000004, -44.999996, 50.0, 191.0, 191.00002, -321.0, -321.00003, 2000.0,
                 -3000.0, 1e6, -1e6, 1e30, -1e38, 3e38, np.inf, -np.inf, np.nan, -54.999996, -55.000004, -39.999996]


@pytest.mark.parametrize("n", [1, 3, 4, 5, 24, 257])
def test_hh_substeps_match_oracle(n):
    """State and firing equal the oracle's, step by step, with neighbours in a
    wave that take the general path and ones that do not, and with currents
    that turn the potential down from both sides of -45."""
    rng = np.random.default_rng(n)
    v = np.resize(np.asarray(HH_POTENTIALS, np.float32), n)
    if n == 257:
        v[24:] = (rng.random(n - 24, dtype=np.float32) * 120 - 80).astype(np.float32)
    gates = [rng.random(n, dtype=np.float32) for _ in range(3)]
    dirs = rng.choice(np.asarray([0.0, -1e-10, 1e-3, -0.5], np.float32), n)
    sims = [hh_cells(api, v, gates, dirs) for api in (oa, nemo_amd)]
    for t in range(30):
        istim = [(i, float(x)) for i, x in enumerate(rng.normal(0, 40, n).astype(np.float32))]
        fr, fh = (s.step(istim=istim) for s in sims)
        assert list(fr) == list(fh), t
        for k in range(5):
            a, b = (np.asarray(s.neuron_states(k), np.float32) for s in sims)
            same = (a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))
            assert same.all(), (t, k, np.flatnonzero(~same)[:5])


# ------------------------------------------------- float mode's staged forms
def float_results(spec, n, T, monkeypatch):
    """Spikes, potentials and gradients with the staged kernels and with the
    general ones, the second pass of each (which starts from the first one's
    leavings)."""
    torch = pytest.importorskip("torch")
    from nemo_amd.differentiable import FloatNetwork
    rng = np.random.default_rng(n)
    a, b, c, d, _, u, v = [np.asarray(x, np.float32) * np.ones(n, np.float32) for x in spec.blocks[0].args]
    x = (8.0 * rng.standard_normal((T, n))).astype(np.float32)
    gS, gV = (torch.tensor(rng.standard_normal((T, n)).astype(np.float32), device="cuda") for _ in range(2))
    out = []
    for stage in ("1", "0"):
        monkeypatch.setenv("NEMO_HIP_FLOAT_STAGE", stage)
        net = nemo_amd.Network()
        spec.load(net)
        fnet = FloatNetwork(net, 0)
        p = {k: torch.tensor(t, device="cuda") for k, t in dict(w=spec.weight, a=a, b=b, d=d, x=x, v0=v, u0=u).items()}
        for t in p.values():
            t.requires_grad_(True)
        for _ in range(2):
            for t in p.values():
                t.grad = None
            S, V = fnet(p["w"], p["a"], p["b"], p["d"], p["x"], c=torch.tensor(c, device="cuda"), v0=p["v0"],
                        u0=p["u0"], checkpoint_every=17)
            torch.autograd.backward([S, V], [gS, gV])
        out.append((S.detach().cpu().numpy(), V.detach().cpu().numpy(),
                    {k: t.grad.double().cpu().numpy() for k, t in p.items()}))
    return out


def check_float_results(staged, general, T):
    """The forward sums in the same order, so spikes and potentials are the
    same bits.  The backward sums the same doubles in another order, so the
    gradients, which are accumulated over T steps in float, differ by at most T
    roundings of 2^-24."""
    assert np.array_equal(staged[0], general[0]) and same_f32(staged[1], general[1])
    for k in staged[2]:
        a, b = staged[2][k], general[2][k]
        assert np.linalg.norm(a - b) <= T * 2.0 ** -24 * np.linalg.norm(b), k


@pytest.mark.parametrize("n,m,dmax,T", [
    (2, 1, 1, 5),          # one delay: every row starts its slot
    (255, 7, 2, 9),        # an odd size, one neuron per block, slices of one row
    (1025, 40, 3, 30),     # a last block of neurons that is not full
    (400, 300, 5, 40),     # more synapses than a wave has in flight
    (300, 40, 57, 60),     # the longest delay of the windowed replay
    (600, 130, 64, 90),    # beyond it; more slices than waves
    (12000, 25, 19, 40),   # a lane per row
    (20398, 12, 5, 12),    # the largest network whose adjoints fit in LDS
    (20480, 12, 5, 12),    # beyond that, the largest whose windows do
    (20481, 12, 5, 12),    # beyond both
])
def test_float_staged_and_general_agree(n, m, dmax, T, monkeypatch):
    """The kernels that read their synapses in slices, with spikes and adjoints
    in LDS, and the general ones; fired sources, steps before the first and
    after the last included."""
    spec = gen.random_izhikevich(n, m, dmax=dmax, seed=n)
    spec.weight = (spec.weight * np.float32(30.0 / m)).astype(np.float32)
    staged, general = float_results(spec, n, T, monkeypatch)
    assert n == 2 or staged[0].sum() > 0  # two neurons are silent
    check_float_results(staged, general, T)


@pytest.mark.parametrize("n,count,sources,targets", [
    (500, 25000, None, 7),     # one target has all synapses: its slice would be mostly empty
    (500, 20000, 3, None),     # one source: its row would be
    (700, 9000, 2.0, 1.5),     # uneven, to powers of a uniform draw
    (40, 30000, None, None),   # several synapses from each neuron to each
])
def test_float_uneven_networks_agree(n, count, sources, targets, monkeypatch):
    """The same where degrees are uneven, on both sides of the rule that gives
    such networks to the general kernels."""
    rng = np.random.default_rng(count)

    def draw(kind):
        if isinstance(kind, int):
            return np.full(count, kind)
        return (n * rng.random(count) ** (kind or 1.0)).astype(np.int64)

    src = np.sort(draw(sources))
    spec = gen.random_izhikevich(n, 0, dmax=1, seed=3)
    spec.source, spec.target = src.astype(np.uint32), draw(targets).astype(np.uint32)
    spec.delay = rng.integers(1, 9, count).astype(np.uint32)
    spec.weight = (rng.random(count) * 0.05).astype(np.float32)
    spec.plastic = np.zeros(count, np.uint8)
    staged, general = float_results(spec, n, 60, monkeypatch)
    assert staged[0].sum() > 0
    check_float_results(staged, general, 60)


# ------------------------------------------------- applyStdp over tiles
@pytest.mark.parametrize("n,m", [(14000, 1200), (9001, 1777)])
def test_apply_stdp_over_tiles(n, m):
    """From 12 x 2^20 plastic synapses on, applyStdp moves the accumulators to
    tiles of the forward matrix (more than 8 of them, the last one partial, an
    odd number of synapses in the second case).  The weights equal the ones
    that the reward's definition gives for the accumulators read before, in
    whole numbers, and the accumulators are zero afterwards; twice, and with a
    reward of zero, which only clears them."""
    spec = gen.random_izhikevich(n, m, dmax=12, seed=n, stdp=True)
    assert spec.plastic.sum() > 12 << 20
    net = nemo_amd.Network()
    spec.load(net)
    sim = nemo_amd.Simulation(net, stdp(nemo_amd.Configuration()))
    for reward in (1.0, -0.5, 0.0):
        sim.run(60)
        acc, w = np.asarray(sim.stdp_accumulators(), np.int64), np.asarray(sim.fixed_weights(), np.int64)
        assert np.count_nonzero(acc) > 1000
        sim.apply_stdp(reward)
        dw = (int(reward * (1 << 20)) * acc) >> 20
        top, bottom = 10 << 20, -(10 << 20)
        want = np.where(w > 0, np.clip(w + dw, 0, top), np.where(w < 0, np.clip(w + dw, bottom, 0), 0))
        want = np.where(spec.plastic != 0, want, w)
        assert np.array_equal(np.asarray(sim.fixed_weights(), np.int64), want), reward
        assert not np.any(sim.stdp_accumulators())


# ------------------------------------------------- STDP rows by waves
@pytest.mark.parametrize("n,m", [
    (300, 130),   # about 104 plastic synapses per target: looked up one by one
    (300, 150),   # about 120: a wave per target, most of a second chunk idle
    (257, 640),   # exactly as many loads in flight as a wave takes, and a last word of one target
    (700, 1300),  # more than one round of them
])
def test_stdp_rows_match_oracle(n, m):
    """Accumulators and weights equal the oracle's after batches beside the
    steps, a flush and an applyStdp."""
    spec = gen.random_izhikevich(n, m, dmax=9, seed=n + m, stdp=True)
    ref, hip = pair(spec, True)
    for steps in (150, 7):
        for _ in range(steps):
            ref.step()
        hip.run(steps)
        assert np.array_equal(ref.stdp_accumulators(n * m), hip.stdp_accumulators())
        assert np.any(hip.stdp_accumulators())
        for sim in (ref, hip):
            sim.apply_stdp(0.5)
        assert np.array_equal(ref.fixed_weights(n * m), hip.fixed_weights())
