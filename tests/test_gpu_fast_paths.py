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
