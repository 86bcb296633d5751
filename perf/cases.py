"""Performance cases: the work a user of nemo_amd has it do, through its
public entry points.

Every case is a dict of plain values with a "kind":

  step       a closed loop that steps a small network with stimulus every step
             and reads the firing and a few membrane potentials back
  run        Simulation.run of an Izhikevich network, firing read back, with or
             without STDP (applied every `period` steps) and the learned weights
  batch      Batch.run of independent networks of mixed sizes
  mixed      Simulation.run of the four-model torus network (LIF, QIF, HH,
             Poisson)
  kuramoto   coupled oscillators advanced and their phases read
  propagate  Brian's propagate: given firing in, synaptic input out
  forward    the float-weight mode's forward pass (inference)
  train      its forward and adjoint (a training step's gradients)

listed() are fixed cases, draw() more of the same ranges, prepare() what a
program holds before the call (a built simulation that has run its first
steps, or the weights and inputs on the device), run() one pass, work() the
bytes and operations of a pass that no implementation avoids, and exact() the
results in 64 bits from plain torch or numpy where they are real numbers (the
spiking simulations compute in fixed point: their firing, events and weights
are whole numbers).
"""
import math

import numpy as np
import torch

import nemo_amd
from nemo_amd import generators as gen
from nemo_amd.differentiable import FloatNetwork

# firing of the 80/20 Izhikevich network in its settled state (per neuron and
# step) and of the torus network, for the work estimates
IZH_RATE = 0.0065
TORUS_RATE = 0.008


def listed():
    return [
        # latency: a controller in the loop with the smallest network in use
        {"name": "closed-loop-1k", "kind": "step", "neurons": 1000, "synapses": 100, "dmax": 20, "steps": 10},
        # a small learning experiment, its weights read after every epoch
        {"name": "learn-1k", "kind": "run", "neurons": 1000, "synapses": 100, "dmax": 20, "steps": 100,
         "stdp": True, "period": 50, "weights": True},
        # a medium network without plasticity
        {"name": "run-10k", "kind": "run", "neurons": 10000, "synapses": 200, "dmax": 10, "steps": 200,
         "stdp": False, "period": 0, "weights": False},
        # a ragged learning network: no size a multiple of a tile or a wave
        {"name": "learn-30k", "kind": "run", "neurons": 30011, "synapses": 333, "dmax": 17, "steps": 150,
         "stdp": True, "period": 150, "weights": False},
        # the benchmark network: 1e8 synapses with STDP
        {"name": "learn-100k", "kind": "run", "neurons": 100000, "synapses": 1000, "dmax": 20, "steps": 250,
         "stdp": True, "period": 250, "weights": False},
        # a parameter sweep: many independent networks in the same launches
        {"name": "batch-32", "kind": "batch", "networks": 32, "nmin": 1000, "nmax": 10000, "smin": 100, "smax": 1000,
         "steps": 50},
        # neuron models mixed in one network
        {"name": "mixed-10k", "kind": "mixed", "lif": 8000, "qif": 1600, "hh": 400, "poisson": 200, "synapses": 500,
         "steps": 20},
        # oscillators whose models read their sources' phases
        {"name": "kuramoto-1k", "kind": "kuramoto", "neurons": 1000, "indegree": 100, "dmax": 10, "steps": 20},
        # synaptic propagation for a simulator that updates the neurons itself
        {"name": "propagate-20k", "kind": "propagate", "neurons": 20000, "synapses": 500, "dmax": 20, "fired": 150,
         "steps": 10},
        # inference with trained float weights
        {"name": "forward-10k", "kind": "forward", "neurons": 10000, "synapses": 200, "dmax": 10, "steps": 100},
        # training steps, large and small
        {"name": "train-10k", "kind": "train", "neurons": 10000, "synapses": 200, "dmax": 10, "steps": 100,
         "checkpoint": 50},
        {"name": "train-1k", "kind": "train", "neurons": 1000, "synapses": 100, "dmax": 10, "steps": 50,
         "checkpoint": 25},
    ]


def _log(rng, lo, hi):
    """A whole number, log-uniform in lo..hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "run", "run", "run", "batch", "mixed", "kuramoto", "propagate", "forward", "train"])
    if kind == "step":
        return {"kind": kind, "neurons": _log(rng, 300, 10000), "synapses": _log(rng, 20, 200),
                "dmax": rng.randint(1, 30), "steps": rng.randint(5, 20)}
    if kind == "run":
        n = _log(rng, 500, 100000)
        # at most 3e7 synapses, so that a drawn case stays well below the largest listed one
        m = _log(rng, 30, max(31, min(1000, 30000000 // n)))
        steps = rng.randint(20, 250)
        stdp = rng.random() < 0.5
        return {"kind": kind, "neurons": n, "synapses": m, "dmax": rng.randint(2, 30), "steps": steps, "stdp": stdp,
                "period": steps if stdp else 0, "weights": stdp and n * m < 500000}
    if kind == "batch":
        return {"kind": kind, "networks": rng.randint(4, 32), "nmin": rng.randint(300, 1000),
                "nmax": rng.randint(2000, 10000), "smin": rng.randint(50, 100), "smax": rng.randint(200, 1000),
                "steps": rng.randint(20, 60)}
    if kind == "mixed":
        n = _log(rng, 2000, 12000)
        hh = rng.randint(50, 500)
        qif = rng.randint(200, 2000)
        return {"kind": kind, "lif": n, "qif": qif, "hh": hh, "poisson": rng.randint(50, 300),
                "synapses": rng.randint(50, 500), "steps": rng.randint(10, 30)}
    if kind == "kuramoto":
        return {"kind": kind, "neurons": _log(rng, 100, 4000), "indegree": _log(rng, 10, 300),
                "dmax": rng.randint(1, 40), "steps": rng.randint(5, 30)}
    if kind == "propagate":
        n = _log(rng, 1000, 50000)
        return {"kind": kind, "neurons": n, "synapses": rng.randint(50, 500), "dmax": rng.randint(1, 30),
                "fired": rng.randint(1, max(2, n // 100)), "steps": rng.randint(5, 20)}
    case = {"kind": kind, "neurons": _log(rng, 300, 12000), "synapses": _log(rng, 20, 250), "dmax": rng.randint(1, 20),
            "steps": rng.randint(20, 120)}
    if kind == "train":
        case["checkpoint"] = rng.randint(10, 60)
    return case


# ------------------------------------------------------------------ inputs
def _stdp(conf):
    pre, post = gen.stdp_exp_function(0.1, -0.12, 20.0, 20)
    conf.set_stdp_function(pre, post, 0.0, 10.0, 0.0, -10.0)


def _load(spec):
    net = nemo_amd.Network()
    spec.load(net)
    return net


def _izhikevich(case, seed, stdp=False):
    return gen.random_izhikevich(case["neurons"], case["synapses"], dmax=case["dmax"], seed=seed, stdp=stdp)


def _oscillators(case, seed):
    """omega, theta, and the synapses (source, target, delay, weight), added
    source by source."""
    n, k = case["neurons"], case["indegree"]
    rng = np.random.default_rng(seed)
    omega = rng.random(n, dtype=np.float32)
    theta = (rng.random(n) * 2 * math.pi).astype(np.float32)
    tgt = np.repeat(np.arange(n, dtype=np.uint32), k)
    src = rng.integers(0, n, tgt.size, dtype=np.uint32)
    delay = rng.integers(1, case["dmax"] + 1, tgt.size, dtype=np.uint32)
    w = (rng.random(tgt.size, dtype=np.float32) * 2 - 1).astype(np.float32)
    order = np.argsort(src, kind="stable")
    return omega, theta, src[order], tgt[order], delay[order], w[order]


def _fired_lists(case, seed):
    rng = np.random.default_rng(seed + 1)
    return [np.sort(rng.choice(case["neurons"], case["fired"], replace=False)).astype(np.uint32)
            for _ in range(case["steps"])]


def _float_inputs(case, seed):
    """The network (plain arrays) and the float mode's inputs as numpy float32."""
    spec = _izhikevich(case, seed)
    a, b, c, d, sigma, u, v = spec.blocks[0].args
    rng = np.random.default_rng(seed + 2)
    x = sigma * rng.standard_normal((case["steps"], case["neurons"]), dtype=np.float32)
    gS = rng.standard_normal((case["steps"], case["neurons"]), dtype=np.float32)
    gV = (0.01 * rng.standard_normal((case["steps"], case["neurons"]), dtype=np.float32)).astype(np.float32)
    return spec, dict(w=spec.weight, a=a, b=b, c=c, d=d, v0=v, u0=u, x=x.astype(np.float32), gS=gS, gV=gV)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "run"):
        stdp = case.get("stdp", False)
        conf = nemo_amd.Configuration()
        if stdp:
            _stdp(conf)
        sim = nemo_amd.Simulation(_load(_izhikevich(case, seed, stdp)), conf)
        sim.run(100)  # past the quiet first steps
        if kind == "run":
            sim.prepare(case["steps"], stdp_period=case["period"])
            return {"case": case, "sim": sim, "fired_room": _fired_room(case, case["neurons"])}
        rng = np.random.default_rng(seed + 3)
        n = case["neurons"]
        inputs = []
        for _ in range(case["steps"]):
            idx = rng.choice(n, 20, replace=False)
            inputs.append(([int(i) for i in rng.choice(n, 5, replace=False)],
                           [(int(i), float(v)) for i, v in zip(idx, rng.random(20) * 10)]))
        return {"case": case, "sim": sim, "inputs": inputs, "probes": [int(i) for i in rng.choice(n, 8, replace=False)],
                "fired_room": _fired_room(case, n)}
    if kind == "batch":
        conf = nemo_amd.Configuration()
        _stdp(conf)
        specs = gen.batch_izhikevich(count=case["networks"], nmin=case["nmin"], nmax=case["nmax"], smin=case["smin"],
                                     smax=case["smax"], seed=seed, seed_base=seed + 1000)
        sim = nemo_amd.Batch([_load(spec) for spec, _ in specs], conf)
        sim.run(100)
        sim.prepare(case["steps"])
        return {"case": case, "sim": sim, "fired_room": _fired_room(case, case["networks"] * case["nmax"])}
    if kind == "mixed":
        total = case["lif"] + case["qif"] + case["hh"]
        spec = gen.torus_mixed(n_lif=case["lif"], n_qif=case["qif"], n_hh=case["hh"], n_poisson=case["poisson"],
                               m=case["synapses"], seed=seed, grid=max(2, int(math.sqrt(total / 25.0))))
        sim = nemo_amd.Simulation(_load(spec), nemo_amd.Configuration())
        sim.run(100)
        sim.prepare(case["steps"])
        return {"case": case, "sim": sim, "fired_room": _fired_room(case, total + case["poisson"])}
    if kind == "kuramoto":
        omega, theta, src, tgt, delay, w = _oscillators(case, seed)
        net = nemo_amd.Network()
        t = net.add_neuron_type("Kuramoto")
        cmean = np.full(case["neurons"], float(case["indegree"]), np.float32)
        net.add_neuron(t, np.arange(case["neurons"], dtype=np.uint32), omega, cmean, theta)
        net.add_synapse(src, tgt, delay, w, 0)
        sim = nemo_amd.Simulation(net, nemo_amd.Configuration())
        sim.prepare(case["steps"])
        return {"case": case, "sim": sim}
    if kind == "propagate":
        sim = nemo_amd.Simulation(_load(_izhikevich(case, seed)), nemo_amd.Configuration())
        return {"case": case, "sim": sim, "fired": _fired_lists(case, seed)}
    spec, inp = _float_inputs(case, seed)
    fnet = FloatNetwork(_load(spec), 0)
    dev = {k: torch.tensor(v, device="cuda:0") for k, v in inp.items()}
    if kind == "train":
        for k in ("w", "a", "b", "d", "x"):
            dev[k].requires_grad_(True)
    return {"case": case, "net": fnet, "in": dev}


def _fired_room(case, neurons):
    """The program's own buffer for a pass's fired neurons, several times what
    the network fires; the end of it is filled with ~0."""
    return np.empty(case["steps"] * neurons // 40 + 4096, np.uint32)


def _keep(state, fired):
    room = state["fired_room"]
    if len(fired) > room.size:
        room = state["fired_room"] = np.empty(2 * len(fired), np.uint32)
    room[:len(fired)] = fired
    room[len(fired):] = 0xffffffff
    return room


# -------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        sim = state["sim"]
        fired = [sim.step(fstim=f, istim=i) for f, i in state["inputs"]]
        return {"counts": np.array([len(f) for f in fired], np.int64),
                "fired": _keep(state, [i for f in fired for i in f]),
                "v": np.array(sim.get_neuron_state(state["probes"], 1), np.float32)}
    if kind == "run":
        sim = state["sim"]
        counts, fired, events = sim.run(case["steps"], stdp_period=case["period"], reward=1.0)
        out = {"counts": counts.astype(np.int64), "fired": _keep(state, fired), "events": events}
        if case["weights"]:
            out["weights"] = sim.fixed_weights()
        return out
    if kind in ("batch", "mixed"):
        counts, fired, events = state["sim"].run(case["steps"])
        return {"counts": counts.astype(np.int64), "fired": _keep(state, fired), "events": events}
    if kind == "kuramoto":
        state["sim"].run(case["steps"])
        return state["sim"].neuron_states(0)
    if kind == "propagate":
        got = [state["sim"].propagate(f) for f in state["fired"]]
        return {"E": np.stack([e for e, _ in got]), "I": np.stack([i for _, i in got])}
    p = state["in"]
    if kind == "forward":
        with torch.no_grad():
            S, V = state["net"](p["w"], p["a"], p["b"], p["d"], p["x"], c=p["c"], v0=p["v0"], u0=p["u0"])
        return {"S": S, "V": V}
    S, V = state["net"](p["w"], p["a"], p["b"], p["d"], p["x"], c=p["c"], v0=p["v0"], u0=p["u0"],
                        checkpoint_every=case["checkpoint"])
    g = torch.autograd.grad([S, V], [p["w"], p["a"], p["b"], p["d"], p["x"]], [p["gS"], p["gV"]])
    return {"S": S, "V": V, "gw": g[0], "ga": g[1], "gb": g[2], "gd": g[3], "gx": g[4]}


# -------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind in ("step", "run", "batch"):
        if kind == "batch":
            n = case["networks"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
            m = 0.5 * (case["smin"] + case["smax"])
            plastic = 0.4
        else:
            n, m, plastic = case["neurons"], case["synapses"], 0.8 if case.get("stdp") else 0.0
        # per neuron and step: 20 B parameters, u, v, RNG and history read and
        # written; per event target and weight; per plastic synapse of a target
        # that fired, its source, the source's history and its accumulator
        neuron = case["steps"] * n
        events = neuron * IZH_RATE * m
        visits = neuron * IZH_RATE * m * plastic
        applied = n * m * plastic * 12 if case.get("period") else 0  # accumulator read and cleared, weight written
        return {"bytes": 84 * neuron + 8 * events + 16 * visits + applied, "flops": 120 * neuron + events + 4 * visits}
    if kind == "mixed":
        steps = case["steps"]
        n = case["lif"] + case["qif"] + case["hh"] + case["poisson"]
        events = steps * n * TORUS_RATE * case["synapses"]
        return {"bytes": steps * (68 * case["lif"] + 12 * case["qif"] + 40 * case["hh"] + 36 * case["poisson"])
                + 8 * events,
                "flops": steps * (20 * case["lif"] + 200 * case["qif"] + 999 * 150 * case["hh"]) + events}
    if kind == "kuramoto":
        # per step, four evaluations of the coupling sum over all synapses
        s = case["neurons"] * case["indegree"]
        return {"bytes": case["steps"] * (12 * s + 16 * case["neurons"]), "flops": case["steps"] * 4 * 25 * s}
    if kind == "propagate":
        events = case["steps"] * case["fired"] * case["synapses"]
        return {"bytes": 8 * events + case["steps"] * (8 * case["neurons"] + 4 * case["fired"]), "flops": events}
    T, n, s = case["steps"], case["neurons"], case["neurons"] * case["synapses"]
    if kind == "forward":
        return {"bytes": 8 * s + 12 * T * n, "flops": 60 * T * n + 2 * IZH_RATE * T * s}
    # + spikes, potentials and their gradients read, the input gradient
    # written, the weights read again and their gradient written; every
    # synapse takes part in every step of the adjoint
    return {"bytes": 20 * s + 32 * T * n, "flops": 200 * T * n + 2 * T * s}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "kuramoto":
        return _exact_kuramoto(case, seed)
    if kind == "propagate":
        return _exact_propagate(case, seed)
    if kind in ("forward", "train"):
        return _exact_float(case, seed)
    return None


def _exact_kuramoto(case, seed):
    omega, theta, src, tgt, delay, w = _oscillators(case, seed)
    n, H, h = case["neurons"], 32, 0.05
    omega, w, cmean = omega.astype(np.float64), w.astype(np.float64), float(case["indegree"])
    two_pi = 2 * math.pi

    def wrap(p):
        r = np.fmod(p, two_pi)
        return r + np.where(p < 0, two_pi, 0.0)

    # slot 0 the initial phase, slots H-1, H-2, ... the phases before it
    hist = np.zeros((H, n))
    hist[0] = theta
    for t in range(H - 1):
        hist[(-t - 1) % H] = wrap(hist[(-t) % H] - omega)
    for cycle in range(case["steps"]):
        source = hist[(cycle - (delay.astype(np.int64) - 1)) % H, src]
        # a delay that reads the slot this step writes sees the new phase of
        # lower-index sources; their contribution is left to one pass in order
        late = (delay.astype(np.int64) - 1) % H == H - 1
        here = hist[cycle % H]

        def advance(source, here, tgt, w, om, m):
            def k(p):
                s = np.zeros(m)
                np.add.at(s, tgt, w * np.sin(source - p[tgt]))
                return om + s / cmean
            k0 = k(here)
            k1 = k(here + k0 * 0.5 * h)
            k2 = k(here + k1 * 0.5 * h)
            k3 = k(here + k2 * h)
            return wrap(here + h * (k0 + 2 * k1 + 2 * k2 + k3) / 6.0)

        if not late.any():
            hist[(cycle + 1) % H] = advance(source, here, tgt, w, omega, n)
            continue
        order = np.argsort(tgt, kind="stable")
        ends = np.searchsorted(tgt[order], np.arange(n), side="right")
        begins = np.searchsorted(tgt[order], np.arange(n))
        for i in range(n):
            k = order[begins[i]:ends[i]]
            s = hist[(cycle - (delay[k].astype(np.int64) - 1)) % H, src[k]]
            hist[(cycle + 1) % H, i] = advance(s, here[i:i + 1], np.zeros(k.size, np.int64), w[k], omega[i:i + 1], 1)[0]
    return hist[case["steps"] % H].copy()


def _exact_propagate(case, seed):
    spec = _izhikevich(case, seed)
    fired = _fired_lists(case, seed)
    n, m = case["neurons"], case["synapses"]
    # weights in the simulation's Q11.20 format
    q = np.trunc(spec.weight.astype(np.float64) * (1 << 20)).reshape(n, m)
    tgt, delay = spec.target.reshape(n, m), spec.delay.reshape(n, m)
    E, I = np.zeros((case["steps"], n)), np.zeros((case["steps"], n))
    for s in range(case["steps"]):
        for past in range(s + 1):
            rows = fired[past]
            at = delay[rows] == s + 1 - past
            wt, tt = q[rows][at], tgt[rows][at]
            np.add.at(E[s], tt[wt >= 0], wt[wt >= 0])
            np.add.at(I[s], tt[wt < 0], wt[wt < 0])
    return {"E": E / (1 << 20), "I": I / (1 << 20)}


def _exact_float(case, seed):
    """The float mode's forward and adjoint in float64, step by step: NeMo's
    four substeps while v < 30, reset with the spike held constant, and the
    surrogate 1 / (1 + 10 |v - 30|)^2 where spikes feed synapses and the loss."""
    spec, inp = _float_inputs(case, seed)
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    p = {k: torch.tensor(v, dtype=torch.float64, device=dev) for k, v in inp.items()}
    src, tgt, delay = (torch.tensor(v.astype(np.int64), device=dev) for v in (spec.source, spec.target, spec.delay))
    T, n, D, h = case["steps"], case["neurons"], int(spec.delay.max()), 0.25
    a, b, c, d, w = p["a"], p["b"], p["c"], p["d"], p["w"]
    S = torch.zeros((T + D, n), dtype=torch.float64, device=dev)  # row D + t: step t
    V = torch.zeros((T, n), dtype=torch.float64, device=dev)
    entry, inputs = [], []
    v, u = p["v0"].clone(), p["u0"].clone()

    def substeps(v, u, I):
        vs, us, masks = [v], [u], []
        m = torch.ones(n, dtype=torch.bool, device=dev)
        for _ in range(4):
            masks.append(m)
            v = torch.where(m, v + h * (0.04 * v * v + 5.0 * v + 140.0 - u + I), v)
            u = torch.where(m, u + h * a * (b * v - u), u)
            vs.append(v)
            us.append(u)
            m = m & (v < 30.0)
        return vs, us, masks

    for t in range(T):
        I = p["x"][t].index_add(0, tgt, w * S[D + t - delay, src])
        entry.append((v, u))
        inputs.append(I)
        vs, us, _ = substeps(v, u, I)
        s = (vs[4] >= 30.0).to(torch.float64)
        v = torch.where(s > 0, c, vs[4])
        u = us[4] + s * d
        S[D + t] = s
        V[t] = v
    if case["kind"] == "forward":
        return {"S": S[D:].clone(), "V": V}
    LI = torch.zeros((T + D + 1, n), dtype=torch.float64, device=dev)  # rows from T on: zero
    Lv, Lu = torch.zeros(n, dtype=torch.float64, device=dev), torch.zeros(n, dtype=torch.float64, device=dev)
    gw = torch.zeros_like(w)
    ga, gb, gd = torch.zeros_like(a), torch.zeros_like(a), torch.zeros_like(a)
    gx = torch.zeros_like(p["x"])
    for t in reversed(range(T)):
        ahead = LI[t + delay, tgt]
        lS = p["gS"][t].index_add(0, src, w * ahead)
        gw += S[D + t, src] * ahead
        vs, us, masks = substeps(*entry[t], inputs[t])
        s = S[D + t]
        lv, lu = Lv + p["gV"][t], Lu
        gd += lu * s
        lv = lv * (1.0 - s) + lS / (1.0 + 10.0 * (vs[4] - 30.0).abs()) ** 2
        lI = torch.zeros_like(lv)
        for k in (3, 2, 1, 0):
            m = masks[k].to(torch.float64)
            tot = lv + lu * h * a * b
            ga += m * lu * h * (b * vs[k + 1] - us[k])
            gb += m * lu * h * a * vs[k + 1]
            nlu = lu * (1.0 - h * a) - tot * h
            lv = torch.where(masks[k], tot * (1.0 + h * (0.08 * vs[k] + 5.0)), lv)
            lu = torch.where(masks[k], nlu, lu)
            lI += m * tot * h
        Lv, Lu = lv, lu
        LI[t] = lI
        gx[t] = lI
    return {"S": S[D:].clone(), "V": V, "gw": gw, "ga": ga, "gb": gb, "gd": gd, "gx": gx}
