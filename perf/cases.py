"""Timed cases of the simulation framework: what a user's script has it do
through the nestgpu module and the C entry points of include/nestgpu_C.h.

A case is a small dict of plain values.  `prepare` builds its network
(Create / SetStatus / Connect, calibrated and run past its first transient, as
a script does before it measures), `run` is one Simulate call with the
read-back of the state that a script wants after it.  Every random number of
a network (sources, weights, delays, initial potentials, Poisson input) comes
from the seed.

The library holds one network per loaded library.  A program that keeps
several networks loads it once for each, through the NESTGPU_LIB variable that
nestgpu.py documents; `_Network` does that with copies of the built library
and gives a copy back for the next network when it is dropped.

Networks are the ones of nest-gpu_amd/workloads.py and tests/ at sizes that
can be built in about a second, weights scaled with the indegree so that the
mean input stays the same.
"""
import ctypes
import importlib.util
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

DT = 0.1
ROOT = os.getcwd()
PKG = os.path.join(ROOT, "nest-gpu_amd")

# ---------------------------------------------------------------------------
# the cases


def listed():
    return [
        # a first script, or one point of a parameter scan: one neuron, three
        # receptor ports, a multimeter on it; every step is a few tiny launches
        {"name": "trace_1", "kind": "trace", "model": "aeif_cond_beta_multisynapse", "n": 1,
         "ports": 3, "steps": 200},
        # the 1,000-neuron AdEx network (one Poisson generator per neuron)
        {"name": "adex_1k", "kind": "adex", "n": 1000, "ports": 2, "k": 100, "d_max": 20,
         "own_poisson": True, "hetero": False, "learned": False, "steps": 200},
        # a full cortical indegree on a part of the million-neuron network
        {"name": "adex_60k", "kind": "adex", "n": 60000, "ports": 2, "k": 1000, "d_max": 50,
         "own_poisson": False, "hetero": False, "learned": False, "steps": 200},
        # the million-neuron network, with a tenth of its indegree so that it
        # can be built many times over: the neuron update at full size
        {"name": "adex_1m", "kind": "adex", "n": 1000000, "ports": 2, "k": 100, "d_max": 50,
         "own_poisson": False, "hetero": False, "learned": False, "steps": 300},
        # four ports, learned step sizes, per-neuron Poisson rates
        {"name": "adex_learned_100k", "kind": "adex", "n": 100000, "ports": 4, "k": 200,
         "d_max": 50, "own_poisson": True, "hetero": False, "learned": True, "steps": 200},
        # heterogeneous neurons (parameters drawn per neuron), odd sizes
        {"name": "adex_hetero_9973", "kind": "adex", "n": 9973, "ports": 3, "k": 151, "d_max": 33,
         "own_poisson": False, "hetero": True, "learned": False, "steps": 200},
        # the microcircuit's eight iaf_psc_exp populations, a tenth of the size
        {"name": "circuit_7717", "kind": "circuit", "scale": 0.1, "p_max": 0.15, "steps": 200},
        # ... at full size with an eighth of the connection probabilities
        {"name": "circuit_77k", "kind": "circuit", "scale": 1.0, "p_max": 0.01875, "steps": 200},
        # six populations of five models, as the mixed-model test has them
        {"name": "mixed_840", "kind": "mixed", "n": 840, "k": 50, "steps": 200},
        # ... as the batching workload has them, a tenth of its size
        {"name": "mixed_50k", "kind": "mixed", "n": 50330, "k": 200, "steps": 200},
        # plastic (STDP) synapses between the excitatory neurons
        {"name": "stdp_2k", "kind": "stdp", "n": 2000, "k": 100, "steps": 200},
        # training of the step-size network: forward and backward, Adam
        {"name": "train_8192", "kind": "train", "log": 200000, "batch": 8192, "updates": 50},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["trace", "adex", "adex", "adex", "circuit", "circuit", "mixed", "mixed",
                       "stdp", "train"])
    if kind == "trace":
        return {"kind": kind, "n": _log_int(rng, 1, 64), "ports": rng.randint(1, 6),
                "model": rng.choice(["aeif_cond_beta_multisynapse",
                                     "aeif_cond_alpha_multisynapse"]),
                "steps": rng.randint(100, 200)}
    if kind == "adex":
        n = _log_int(rng, 700, 1000000)
        form = rng.choice(["plain", "plain", "hetero", "learned"])
        if form != "plain":
            n = min(n, 120000)
        k_hi = max(60, min(1000, n // 4, 100000000 // n))
        return {"kind": kind, "n": n, "ports": rng.randint(1, 4) if form != "learned" else 4,
                "k": _log_int(rng, 50, k_hi), "d_max": rng.randint(1, 60),
                "own_poisson": rng.random() < 0.5 and n <= 120000, "hetero": form == "hetero",
                "learned": form == "learned", "steps": rng.randint(100, 250)}
    if kind == "circuit":
        scale = math.exp(rng.uniform(math.log(0.02), 0.0))
        most = 60.0e6 / (0.5 * (77169 * scale) ** 2)    # about 6e7 synapses at most
        return {"kind": kind, "scale": round(scale, 4), "steps": rng.randint(100, 200),
                "p_max": round(min(0.15, most) * rng.uniform(0.3, 1.0), 5)}
    if kind == "mixed":
        n = _log_int(rng, 700, 60000)
        return {"kind": kind, "n": n, "k": _log_int(rng, 40, min(200, n // 4)),
                "steps": rng.randint(100, 200)}
    if kind == "stdp":
        n = _log_int(rng, 300, 4000)
        return {"kind": kind, "n": n, "k": rng.randint(30, 100), "steps": rng.randint(100, 200)}
    return {"kind": "train", "log": rng.randint(20000, 400000), "batch": 64 * rng.randint(1, 256),
            "updates": rng.randint(10, 60)}


# ---------------------------------------------------------------------------
# one network per loaded library
_idle = []
_folder = None


def _load():
    """A nestgpu module with a library of its own."""
    global _folder
    if _folder is None:
        _folder = tempfile.mkdtemp(prefix="nestgpu_cases_")
    copy = os.path.join(_folder, "libnestgpu_amd_%d.so" % len(os.listdir(_folder)))
    shutil.copy(os.path.join(PKG, "libnestgpu_amd.so"), copy)
    before = os.environ.get("NESTGPU_LIB")
    os.environ["NESTGPU_LIB"] = copy
    try:
        spec = importlib.util.spec_from_file_location("nestgpu", os.path.join(PKG, "nestgpu.py"))
        m = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(m)
    finally:
        if before is None:
            del os.environ["NESTGPU_LIB"]
        else:
            os.environ["NESTGPU_LIB"] = before
    m.SetOnException(1)
    return m


class _Network:
    def __init__(self, case, seed):
        self.case = case
        self.m = _idle.pop() if _idle else _load()
        self.m.ResetKernel()
        self.m.SetVerbosityLevel(0)
        self.m.SetStepPredictorMode(0)
        self.m.SetRandomSeed(seed + 1)

    def __del__(self):
        self.m.ResetKernel()
        _idle.append(self.m)

    def var(self, nodes, name):
        """A variable of all nodes as an array (NESTGPU_GetNeuronVar)."""
        m = self.m
        p = m._lib_call("GetNeuronVar", nodes.i0, nodes.n, name.encode())
        size = m.GetNeuronVarSize(nodes.i0, name)
        return np.ctypeslib.as_array(p, shape=(nodes.n * size,)).copy().reshape(nodes.n, size)

    def counts(self, nodes):
        """Spike counts of all nodes (NESTGPU_GetNeuronIntVar)."""
        p = self.m._lib_call("GetNeuronIntVar", nodes.i0, nodes.n, b"spike_count")
        return np.ctypeslib.as_array(p, shape=(nodes.n,)).copy()

    def indegree(self, src, tgt, k, port, w, d, syn_group=0):
        """Fixed indegree k with an array of weights and one of delays."""
        m, lib = self.m, self.m._nestgpu
        w = np.ascontiguousarray(w, np.float32)
        d = np.ascontiguousarray(d, np.float32)
        m.ConnSpecInit()
        m.SynSpecInit()
        m.SetConnSpecParam("rule", 3)      # fixed_indegree
        m.SetConnSpecParam("indegree", int(k))
        m.SetSynSpecIntParam("receptor", port)
        if syn_group:
            m.SetSynSpecIntParam("synapse_group", syn_group)
        lib.NESTGPU_SetSynSpecFloatPtParam(b"weight_array", w.ctypes.data_as(ctypes.c_void_p))
        lib.NESTGPU_SetSynSpecFloatPtParam(b"delay_array", d.ctypes.data_as(ctypes.c_void_p))
        lib.NESTGPU_ConnectSeqSeq(src.i0, src.n, tgt.i0, tgt.n)
        m._check()

    def total(self, src, tgt, n, port, w, d):
        """n synapses between random pairs (fixed_total_number)."""
        m, lib = self.m, self.m._nestgpu
        m.ConnSpecInit()
        m.SynSpecInit()
        m.SetConnSpecParam("rule", 2)
        m.SetConnSpecParam("total_num", int(n))
        m.SetSynSpecIntParam("receptor", port)
        lib.NESTGPU_SetSynSpecFloatPtParam(b"weight_array", w.ctypes.data_as(ctypes.c_void_p))
        lib.NESTGPU_SetSynSpecFloatPtParam(b"delay_array", d.ctypes.data_as(ctypes.c_void_p))
        lib.NESTGPU_ConnectSeqSeq(src.i0, src.n, tgt.i0, tgt.n)
        m._check()

    def poisson(self, tgt, rate, weight, delay=DT):
        """One generator for all targets, or with an array of rates one each."""
        m = self.m
        if np.ndim(rate) == 0:
            pg = m.Create("poisson_generator")
            m.SetStatus(pg, "rate", float(rate))
            rule = "all_to_all"
        else:
            pg = m.Create("poisson_generator", tgt.n)
            for i, r in enumerate(rate.tolist()):
                m.SetNeuronScalParam(pg.i0 + i, 1, "rate", r)
            rule = "one_to_one"
        m.Connect(pg, tgt, {"rule": rule}, {"weight": weight, "delay": delay, "receptor": 0})


def _uniform(rng, n, lo, hi):
    w = rng.random(n, dtype=np.float32)
    w *= np.float32(hi - lo)
    w += np.float32(lo)
    return w


def _delays(rng, n, d_max):
    d = rng.integers(1, d_max + 1, size=n, dtype=np.int16).astype(np.float32)
    d *= np.float32(DT)
    return d


def _scatter(net, nodes, rng, lo, hi):
    net.m.SetStatus(nodes, "V_m", {"array": _uniform(rng, nodes.n, lo, hi).tolist()})


# ---------------------------------------------------------------------------
# kinds


def _trace_inputs(case, seed):
    """Initial states below threshold, currents and receptor parameters."""
    rng = np.random.default_rng(seed)
    n, p = case["n"], case["ports"]
    f = lambda lo, hi, *s: rng.uniform(lo, hi, s).astype(np.float32)  # noqa: E731
    return {"V_m": f(-75.0, -62.0, n), "w": f(-20.0, 60.0, n), "g": f(0.0, 2.0, n, p),
            "g1": f(0.0, 1.0, n, p), "E_rev": f(-85.0, -60.0, p), "tau_rise": f(1.0, 10.0, p),
            "tau_decay": f(11.0, 40.0, p), "I_e": float(f(0.0, 150.0)), "a": 4.0, "b": 80.5}


def _trace(net, case, seed):
    m, x = net.m, _trace_inputs(case, seed)
    net.x = x
    net.nodes = m.Create(case["model"], case["n"], case["ports"])
    st = {"E_rev": x["E_rev"].tolist(), "I_e": x["I_e"], "a": x["a"], "b": x["b"]}
    if "beta" in case["model"]:
        st.update({"tau_rise": x["tau_rise"].tolist(), "tau_decay": x["tau_decay"].tolist()})
    else:
        st["tau_syn"] = x["tau_decay"].tolist()
    m.SetStatus(net.nodes, st)
    n = case["n"]
    net.rec = m.CreateRecord("", ["V_m"] * n, list(range(net.nodes.i0, net.nodes.i0 + n)), [0] * n)
    m.Simulate(DT)


def _run_trace(net):
    """A point of a scan: the initial state set, a stretch simulated, the
    multimeter's rows of it and the final state read."""
    m, x, n, steps = net.m, net.x, net.nodes.n, net.case["steps"]
    for name in ("V_m", "w"):
        for i, v in enumerate(x[name].tolist()):
            m.SetNeuronScalVar(net.nodes.i0 + i, 1, name, v)
    for name in ("g", "g1"):
        for i in range(n):
            m.SetNeuronArrayVar(net.nodes.i0 + i, 1, name, x[name][i])
    m.Simulate(steps * DT)
    rows = m._lib_call("GetRecordData", net.rec)
    last = m.GetRecordDataRows(net.rec)
    v = np.empty((steps, n), np.float32)
    for r in range(steps):
        v[r] = np.ctypeslib.as_array(rows[last - steps + r], shape=(n + 1,))[1:]
    return {"V_m": v, "w": net.var(net.nodes, "w"), "g": net.var(net.nodes, "g"),
            "g1": net.var(net.nodes, "g1")}


def _exact_trace(case, seed):
    x = _trace_inputs(case, seed)
    g = {k: np.asarray(v, np.float64) for k, v in x.items()}
    beta = "beta" in case["model"]
    tr, td = (g["tau_rise"] if beta else g["tau_decay"]), g["tau_decay"]
    V, w, gg, g1 = g["V_m"], g["w"], g["g"], g["g1"]

    def rhs(V, w, gg, g1):
        i_syn = (gg * (g["E_rev"] - V[:, None])).sum(1)
        spike = 2.0 * np.exp((np.minimum(V, 0.0) + 50.4000015258789) / 2.0)
        dv = (-30.0 * (V + 70.5999984741211 - spike) + i_syn - w + g["I_e"]) / 281.0
        return dv, (g["a"] * (V + 70.5999984741211) - w) / 144.0, g1 - gg / td, -g1 / tr

    rows, m = np.empty((case["steps"], case["n"])), 10
    h = float(np.float32(DT)) / m
    for r in range(case["steps"]):
        for _ in range(m):      # classical RK4, step 0.01 ms
            y = (V, w, gg, g1)
            k1 = rhs(*y)
            k2 = rhs(*[a + 0.5 * h * b for a, b in zip(y, k1)])
            k3 = rhs(*[a + 0.5 * h * b for a, b in zip(y, k2)])
            k4 = rhs(*[a + h * b for a, b in zip(y, k3)])
            V, w, gg, g1 = [a + h / 6.0 * (p + 2.0 * q + 2.0 * s + t)
                            for a, p, q, s, t in zip(y, k1, k2, k3, k4)]
        rows[r] = V
    return {"V_m": rows, "w": w[:, None], "g": gg, "g1": g1}


def _adex(net, case, seed):
    """scale_adex / predictor_adex / the 1,000-neuron network of the tests:
    80% excitatory sources; half of the even ports fast, as the ports of
    predictor_adex; weights x 1000 / k."""
    rng = np.random.default_rng(seed)
    m, n, k, ports = net.m, case["n"], case["k"], case["ports"]
    ne = int(0.8 * n)
    model = "aeif_cond_alpha_multisynapse" if case["hetero"] else "aeif_cond_beta_multisynapse"
    net.nodes = m.Create(model, n, ports)
    inh = [p % 2 == 1 for p in range(ports)]
    st = {"E_rev": [-85.0 if i else 0.0 for i in inh]}
    slow = [p >= 2 for p in range(ports)]
    if case["hetero"]:
        st["tau_syn"] = [5.0 if s else 1.0 for s in slow]
    else:
        st.update({"tau_rise": [2.0 if s else 1.0 for s in slow],
                   "tau_decay": [10.0 if s else 1.0 for s in slow]})
    m.SetStatus(net.nodes, st)
    if case["hetero"]:
        for name, mean in (("C_m", 281.0), ("g_L", 30.0), ("tau_w", 144.0)):
            m.SetStatus(net.nodes, name, {"array": _uniform(rng, n, 0.9 * mean, 1.1 * mean).tolist()})
    if case["learned"]:
        with open(os.path.join(PKG, "predictors", "predictor_adex.json")) as f:
            m.SetPredictorParams(np.array(json.load(f)["params"], np.float32))
        m.SetStepPredictorMode("learned")
    if n <= 120000:     # one call per neuron
        _scatter(net, net.nodes, rng, -70.0, -55.0)
    s = 1000.0 / k
    pw = 0.237 if ports < 4 else 0.2
    rate = _uniform(rng, n, 12000.0, 28000.0) if case["own_poisson"] else 20000.0
    if case["learned"]:
        rate = _uniform(rng, n, 5000.0, 40000.0)
    net.poisson(net.nodes, rate, pw)
    exc, inhib = net.nodes[0:ne], net.nodes[ne:n]
    for p in range(ports):
        peers = sum(i == inh[p] for i in inh)
        kp = max(1, int(k * (0.2 if inh[p] else 0.8) / peers))
        lo, hi = (0.175, 0.525) if inh[p] else (0.025, 0.075)
        f = s * (0.2 if slow[p] else 1.0)
        net.indegree(inhib if inh[p] else exc, net.nodes, kp, p,
                     _uniform(rng, n * kp, f * lo, f * hi), _delays(rng, n * kp, case["d_max"]))
    m.ActivateSpikeCount(net.nodes)
    m.Simulate(30.0)


def _run_net(net):
    """A stretch of the simulation, then the state a script looks at."""
    net.m.Simulate(net.case["steps"] * DT)
    return [{"V_m": net.var(p, "V_m_rel" if iaf else "V_m"), "spikes": net.counts(p)}
            for p, iaf in net.pops]


MC_SIZES = [20683, 5834, 21915, 5479, 4850, 1065, 14395, 2948]
MC_K_EXT = [1600, 1500, 2100, 1900, 2000, 1900, 2900, 2100]
MC_PARAMS = {"E_L": -65.0, "Theta_rel": 15.0, "V_reset_rel": 0.0, "C_m": 250.0, "tau_m": 10.0,
             "tau_ex": 0.5, "tau_in": 0.5, "t_ref": 2.0}


def _circuit(net, case, seed):
    """The microcircuit workload: sizes x scale, connection probabilities
    U(p_max / 15, p_max) per population pair."""
    rng = np.random.default_rng(seed)
    m = net.m
    pops = [m.Create("iaf_psc_exp", max(2, int(round(s * case["scale"]))), 2) for s in MC_SIZES]
    for p in pops:
        m.SetStatus(p, MC_PARAMS)
        m.SetStatus(p, "V_m_rel", {"array": _uniform(rng, p.n, 0.0, 15.0).tolist()})
    prob = rng.uniform(case["p_max"] / 15.0, case["p_max"], (8, 8))
    for j, pre in enumerate(pops):
        exc = j % 2 == 0
        for i, post in enumerate(pops):
            k = max(1, int(round(prob[i, j] * pre.n * post.n)))
            w = rng.standard_normal(k, np.float32)
            d = rng.standard_normal(k, np.float32)
            if exc:
                w = np.maximum(w * np.float32(8.78) + np.float32(87.8), 0)
                d = np.maximum(d * np.float32(0.75) + np.float32(1.5), np.float32(DT))
            else:
                w = np.minimum(w * np.float32(35.12) - np.float32(351.2), 0)
                d = np.maximum(d * np.float32(0.375) + np.float32(0.75), np.float32(DT))
            net.total(pre, post, k, 0 if exc else 1, w, d)
    for p, kx in zip(pops, MC_K_EXT):
        net.poisson(p, 8.0 * kx, 87.8, 1.5)
        m.ActivateSpikeCount(p)
    net.pops = [(p, True) for p in pops]
    m.Simulate(30.0)


# model, share of the neurons, ports, status, excitatory mean weight at an
# indegree of 500, inhibitory sign, Poisson rate and weight (the batching
# workload's populations)
MIX = [
    ("izhikevich_cond_beta", 300, 2,
     {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [2.0, 2.0]}, 0.0004, 1.0,
     8000.0, 0.006),
    ("izhikevich_cond_beta", 3000, 2,
     {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [2.0, 2.0]}, 0.0004, 1.0,
     8000.0, 0.006),
    ("aeif_psc_exp", 30000, 2, {}, 4.0, 1.0, 20000.0, 170.0),
    ("aeif_cond_alpha_multisynapse", 120000, 4,
     {"E_rev": [0.0, -85.0, 0.0, -85.0], "tau_syn": [1.0, 1.0, 5.0, 5.0]}, 0.065, 1.0,
     20000.0, 0.25),
    ("aeif_cond_beta_multisynapse", 300000, 2,
     {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [1.0, 1.0]}, 0.1, 1.0,
     20000.0, 0.3),
    ("iaf_psc_exp", 50000, 2, {}, 9.0, -1.0, 8000.0, 22.0),
]
# shares of the mixed-model test network, used below 5,000 neurons
MIX_SMALL = [30, 60, 100, 200, 300, 150]


def _mixed(net, case, seed):
    rng = np.random.default_rng(seed)
    m, n, k = net.m, case["n"], case["k"]
    share = [p[1] for p in MIX] if n >= 5000 else MIX_SMALL
    sizes = [max(5, int(n * s / sum(share))) for s in share]
    pops = [m.Create(p[0], s, p[2]) for p, s in zip(MIX, sizes)]
    for p, pop in zip(MIX, pops):
        if p[3]:
            m.SetStatus(pop, p[3])
    n_tot = sum(sizes)
    ne = int(0.8 * n_tot)
    i0 = pops[0].i0
    exc, inh = m.NodeSeq(i0, ne), m.NodeSeq(i0 + ne, n_tot - ne)
    ke = int(0.8 * k)
    for p, pop in zip(MIX, pops):
        we = p[4] * 500.0 / k
        for src, kk, port, mean, d_mu, d_sd in ((exc, ke, 0, we, 1.5, 0.75),
                                                (inh, k - ke, 1, 4.0 * we * p[5], 0.75, 0.375)):
            c = pop.n * kk
            w = (rng.standard_normal(c, np.float32) * np.float32(0.1) + 1) * np.float32(mean)
            w = np.maximum(w, 0) if mean > 0 else np.minimum(w, 0)
            d = np.maximum(rng.standard_normal(c, np.float32) * np.float32(d_sd) + np.float32(d_mu),
                           np.float32(DT))
            net.indegree(src, pop, kk, port, w, d)
    for p, pop in zip(MIX, pops):
        net.poisson(pop, p[6], p[7])
        m.ActivateSpikeCount(pop)
    net.pops = [(pop, p[0] == "iaf_psc_exp") for p, pop in zip(MIX, pops)]
    m.Simulate(30.0)


def _stdp(net, case, seed):
    """The 1,000-neuron network's shape with STDP from excitatory sources."""
    rng = np.random.default_rng(seed)
    m, n, k = net.m, case["n"], case["k"]
    ne, ke = int(0.8 * n), int(0.8 * k)
    net.nodes = m.Create("aeif_cond_beta_multisynapse", n, 2)
    m.SetStatus(net.nodes, {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [1.0, 1.0]})
    _scatter(net, net.nodes, rng, -70.0, -55.0)
    s = 1000.0 / k
    g = m.CreateSynGroup("stdp", {"tau_plus": 20.0, "tau_minus": 20.0, "lambda": 0.01, "alpha": 1.0,
                                  "mu_plus": 1.0, "mu_minus": 1.0, "Wmax": 0.2 * s})
    net.indegree(net.nodes[0:ne], net.nodes, ke, 0, _uniform(rng, n * ke, 0.025 * s, 0.075 * s),
                 _delays(rng, n * ke, 20), g.i_syn_group)
    net.indegree(net.nodes[ne:n], net.nodes, k - ke, 1,
                 _uniform(rng, n * (k - ke), 0.175 * s, 0.525 * s), _delays(rng, n * (k - ke), 20))
    net.poisson(net.nodes, 20000.0, 0.237)
    m.ActivateSpikeCount(net.nodes)
    m.Simulate(30.0)


def _train(net, case, seed):
    """A log in the shape of logged steps: states near rest and on the spike
    upswing, the step sizes falling with the potential."""
    rng = np.random.default_rng(seed)
    n = case["log"]
    rec = np.empty((n, 10), np.float32)
    rec[:, 0] = rng.normal(-55.0, 8.0, n) + 40.0 * (rng.random(n) < 0.1)
    rec[:, 1] = rng.normal(60.0, 30.0, n)
    rec[:, 2:6] = np.abs(rng.normal(0.0, 2.0, (n, 4)))
    rec[:, 6] = -np.abs(rng.normal(0.0, 4.0, n))
    rec[:, 7] = rng.normal(-6.0, 3.0, n)
    rec[:, 8] = np.minimum(0.0, rec[:, 6] - 0.05 * np.maximum(rec[:, 0] + 50.0, 0.0)
                           + rng.normal(0.0, 0.3, n))
    rec[:, 9] = rng.random(n) < 0.4
    net.m.StartPredictorLog(n)
    net.m.AppendPredictorLog(rec)
    net.m.InitPredictor(seed + 1)
    net.start = net.m.GetPredictorParams()
    net.seed = seed


def _run_train(net):
    net.m.SetPredictorParams(net.start)
    loss = net.m.TrainPredictor(net.case["updates"], net.case["batch"], 1e-3, net.seed + 2)
    return {"loss": loss, "params": net.m.GetPredictorParams()}


# ---------------------------------------------------------------------------
_PREPARE = {"trace": _trace, "adex": _adex, "circuit": _circuit, "mixed": _mixed, "stdp": _stdp,
            "train": _train}


def prepare(case, seed):
    torch.cuda.init()
    net = _Network(case, seed)
    _PREPARE[case["kind"]](net, case, seed)
    if case["kind"] in ("adex", "stdp"):
        net.pops = [(net.nodes, False)]
    return net


def run(net):
    kind = net.case["kind"]
    return _run_trace(net) if kind == "trace" else _run_train(net) if kind == "train" \
        else _run_net(net)


def exact(case, seed):
    """Below threshold the equations have one solution; spiking networks
    amplify any difference in rounding without bound, so they have none."""
    return _exact_trace(case, seed) if case["kind"] == "trace" else None


def work(case):
    """Per neuron-step the state read and written, per port one ring entry
    read and cleared, per RK5 attempt (one per neuron-step but for spikes) its
    arithmetic; per synaptic event its record and the ring entry."""
    steps = case.get("steps", 0)
    kind = case["kind"]
    if kind == "train":
        per = 2 * (8 * 32 + 32 * 32 + 32) * 3
        return {"bytes": case["updates"] * (case["batch"] * 40 + 3 * 4 * 1393),
                "flops": case["updates"] * case["batch"] * per}
    if kind == "circuit":
        n = 77169 * case["scale"]
        n_syn = 0.53 * case["p_max"] * n * n
        rate = 100.0
        return {"bytes": steps * (n * (32 + 2 * 16) + n_syn * rate * 1e-4 * 16),
                "flops": steps * n * 20}
    n = case["n"]
    ports = case.get("ports", 2)
    nv = 2 + 2 * ports
    k = case.get("k", 0)
    rate = 0.0 if kind == "trace" else 10.0
    return {"bytes": steps * (n * (8 * nv + 24 + 16 * ports) + n * k * rate * 1e-4 * 26),
            "flops": steps * n * (56 * nv + 6 * (15 + 6 * ports))}
