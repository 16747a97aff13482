"""The batch launch's configuration: what SetBatchConfig leaves out is the
engine's default, every default can be set again after another value, and the
autotuner leaves the choice of delivery to the engine where it was."""
import numpy as np
import pytest

from conftest import gpu_available
import netbuild
from test_gpu_delivery_choice import _batch

pytestmark = pytest.mark.gpu

KNOBS = ("variant", "iaf_unroll", "rk5_weight", "graph")


@pytest.fixture
def net(monkeypatch):
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu as ngpu
    monkeypatch.setenv("NGPU_FUSED_EVENTS", "100")
    ngpu.ResetKernel()
    ngpu.SetVerbosityLevel(0)
    ngpu.SetRandomSeed(5)
    pops = _batch(ngpu)
    ngpu.Calibrate()
    yield ngpu, pops[0][0]
    ngpu.ResetKernel()


def _knobs(ngpu):
    c = ngpu.GetBatchConfig()
    assert c["on"] == 1 and c["tiled_available"] == 1
    return tuple(c[k] for k in KNOBS)


def test_defaults_are_the_engines(net):
    ngpu, _ = net
    first = _knobs(ngpu)
    grid = ngpu.GetBatchConfig()["grid"]
    ngpu.SetBatchConfig(tiled=False)
    assert _knobs(ngpu) == first and ngpu.GetBatchConfig()["grid"] == grid
    ngpu.SetBatchConfig(variant=1, iaf_unroll=4, rk5_weight=2.0, graph=True)
    assert _knobs(ngpu) == (1, 4, 2.0, 1)
    ngpu.SetBatchConfig(iaf_unroll=first[1])
    assert _knobs(ngpu) == first
    with pytest.raises(ValueError):
        ngpu.SetBatchConfig(iaf_unroll=3)


def test_delivery_choice_can_be_given_back(net):
    ngpu, pop = net
    used = []

    def call(i_e, ms=30.0):
        ngpu.SetStatus(pop, "I_e", i_e)
        ngpu.Simulate(ms)
        used.append(ngpu.GetBatchConfig()["tiled"])

    ngpu.SetBatchConfig(tiled=True)
    call(0.0)               # silent, but tiled as set
    ngpu.SetBatchConfig()
    call(0.0)
    ngpu.SetBatchConfig(tiled="auto")
    call(0.0)
    call(3000.0)
    ms, n = ngpu.AutotuneBatch(4)
    assert n == 36
    call(0.0)
    call(3000.0)
    assert used == [1, 1, 0, 1, 0, 1]


def test_graph_replay_matches_direct_launches(monkeypatch):
    # the six-population mixed network, each step's launch replayed as a graph
    # node with the step's arguments, against one launch per population: three
    # Simulate calls, the graph made anew by the change of configuration
    # before the last one
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu as ngpu
    net = netbuild.mixed_network(seed=11)

    def run(batch, graph):
        monkeypatch.setenv("NGPU_BATCH", batch)
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        pops = []
        for p in net["pops"]:
            pops.append(ngpu.Create(p["model"], p["n"], p["n_port"]))
            if p["status"]:
                ngpu.SetStatus(pops[-1], p["status"])
        for p, nrn in zip(net["pops"], pops):
            pg = ngpu.Create("poisson_generator")
            ngpu.SetStatus(pg, "rate", p["rate"])
            ngpu.Connect(pg, nrn, {"rule": "all_to_all"},
                         {"weight": p["pw"], "delay": 0.1, "receptor": 0})
        for (s, t, port, w, d) in net["edges"]:
            for q in (0, 1):
                m = port == q
                netbuild.connect_edges_fast(ngpu, s[m], t[m], q, w[m], d[m])
        for nrn in pops:
            ngpu.ActivateRecSpikeTimes(nrn, 5000)
        ngpu.Calibrate()
        out = []
        for k, ms in enumerate((30.0, 20.1, 30.0)):
            if graph and k != 1:
                ngpu.SetBatchConfig(variant=k // 2, graph=True)
            ngpu.Simulate(ms)
            c = ngpu.GetBatchConfig()
            assert (c["on"], c["graph"]) == ((1, 1) if graph else (0, 0))
            st = ngpu.GetStepStats()
            out.append([st[k] for k in ("attempts", "rejected", "syn_events", "spikes")])
            out += [np.array(ngpu.GetStatus(nrn, "V_m_rel" if p["model"] == "iaf_psc_exp" else "V_m"),
                             np.float32).view(np.uint32).ravel().tolist()
                    for p, nrn in zip(net["pops"], pops)]
        out += [ngpu.GetRecSpikeTimes(nrn) for nrn in pops]
        ngpu.ResetKernel()
        return out

    ref = run("0", False)
    assert sum(len(t) for pop in ref[-6:] for t in pop) > 500
    assert run("1", True) == ref
