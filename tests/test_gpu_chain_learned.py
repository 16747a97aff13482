"""Learned step sizes in the chain form of the RK5 update, with proposals that
bind: the network's inputs gathered from the lanes of a neuron's group, its
output handed back to them, and the error ratio kept as its next input.  A
wrong port or neuron changes only step sizes, so rasters, state and attempt
counts are compared bit for bit with one lane per neuron (no chain waves),
which evaluates the same predictor from its own registers."""
import numpy as np
import pytest

from conftest import gpu_available
from test_gpu_predictor import NH, NI, O_B1, O_B2, O_B3, O_W1, O_W2, O_W3
from test_gpu_chain import _same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ngpu():
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu
    yield nestgpu
    nestgpu.SetStepPredictorMode(0)


def _params(ngpu):
    # inputs scaled to the network's range, every one with weight in the
    # proposal; log2(h / dt) around -2, mostly below the controller's
    rng = np.random.default_rng(8)
    P = np.zeros(ngpu.PREDICTOR_N_PARAMS, np.float32)
    P[0:NI] = [-55.0, 60.0, 2.0, 2.0, 2.0, 2.0, -2.0, -5.0]
    P[NI:2 * NI] = [0.1, 0.03, 0.5, 0.5, 0.5, 0.5, 0.4, 0.3]
    P[O_W1:O_B1] = rng.normal(0.0, 0.5, O_B1 - O_W1)
    P[O_B1:O_W2] = rng.normal(0.0, 0.1, NH)
    P[O_W2:O_B2] = rng.normal(0.0, 0.25, NH * NH)
    P[O_W3:O_B3] = rng.normal(0.0, 0.2, NH)
    P[O_B3] = -2.0
    return P


def _run(ngpu, monkeypatch, env, ports, n, mode):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        ngpu.SetRandomSeed(77)
        ngpu.SetPredictorParams(_params(ngpu))
        ngpu.SetStepPredictorMode(mode)
        nodes = ngpu.Create("aeif_cond_beta_multisynapse", n, ports)
        ngpu.SetStatus(nodes, "I_e", 700.0)
        rng = np.random.default_rng(3)
        ngpu.SetStatus(nodes, "V_m", {"array": rng.uniform(-70.0, -58.0, n).tolist()})
        pg = ngpu.Create("poisson_generator")
        ngpu.SetStatus(pg, {"rate": 8000.0, "stop": 30.0})
        ngpu.Connect(pg, nodes, {"rule": "all_to_all"}, {"weight": 0.3, "delay": 0.1, "receptor": 0})
        for p in range(ports):
            ngpu.Connect(nodes, nodes, {"rule": "fixed_indegree", "indegree": 5},
                         {"weight": (0.3 + 0.2 * p) / ports, "delay": 0.1 * (p + 1), "receptor": p})
        ngpu.ActivateRecSpikeTimes(nodes, 500)
        ngpu.Simulate(15.0)
        ngpu.Simulate(25.1)
        names = list(ngpu.GetScalVarNames(nodes[0])) + list(ngpu.GetPortVarNames(nodes[0]))
        state = {k: np.array(ngpu.GetStatus(nodes, k), np.float32) for k in names}
        return ngpu.GetRecSpikeTimes(nodes), state, ngpu.GetStepStats()
    finally:
        ngpu.SetStepPredictorMode(0)
        for k in env:
            monkeypatch.delenv(k)
        ngpu.ResetKernel()


@pytest.mark.parametrize("ports", [1, 2, 3, 4, 7])
def test_binding_proposals_match_lane_per_neuron(ngpu, monkeypatch, ports):
    # the split cap: none, the default's, and one that splits most spiking
    # steps; one chain wave holds 16 (8 from four ports on) neurons at once
    n = 200
    whole = {"NGPU_RK5_DEFER": "0"}
    plain = _run(ngpu, monkeypatch, {"NGPU_RK5_CHAIN_WAVES": "0", **whole}, ports, n, "plain")
    ref = _run(ngpu, monkeypatch, {"NGPU_RK5_CHAIN_WAVES": "0", **whole}, ports, n, "learned")
    assert sum(len(t) for t in ref[0]) > 100 and ref[2]["dropped_spikes"] == 0
    assert ref[2]["attempts"] > 1.1 * plain[2]["attempts"]      # the proposals bind
    for env in ({}, whole, {"NGPU_RK5_DEFER": "5"}, {"NGPU_RK5_CHAIN_WAVES": "1"},
                {"NGPU_RK5_CHAIN_WAVES": "4", "NGPU_RK5_HOT_MARGIN": "0"},
                {"NGPU_RK5_CHAIN_WAVES": "0"}):
        got = _run(ngpu, monkeypatch, env, ports, n, "learned")
        assert got[2]["hot_listed"] > 50
        _same(got, ref)
