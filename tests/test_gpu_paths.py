"""Choices made by size or by rate give the same bits either way: Poisson draws
by blocks for a whole wave (one chunk of the mean) or lane by lane (a lane of
the wave above 160 kHz at 0.1 ms), and the delivery of a dense network, fused
into the next launch with its spikes in parts (512 synapses and more a
neuron) or tiled, chosen at each Simulate call."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ngpu():
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu
    return nestgpu


@pytest.mark.parametrize("runs", ["1", "0"])
@pytest.mark.parametrize("model,weight", [("aeif_cond_beta_multisynapse", 0.05),
                                          ("iaf_psc_exp", 5.0)])
def test_poisson_blocks_match_lane_draws(ngpu, monkeypatch, runs, model, weight):
    monkeypatch.setenv("NGPU_POISSON_RUNS", runs)
    n, odd = 130, (5, 70, 129)     # one lane of every wave

    def run(fast):
        try:
            ngpu.ResetKernel()
            ngpu.SetVerbosityLevel(0)
            ngpu.SetRandomSeed(9)
            nodes = ngpu.Create(model, n, 2)
            gen = ngpu.Create("poisson_generator", n)
            rate = np.resize([0.0, 500.0, 8000.0, 40000.0, 159999.0, 160000.0], n)
            rate[list(odd)] = 200000.0 if fast else 0.0
            ngpu.SetStatus(gen, "rate", {"array": rate.tolist()})
            ngpu.Connect(gen, nodes, {"rule": "one_to_one"},
                         {"weight": weight, "delay": 0.1, "receptor": 0})
            ngpu.ActivateRecSpikeTimes(nodes, 200)
            ngpu.Simulate(10.0)
            names = list(ngpu.GetScalVarNames(nodes[0])) + list(ngpu.GetPortVarNames(nodes[0]))
            state = {k: np.array(ngpu.GetStatus(nodes, k), np.float32).reshape(n, -1) for k in names}
            return ngpu.GetRecSpikeTimes(nodes), state
        finally:
            ngpu.ResetKernel()

    by_lane, by_block = run(True), run(False)
    rest = [i for i in range(n) if i not in odd]
    assert [by_lane[0][i] for i in rest] == [by_block[0][i] for i in rest]
    moved = 0
    for k in by_lane[1]:
        a, b = by_lane[1][k], by_block[1][k]
        assert np.array_equal(a[rest].view(np.uint32), b[rest].view(np.uint32)), k
        moved += int((a[list(odd)] != b[list(odd)]).any())
    assert moved > 0


def test_dense_network_fused_or_tiled(ngpu, monkeypatch):
    n, k = 20000, 1000

    def run(env):
        for key, v in env.items():
            monkeypatch.setenv(key, v)
        try:
            ngpu.ResetKernel()
            ngpu.SetVerbosityLevel(0)
            ngpu.SetRandomSeed(4)
            nodes = ngpu.Create("aeif_cond_beta_multisynapse", n, 2)
            rng = np.random.default_rng(2)
            ngpu.SetStatus(nodes, "I_e", 1500.0)
            ngpu.SetStatus(nodes, "V_m", {"array": rng.uniform(-70.0, -52.0, n).tolist()})
            ngpu.Connect(nodes, nodes, {"rule": "fixed_indegree", "indegree": k},
                         {"weight": 0.01, "receptor": 1,
                          "delay": {"distribution": "normal_clipped", "mu": 1.0, "low": 0.1,
                                    "high": 2.0, "sigma": 0.5}})
            ngpu.ActivateRecSpikeTimes(nodes, 200)
            events = []
            for ms in (12.0, 6.0, 6.0):
                ngpu.Simulate(ms)
                events.append(ngpu.GetStepStats()["syn_events"])
            return (ngpu.GetRecSpikeTimes(nodes), np.array(ngpu.GetStatus(nodes, "V_m"), np.float32),
                    events)
        finally:
            for key in env:
                monkeypatch.delenv(key)
            ngpu.ResetKernel()

    ref = run({"NGPU_TILED": "0", "NGPU_FUSED_DELIVER": "0"})
    assert ref[2][0] / 120 > 100000      # dense enough for tiles in the second call
    for env in ({}, {"NGPU_TILED": "0"}, {"NGPU_TILED": "1"}):
        got = run(env)
        assert got[0] == ref[0], env
        np.testing.assert_array_equal(got[1], ref[1])
        assert got[2] == ref[2], env
