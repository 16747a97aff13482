"""The persistent RK5 kernels of models with many ports (refills that fold the
ports in a loop, chain waves with a tableau of their own) against the
lane-per-neuron kernel with its fold launch: the same bits on both sides of
the port counts where their form changes, split and unsplit steps, Poisson
input kept as a run and per edge."""
import numpy as np
import pytest

from conftest import gpu_available
from test_gpu_chain import _same

pytestmark = pytest.mark.gpu

# model, ports, constant current, Poisson weight, recurrent weight
CASES = [
    ("aeif_cond_beta_multisynapse", 6, 700.0, 0.3, 0.2),
    ("aeif_cond_beta_multisynapse", 9, 700.0, 0.3, 0.2),
    ("aeif_cond_beta_multisynapse", 20, 700.0, 0.3, 0.2),
    ("aeif_cond_alpha_multisynapse", 8, 700.0, 0.3, 0.2),
    ("aeif_psc_alpha_multisynapse", 10, 700.0, 60.0, 20.0),
    ("aeif_psc_exp_multisynapse", 12, 700.0, 60.0, 20.0),
    ("aeif_psc_exp_multisynapse", 13, 700.0, 60.0, 20.0),
    ("aeif_psc_exp_multisynapse", 17, 700.0, 60.0, 20.0),
    ("izhikevich_cond_beta", 9, 8.0, 0.01, 0.01),
]


def _run(ngpu, monkeypatch, env, model, ports, i_e, pw, rw, hetero):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        ngpu.SetRandomSeed(77)
        n = 150
        nodes = ngpu.Create(model, n, ports)
        ngpu.SetStatus(nodes, "I_e", i_e)
        if "cond" in model:
            ngpu.SetStatus(nodes, "E_rev", [0.0 if p % 2 == 0 else -85.0 for p in range(ports)])
        rng = np.random.default_rng(3)
        ngpu.SetStatus(nodes, "V_m", {"array": rng.uniform(-70.0, -58.0, n).tolist()})
        if hetero:
            name, mean = ("a", 0.02) if "izh" in model else ("C_m", 281.0)
            ngpu.SetStatus(nodes, name, {"array": rng.uniform(0.8 * mean, 1.2 * mean, n).tolist()})
        pg = ngpu.Create("poisson_generator")
        ngpu.SetStatus(pg, {"rate": 8000.0, "stop": 20.0})
        ngpu.Connect(pg, nodes, {"rule": "all_to_all"},
                     {"weight": pw, "delay": 0.1, "receptor": (ports - 1) // 2 * 2})
        for p in range(ports):
            ngpu.Connect(nodes, nodes, {"rule": "fixed_indegree", "indegree": 3},
                         {"weight": rw, "delay": 0.1 * (p % 4 + 1), "receptor": p})
        ngpu.ActivateRecSpikeTimes(nodes, 500)
        ngpu.Simulate(15.0)
        ngpu.Simulate(20.1)
        names = list(ngpu.GetScalVarNames(nodes[0])) + list(ngpu.GetPortVarNames(nodes[0]))
        state = {k: np.array(ngpu.GetStatus(nodes, k), np.float32) for k in names}
        return ngpu.GetRecSpikeTimes(nodes), state, ngpu.GetStepStats()
    finally:
        for k in env:
            monkeypatch.delenv(k)
        ngpu.ResetKernel()


@pytest.mark.parametrize("hetero", [False, True])
@pytest.mark.parametrize("model,ports,i_e,pw,rw", CASES)
def test_many_ports_match_lane_per_neuron(monkeypatch, model, ports, i_e, pw, rw, hetero):
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu as ngpu
    args = (model, ports, i_e, pw, rw, hetero)
    ref = _run(ngpu, monkeypatch, {"NGPU_RK5_PERSISTENT": "0"}, *args)
    assert sum(len(t) for t in ref[0]) > 40 and ref[2]["dropped_spikes"] == 0
    for env in ({}, {"NGPU_RK5_DEFER": "3"}, {"NGPU_POISSON_RUNS": "0", "NGPU_RK5_DEFER": "3"}):
        _same(_run(ngpu, monkeypatch, env, *args), ref)
