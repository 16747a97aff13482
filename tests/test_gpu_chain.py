"""The chain form of the RK5 update (one neuron over a group of lanes) and the
division by a double reciprocal against the lane-per-neuron kernel, which
divides with IEEE divisions and takes no part in either: rasters, state and
attempt counts are the same bits, for every model family and group width, for
uniform and per-neuron parameters, few and many hot neurons per wave, split
and unsplit steps, folds inside the launch and by a launch of their own, and
conductances that decay into the subnormal range."""
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


# model, ports, constant current, Poisson weight, recurrent weight
FAMILIES = [
    ("aeif_cond_beta_multisynapse", 1, 700.0, 0.3, 0.5),
    ("aeif_cond_beta_multisynapse", 2, 700.0, 0.3, 0.5),
    ("aeif_cond_beta_multisynapse", 3, 700.0, 0.3, 0.5),
    ("aeif_cond_beta_multisynapse", 7, 700.0, 0.3, 0.5),
    ("aeif_cond_beta_multisynapse", 8, 700.0, 0.3, 0.5),
    ("aeif_cond_alpha_multisynapse", 4, 700.0, 0.3, 0.5),
    ("aeif_cond_alpha", 2, 700.0, 0.3, 0.5),
    ("aeif_cond_beta", 2, 700.0, 0.3, 0.5),
    ("aeif_psc_exp", 2, 700.0, 60.0, 40.0),
    ("aeif_psc_alpha", 2, 700.0, 60.0, 40.0),
    ("aeif_psc_exp_multisynapse", 5, 700.0, 60.0, 40.0),
    ("aeif_psc_alpha_multisynapse", 3, 700.0, 60.0, 40.0),
    ("aeif_psc_delta", 2, 700.0, 0.4, 0.3),
    ("izhikevich_cond_beta", 1, 8.0, 0.01, 0.02),
    ("izhikevich_cond_beta", 2, 8.0, 0.01, 0.02),
]


def _run(ngpu, monkeypatch, env, model, ports, i_e, pw, rw, n, hetero):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        ngpu.SetRandomSeed(77)
        nodes = ngpu.Create(model, n, ports)
        ngpu.SetStatus(nodes, "I_e", i_e)
        rng = np.random.default_rng(3)
        if hetero:
            name, mean = ("a", 0.02) if "izh" in model else ("C_m", 281.0)
            ngpu.SetStatus(nodes, name, {"array": rng.uniform(0.8 * mean, 1.2 * mean, n).tolist()})
        else:
            # starting points apart, so that few neurons fire together
            ngpu.SetStatus(nodes, "V_m", {"array": rng.uniform(-70.0, -58.0, n).tolist()})
        pg = ngpu.Create("poisson_generator")
        ngpu.SetStatus(pg, {"rate": 8000.0, "stop": 30.0})
        ngpu.Connect(pg, nodes, {"rule": "all_to_all"}, {"weight": pw, "delay": 0.1, "receptor": 0})
        for p in range(ports - 1 if ports > 1 else 1):   # the last port stays silent
            ngpu.Connect(nodes, nodes, {"rule": "fixed_indegree", "indegree": min(5, n)},
                         {"weight": rw, "delay": 0.1 * (p + 1), "receptor": p})
        ngpu.ActivateRecSpikeTimes(nodes, 500)
        ngpu.Simulate(20.0)
        ngpu.Simulate(40.1)
        names = list(ngpu.GetScalVarNames(nodes[0])) + list(ngpu.GetPortVarNames(nodes[0]))
        state = {k: np.array(ngpu.GetStatus(nodes, k), np.float32) for k in names}
        return ngpu.GetRecSpikeTimes(nodes), state, ngpu.GetStepStats()
    finally:
        for k in env:
            monkeypatch.delenv(k)
        ngpu.ResetKernel()


def _same(a, b):
    assert a[0] == b[0]                      # every neuron's spike times
    for k in a[1]:
        assert np.array_equal(a[1][k].view(np.uint32), b[1][k].view(np.uint32)), k
    for k in ("attempts", "rejected", "substeps", "syn_events"):
        assert a[2][k] == b[2][k], k


@pytest.mark.parametrize("hetero", [False, True])
@pytest.mark.parametrize("model,ports,i_e,pw,rw", FAMILIES)
def test_chain_form_matches_lane_per_neuron(ngpu, monkeypatch, model, ports, i_e, pw, rw, hetero):
    args = (model, ports, i_e, pw, rw, 83, hetero)
    ref = _run(ngpu, monkeypatch, {"NGPU_RK5_PERSISTENT": "0"}, *args)
    assert sum(len(t) for t in ref[0]) > 40
    _same(_run(ngpu, monkeypatch, {}, *args), ref)
    _same(_run(ngpu, monkeypatch, {"NGPU_RK5_DEFER": "3", "NGPU_RK5_CHAIN_WAVES": "1"}, *args), ref)


@pytest.mark.parametrize("n", [1, 64, 1000])
@pytest.mark.parametrize("env", [{}, {"NGPU_RK5_DEFER": "0"}, {"NGPU_RK5_DEFER": "5"},
                                 {"NGPU_FOLD_IN_RK5": "0", "NGPU_RK5_DEFER": "4"},
                                 {"NGPU_RK5_CHAIN_WAVES": "2"}, {"NGPU_RK5_CHAIN_WAVES": "0"},
                                 {"NGPU_RK5_HOT_MARGIN": "-5"}])
def test_chain_form_schedules(ngpu, monkeypatch, n, env):
    # a margin of -5 Delta_T lists most neurons hot: more than the chain
    # waves hold, so the launch falls back to one lane per hot neuron
    args = ("aeif_cond_beta_multisynapse", 2, 700.0, 0.3, 0.5, n, False)
    ref = _run(ngpu, monkeypatch, {"NGPU_RK5_PERSISTENT": "0"}, *args)
    assert sum(len(t) for t in ref[0]) >= 1
    _same(_run(ngpu, monkeypatch, env, *args), ref)
