"""The form of delivery of a dense network (fused into the next launch, or
tiled) follows its activity from one stretch of steps to the next, inside a
Simulate call as well as between calls, and counts the events of the sources
that fire rather than of the mean source.  Whatever it takes, rasters, state
and counters are those of one fixed form."""
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


def _run(ngpu, monkeypatch, env, build, calls):
    """calls: (constant current of the first population, ms); the form after each."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        ngpu.SetRandomSeed(5)
        pops = build(ngpu)
        for p, _ in pops:
            ngpu.ActivateRecSpikeTimes(p, 1000)
        forms = []
        for i_e, ms in calls:
            if i_e is not None:
                ngpu.SetStatus(pops[0][0], "I_e", i_e)
            ngpu.Simulate(ms)
            forms.append(ngpu.GetBatchConfig()["tiled"])
        st = ngpu.GetStepStats()
        return ([ngpu.GetRecSpikeTimes(p) for p, _ in pops],
                [np.array(ngpu.GetStatus(p, v), np.float32) for p, v in pops],
                [st[k] for k in ("syn_events", "spikes", "dropped_spikes")], forms)
    finally:
        for k in env:
            monkeypatch.delenv(k)
        ngpu.ResetKernel()


def _same(a, b):
    assert a[0] == b[0]
    for x, y in zip(a[1], b[1]):
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))
    assert a[2] == b[2]


def _delay(high):
    return {"distribution": "normal_clipped", "mu": 0.3, "low": 0.1, "high": high, "sigma": 0.1}


def _one(ngpu):
    n = 301
    p = ngpu.Create("aeif_cond_beta_multisynapse", n, 2)
    ngpu.SetStatus(p, {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [1.0, 1.0]})
    ngpu.SetStatus(p, "V_m", {"array": np.linspace(-70.0, -56.0, n).tolist()})
    ngpu.Connect(p, p, {"rule": "fixed_indegree", "indegree": 90},
                 {"weight": 0.01, "receptor": 0, "delay": _delay(0.5)})
    return [(p, "V_m")]


def _batch(ngpu):
    (p, v), = _one(ngpu)
    q = ngpu.Create("iaf_psc_exp", 40, 2)
    ngpu.Connect(p, q, {"rule": "fixed_indegree", "indegree": 90},
                 {"weight": 5.0, "receptor": 0, "delay": _delay(0.5)})
    return [(p, v), (q, "V_m_rel")]


# (quiet, driven, quiet) calls: every change falls inside a call, since a
# call begins with the form of the one before
CALLS = ((0.0, 30.0), (3000.0, 40.0), (0.0, 40.0), (3000.0, 0.1), (None, 20.0))


@pytest.mark.parametrize("defer", [None, "3"])
@pytest.mark.parametrize("build", [_one, _batch])
def test_form_follows_activity(ngpu, monkeypatch, build, defer):
    # a low cap on attempts splits most spiking steps, so spikes that count
    # for the step before are in the list when the form changes
    extra = {"NGPU_RK5_DEFER": defer} if defer else {}
    ref = _run(ngpu, monkeypatch, {"NGPU_TILED": "0", "NGPU_BATCH": "0", "NGPU_FUSED_DELIVER": "0",
                                   **extra}, build, CALLS)
    assert sum(len(t) for p in ref[0] for t in p) > 300
    got = _run(ngpu, monkeypatch, {"NGPU_FUSED_EVENTS": "100", "NGPU_TILE_SPARSE": "300", **extra},
               build, CALLS)
    _same(got, ref)
    assert got[3] == [0, 1, 0, 0, 1]


def _hubs(ngpu):
    # two neurons that hold three quarters of the synapses
    n = 301
    p = ngpu.Create("aeif_cond_beta_multisynapse", n, 2)
    ngpu.SetStatus(p, {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [1.0, 1.0]})
    hubs = p[0:2]
    for src, k in ((hubs, 2), (p, 20)):
        for _ in range(30 if k == 2 else 1):
            ngpu.Connect(src, p, {"rule": "fixed_indegree", "indegree": k},
                         {"weight": 0.001, "receptor": 1, "delay": _delay(0.5)})
    ngpu.SetStatus(hubs, "I_e", 3000.0)
    return [(p, "V_m")]


def test_form_counts_the_hubs(ngpu, monkeypatch):
    # ~0.04 spikes a step: 300 events a step, 3 by the mean out-degree (80)
    calls = ((None, 40.0), (None, 40.0))
    ref = _run(ngpu, monkeypatch, {"NGPU_TILED": "0", "NGPU_FUSED_DELIVER": "0"}, _hubs, calls)
    n_spk = [len(t) for t in ref[0][0]]
    assert sum(n_spk[:2]) >= 8 and sum(n_spk[2:]) == 0
    got = _run(ngpu, monkeypatch, {"NGPU_FUSED_EVENTS": "50"}, _hubs, calls)
    _same(got, ref)
    assert got[3] == [1, 1]
