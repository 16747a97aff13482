"""Steps with few spikes under the dense (tiled) delivery are delivered by
global atomics instead (NGPU_TILE_SPARSE: the limit in events): the same
rasters and state as the delivery launch without tiles, for networks whose
steps all take one form, and for limits that the steps cross back and forth
(a tile plan then outlives the steps between)."""
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


def _run(ngpu, monkeypatch, env, model):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        ngpu.ResetKernel()
        ngpu.SetVerbosityLevel(0)
        ngpu.SetRandomSeed(5)
        n, k = 301, 90
        iaf = model == "iaf_psc_exp"
        pops = [ngpu.Create(model, n, 2)] + ([ngpu.Create(model, 40, 2)] if iaf else [])
        st = {} if iaf else {"E_rev": [0.0, -85.0], "tau_rise": [1.0, 1.0], "tau_decay": [1.0, 1.0]}
        for p in pops:
            if st:
                ngpu.SetStatus(p, st)
            pg = ngpu.Create("poisson_generator")
            ngpu.SetStatus(pg, "rate", 8000.0 if iaf else 20000.0)
            ngpu.Connect(pg, p, {"rule": "all_to_all"},
                         {"weight": 60.0 if iaf else 0.24, "delay": 0.1, "receptor": 0})
            ngpu.Connect(pops[0], p, {"rule": "fixed_indegree", "indegree": k},
                         {"weight": 12.0 if iaf else 0.2, "receptor": 0,
                          "delay": {"distribution": "normal_clipped", "mu": 1.0, "low": 0.1,
                                    "high": 3.0, "sigma": 0.7}})
            ngpu.ActivateRecSpikeTimes(p, 1000)
        ngpu.Simulate(15.0)
        ngpu.Simulate(35.0)
        cfg = ngpu.GetBatchConfig()
        assert cfg["tiled"] == (1 if env["NGPU_TILED"] == "1" else 0)
        return ([ngpu.GetRecSpikeTimes(p) for p in pops],
                [np.array(ngpu.GetStatus(p, "V_m_rel" if iaf else "V_m")) for p in pops],
                ngpu.GetStepStats())
    finally:
        for k in env:
            monkeypatch.delenv(k)
        ngpu.ResetKernel()


@pytest.mark.parametrize("model", ["iaf_psc_exp", "aeif_cond_beta_multisynapse"])
def test_sparse_steps_match_delivery_launch(ngpu, monkeypatch, model):
    ref = _run(ngpu, monkeypatch, {"NGPU_TILED": "0"}, model)
    assert sum(len(t) for p in ref[0] for t in p) > 300
    for limit in ("0", "100", "500", "1000000000"):
        got = _run(ngpu, monkeypatch, {"NGPU_TILED": "1", "NGPU_TILE_SPARSE": limit}, model)
        assert got[0] == ref[0], limit
        for a, b in zip(got[1], ref[1]):
            np.testing.assert_array_equal(a, b)
        for key in ("syn_events", "spikes", "dropped_spikes"):
            assert got[2][key] == ref[2][key], (limit, key)
