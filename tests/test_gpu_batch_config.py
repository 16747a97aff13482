"""The batch launch's configuration: what SetBatchConfig leaves out is the
engine's default, every default can be set again after another value, and the
autotuner leaves the choice of delivery to the engine where it was."""
import pytest

from conftest import gpu_available
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
