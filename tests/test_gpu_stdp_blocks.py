"""More simultaneous spikes than the blocks that take them: the linear rule of
test_gpu_stdp.py (arrivals 2 and 1 steps before, with, and 1 and 2 steps after
the target's spike) on c copies of its network, whose deliveries, arrivals and
post-synaptic updates share two launches (kernels.hip deliver_arrive_kernel,
fold_post_kernel; 128 blocks up to 2,048 nodes, then one per 16 nodes)."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c", [1, 129, 700])
def test_linear_rule_many_spikes(c):
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu as ngpu
    ngpu.ResetKernel()
    ngpu.SetVerbosityLevel(0)
    fact, offset, k, time_diff = 0.2, 0.03, 5, 10.0
    g = ngpu.CreateSynGroup("test_syn_model")
    ngpu.SetSynGroupParam(g, "fact", fact)
    ngpu.SetSynGroupParam(g, "offset", offset)
    n = k * c
    sg = ngpu.Create("spike_generator", n)
    neuron = ngpu.Create("aeif_cond_beta_multisynapse", 2 * n)
    ngpu.SetStatus(neuron, {"t_ref": 10.0})
    pre, post = neuron[0:n], neuron[n:2 * n]
    ngpu.SetStatus(sg, {"spike_times": [50.0], "spike_heights": [1.0]})
    one = {"rule": "one_to_one"}
    ngpu.Connect(sg, pre, one, {"weight": 17.9, "delay": 1.0, "receptor": 0, "synapse_group": 0})
    ngpu.Connect(sg, post, one, {"weight": 17.9, "delay": 1.0 + time_diff, "receptor": 0,
                                 "synapse_group": 0})
    dts = [0.1 * (-0.5 * (k - 1) + i) for i in range(k)]
    for i in range(k):
        ngpu.Connect(neuron[i * c:(i + 1) * c], neuron[n + i * c:n + (i + 1) * c], one,
                     {"weight": 0.0, "delay": time_diff - dts[i], "receptor": 0, "synapse_group": g})
    ngpu.Simulate(120.0)
    w = np.array(ngpu.GetStatus(ngpu.GetConnections(pre, post), "weight"), dtype=np.float64)
    expect = np.repeat([dt * fact + offset for dt in dts], c)
    np.testing.assert_allclose(w, expect, rtol=0, atol=1e-6)
