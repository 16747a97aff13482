"""Loss and gradient of the predictor's training kernels against the FP64
oracle at batch sizes around their partition: a sample alone, one short of
and one past a block's 64 samples, and block counts around the 128 rows that
the update kernel takes at once (rounding: inputs and weights on a grid that
bfloat16 holds exactly, so only FP32 sums differ from the oracle's; 64-term
sums of 64-term sums, a relative error of some 1e-6 of the largest term)."""
import numpy as np
import pytest

from conftest import gpu_available
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127 * 64, 128 * 64 + 1, 300 * 64 - 1])
def test_loss_grad_batch_edges(n):
    if not gpu_available():
        pytest.skip("no GPU")
    import nestgpu
    from test_gpu_predictor import NI, _random_params
    rng = np.random.default_rng(n)
    P = _random_params(rng, grid=True)
    nestgpu.SetPredictorParams(P.astype(np.float32))
    X = (rng.integers(-24, 25, (n, NI)) / 16.0).astype(np.float32)
    T = (O.mlp_forward(P, X, quant=1) + rng.normal(0, 1.0, n)).astype(np.float32)
    C = (rng.random(n) < 0.3).astype(np.uint8)
    loss, g = nestgpu.PredictorLossGrad(X, T, C)
    lref, gref = O.mlp_loss_grad(P, X, T, C, quant=1)
    assert abs(loss - lref) <= 1e-5 * max(lref, 1e-30)
    np.testing.assert_allclose(g, gref[16:], rtol=1e-4, atol=1e-5 * max(np.abs(gref).max(), 1e-30))
