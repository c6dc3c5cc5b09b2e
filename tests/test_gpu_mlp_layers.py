"""Networks that go through the row blocks or layer by layer by the number of rows: the
same bits on both sides of the rule, and training layer by layer leaves the row blocks'
copies of the weights up to date."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("shape", [(5, 8, 1, 1), (5, 32, 4, 1), (7, 64, 2, 3), (5, 128, 2, 1), (40, 20, 3, 9)])
def test_prediction_is_the_same_by_rows_and_by_layers(bf16, shape):
    print("case: mlp prediction by layers", shape, "bf16", bf16, flush=True)
    n, some = 70001, 1500
    X = np.random.default_rng(2).normal(size=(n, shape[0])).astype(np.float32)
    with bnm.MLP(*shape, bf16=bf16, seed=3) as net:
        Y = net.predict(X)
        for s in (0, 30000, 65536 - 700, n - some):
            np.testing.assert_array_equal(Y[s:s + some], net.predict(X[s:s + some]))


@pytest.mark.parametrize("bf16", [False, True])
def test_gradient_and_training_of_many_rows(bf16):
    """330000 rows through one hidden layer of 8 nodes: the gradient against the FP64 oracle
    (sums in FP32: 1e-3 in norm; BF16 operands near a rounding boundary move by 2^-8,
    three times 2^-8 sqrt 2, there and back), and predictions of few rows after training
    with such batches against those of an object that was given the parameters."""
    print("case: mlp gradient by layers, bf16", bf16, flush=True)
    n = 330000
    rng = np.random.default_rng(4)
    X = rng.normal(size=(n, 5)).astype(np.float32)
    T = np.tanh(X[:, :1] * X[:, 1:2])
    with bnm.MLP(5, 8, 1, 1, bf16=bf16, seed=3) as net, bnm.MLP(5, 8, 1, 1, bf16=bf16, seed=9) as other:
        p, ds = net.get_params(), net.dims()
        loss, g = net.loss_grad(X, T)
        lo, go = M.loss_grad(p, ds, X, T, bf16)
        r = 3 * 2.0 ** -8 * np.sqrt(2)
        ty, tg = (r, 2 * r) if bf16 else (1e-4, 1e-3)
        assert abs(loss - lo) <= 2 * ty * lo + 1e-7
        assert np.linalg.norm(g - go) <= tg * np.linalg.norm(go) + 1e-7
        net.fit(X, T, epochs=2, batch=n, lr=1e-2, seed=1)
        assert np.abs(net.get_params() - p).max() > 1e-3
        other.set_params(net.get_params())
        np.testing.assert_array_equal(net.predict(X[:100]), other.predict(X[:100]))
