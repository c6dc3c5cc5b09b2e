"""Row-block MLP path (layers up to 256 wide): row and width remainders, the
two-tile row blocks, and the networks just beyond its limits."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("shape", [
    (1, 1, 1, 1, 1), (5, 16, 1, 1, 15), (5, 17, 2, 3, 17), (33, 64, 2, 16, 31), (4, 256, 15, 1, 40),
    (256, 256, 1, 256, 65), (200, 130, 3, 40, 511), (5, 64, 2, 1, 1000), (5, 64, 2, 1, 2048), (5, 64, 2, 1, 2049), (6, 200, 2, 1, 8192), (5, 48, 2, 1, 8209),
    (5, 257, 2, 1, 70), (257, 32, 2, 1, 70), (4, 32, 16, 1, 70)])
def test_gradient_and_prediction(bf16, shape):
    in_dim, hid, depth, out_dim, n = shape
    print("case: mlp rows", shape, "bf16", bf16, flush=True)
    rng = np.random.default_rng(7)
    X = rng.normal(size=(n, in_dim)).astype(np.float32)
    T = rng.normal(size=(n, out_dim)).astype(np.float32)
    with bnm.MLP(in_dim, hid, depth, out_dim, bf16=bf16, seed=3) as net:
        p, ds = net.get_params(), net.dims()
        Y = net.predict(X)
        loss, g = net.loss_grad(X, T)
        loss2, g2 = net.loss_grad(X[:(n + 1) // 2], T[:(n + 1) // 2])
    # FP32 sums against FP64: 1e-4 / 1e-3 in norm.  With BF16 operands an operand
    # near a rounding boundary moves by 2^-8; 16 layers add such moves up, each
    # passed on with a factor of about one: 2^-8 sqrt(depth + 1) for results and
    # twice that (there and back) for gradients, with the margin of 3 for the norm.
    r = 3 * 2.0 ** -8 * np.sqrt(depth + 1)
    ty, tg = (r, 2 * r) if bf16 else (1e-4, 1e-3)
    Yo, _ = M.forward(p, ds, X, bf16)
    assert np.linalg.norm(Y - Yo) <= ty * max(1.0, np.linalg.norm(Yo))
    for rows, l, gr in ((n, loss, g), ((n + 1) // 2, loss2, g2)):
        lo, go = M.loss_grad(p, ds, X[:rows], T[:rows], bf16)
        assert abs(l - lo) <= 2 * ty * lo + 1e-7
        assert np.linalg.norm(gr - go) <= tg * np.linalg.norm(go) + 1e-7


def test_second_data_set_and_set_params():
    print("case: mlp data set of another size, parameters set between", flush=True)
    rng = np.random.default_rng(1)
    X = rng.normal(size=(300, 4)).astype(np.float32)
    T = X[:, :1] * 0.5
    with bnm.MLP(4, 32, 2, 1, bf16=True, seed=1) as a, bnm.MLP(4, 32, 2, 1, bf16=True, seed=2) as b:
        a.fit(X, T, epochs=1, batch=100, lr=1e-3, seed=0)
        a.fit(X[:150], T[:150], epochs=1, batch=50, lr=1e-3, seed=0)
        b.set_params(a.get_params())
        assert np.array_equal(a.predict(X), b.predict(X))
