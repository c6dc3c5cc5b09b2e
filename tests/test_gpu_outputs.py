"""Outputs through pinned memory on several threads: the same values as in one
simulation at a time, at sizes on both sides of the 2 MB line and with a last piece
that is not full."""
import threading

import numpy as np
import pytest

import bnm_cuda_amd as bnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("B", [3, 700, 2100])
def test_outputs_do_not_depend_on_their_size(B, f64):
    N, vols = 20, 67
    print("case: outputs B", B, "f64", f64, flush=True)
    rng = np.random.default_rng(B)
    bold = rng.normal(size=(B, vols, N)).astype(np.float32).astype(np.float64)

    def fetch(rows):
        cfg = bnm.default_config(nodes=N, n_sims=len(rows), time_steps=(vols - 1) * 100, bold_tr=100, n_vols_remove=0,
                                 window_size=10, window_step=1, exc_interhemispheric=0, noise_period_ms=1,
                                 precision=bnm.PREC_F64 if f64 else bnm.PREC_F32,
                                 fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32, autotune=0)
        with bnm.Context(cfg) as c:
            c.set_empirical(np.linspace(-0.2, 0.8, bnm.n_pairs(N, False)), np.linspace(-0.5, 1.0, 50))
            c.set_bold(bold[rows])
            c.analyze()
            out = []
            ts = [threading.Thread(target=lambda: out.append(c.outputs())) for _ in range(2)]
            for t in ts:
                t.start()
            for t in ts:
                t.join()
            for k in ("bold", "fc", "fcd", "ext"):
                np.testing.assert_array_equal(out[0][k], out[1][k])
            return out[0]

    o = fetch(np.arange(B))
    np.testing.assert_array_equal(o["bold"], bold)
    for b in (0, B // 2, B - 1):
        one = fetch(np.array([b]))
        for k in ("fc", "fcd"):
            np.testing.assert_array_equal(o[k][b], one[k][0])
    assert o["ext"].shape == (B, 6, N)
