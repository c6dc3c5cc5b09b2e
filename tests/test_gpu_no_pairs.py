"""Two nodes without the pair between the hemispheres leave no pairs: window FC has no
columns, so no FCD kernel may read any, and every FCD value is the empty sum, 0."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fc", [bnm.FC_F64, bnm.FC_F32, bnm.FC_BF16X3], ids=str)
@pytest.mark.parametrize("direct", [0, 1])
def test_fcd_without_pairs(monkeypatch, fc, direct):
    print("case: no pairs, FC precision", fc, "direct", direct, flush=True)
    monkeypatch.setenv("BNM_FCD_DIRECT", str(direct))
    assert bnm.n_pairs(2, True) == 0
    cfg = bnm.default_config(nodes=2, n_sims=3, time_steps=2000, bold_tr=100, n_vols_remove=1, window_size=4,
                             window_step=2, exc_interhemispheric=1, noise_period_ms=1, fc_precision=fc)
    with bnm.Context(cfg) as c:
        c.set_empirical(np.zeros(0), np.linspace(-0.2, 1.0, 7))
        c.set_bold(np.random.default_rng(1).normal(size=(3, 21, 2)))
        c.analyze()
        o = c.outputs()
    assert o["fcd"].shape[1] > 1
    np.testing.assert_array_equal(o["fcd"], 0.0)
