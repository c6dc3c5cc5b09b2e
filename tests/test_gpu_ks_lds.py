"""KS counts in LDS: the cost against the oracle's KS distance and Pearson cost of
the FC and FCD that the device itself returns, at the line between the two binning
kernels, with ties, values outside the empirical range, and NaN."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("m,N,B", [
    (1, 12, 2), (300, 12, 53), (1, 12, 54), (2, 12, 54), (300, 12, 54), (3000, 12, 300), (9, 140, 2)])
def test_cost(oracle_mod, m, N, B, f64):
    print("case: ks lds m", m, "N", N, "B", B, "f64", f64, flush=True)
    vols, ws = 60, 10                      # 50 windows, 1225 FCD values: 65536 in all from 54 simulations on
    rng = np.random.default_rng(m + N)
    bold = rng.normal(size=(B, vols, N)) + rng.uniform(0, 1.5, size=(1, 1, N)) * rng.normal(size=(B, vols, 1))
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=(vols - 1) * 100, bold_tr=100, n_vols_remove=0,
                             window_size=ws, window_step=1, exc_interhemispheric=0, noise_period_ms=1,
                             precision=bnm.PREC_F64 if f64 else bnm.PREC_F32,
                             fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32, autotune=0)
    emp_fc = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False))
    with bnm.Context(cfg) as c:
        c.set_empirical(emp_fc, rng.uniform(-0.1, 0.4, max(m, 2)))
        c.set_bold(bold)
        c.analyze()
        o = c.outputs(bold=False)
        # the last simulation's own FCD as part of the sample: ties
        emp_fcd = np.concatenate([o["fcd"][-1][: m // 2], rng.uniform(-0.1, 0.4, m - m // 2)])
        c.set_empirical(emp_fc, emp_fcd)
        bad = bold.copy()
        bad[0, :, 1] = bad[0, 0, 1]        # a node without variance: NaN
        c.set_bold(bad)
        c.analyze()
        o = c.outputs(bold=False)
    assert o["corr"][0] == cfg.max_cost
    for b in range(1, B):
        fc = o["fc"][b]
        # counts are whole numbers: only the FC's FP64 sums round
        want = 1 - np.corrcoef(emp_fc, fc)[0, 1] + abs(emp_fc.mean() - fc.mean()) + oracle_mod.ks(emp_fcd, o["fcd"][b])
        assert abs(o["corr"][b] - want) <= 1e-12, (b, o["corr"][b], want)
