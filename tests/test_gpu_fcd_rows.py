"""FCD over window-FC rows: FP64 tiles of 32 rows with the edges in quarters, and the
FP32 rows z-scored in LDS or, when too long for it, from memory; against the FP64
Pearson correlation of the oracle's window FCs, hemispheres included."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("N,vols,ws,step", [
    (4, 20, 10, 6), (4, 40, 8, 1), (6, 41, 9, 1), (10, 75, 10, 1), (18, 76, 11, 1), (30, 140, 12, 1), (300, 40, 20, 8)])
def test_rows(oracle_mod, N, vols, ws, step, f64):
    print("case: fcd rows N", N, "vols", vols, "f64", f64, flush=True)
    B = 9
    rng = np.random.default_rng(3 * N + vols)
    common = rng.normal(size=(B, vols, 1))
    bold = rng.normal(size=(B, vols, N)) + rng.uniform(0.2, 1.5, size=(1, 1, N)) * common + 2.0
    if not f64:
        bold = bold.astype(np.float32).astype(np.float64)
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=(vols - 1) * 100, bold_tr=100, n_vols_remove=0,
                             window_size=ws, window_step=step, exc_interhemispheric=0, noise_period_ms=1,
                             precision=bnm.PREC_F64 if f64 else bnm.PREC_F32,
                             fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32, autotune=0)
    with bnm.Context(cfg) as c:
        c.set_empirical(rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 100))
        c.set_bold(bold)
        c.analyze()
        o = c.outputs(bold=False)
    # FP64: 1e-10 as for every FCD.  FP32: window FC to 1e-6 and z-scores to 2^-24;
    # rows of few edges (six at N = 4) can have a spread of 0.05, which makes 1e-6 into
    # 2e-5 a z-score and twice that a correlation, with a margin of two.
    tol = 1e-10 if f64 else 1e-4
    for b in range(B):
        np.testing.assert_allclose(o["fcd"][b], oracle_mod.fcd_tril(bold[b], step, ws, False), atol=tol, rtol=0)
