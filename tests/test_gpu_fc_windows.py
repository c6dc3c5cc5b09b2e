"""Window FC formed in LDS: tile, row and window remainders, windows too long for
LDS, and both Gram precisions, against the CPU oracle's FC and FCD of the same
BOLD (the FCD is formed from every entry of every window FC)."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("N,vols,ws,step,exc", [
    (5, 40, 8, 1, 0), (16, 40, 9, 2, 1), (17, 33, 14, 1, 0), (31, 50, 30, 1, 0), (32, 36, 16, 3, 0),
    (33, 60, 20, 1, 0), (64, 101, 29, 2, 1), (100, 160, 30, 5, 0), (129, 70, 43, 2, 0), (400, 60, 44, 4, 1),
    (400, 120, 104, 8, 0)])
def test_windows_against_oracle(oracle_mod, N, vols, ws, step, exc, f64):
    print("case: fc windows N", N, "vols", vols, "ws", ws, "f64", f64, flush=True)
    B = 2
    rng = np.random.default_rng(N + ws)
    common = rng.normal(size=(B, vols, 1))
    bold = rng.normal(size=(B, vols, N)) + rng.uniform(0, 1.5, size=(1, 1, N)) * common + 3.0
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=(vols - 1) * 100, bold_tr=100, n_vols_remove=0,
                             window_size=ws, window_step=step, exc_interhemispheric=exc, noise_period_ms=1,
                             precision=bnm.PREC_F64 if f64 else bnm.PREC_F32,
                             fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32, autotune=0)
    if not f64:
        bold = bold.astype(np.float32).astype(np.float64)
    with bnm.Context(cfg) as c:
        c.set_empirical(rng.uniform(-0.2, 0.8, bnm.n_pairs(N, bool(exc))), rng.uniform(-0.5, 1.0, 500))
        c.set_bold(bold)
        c.analyze()
        o = c.outputs(bold=False)
    # FP64: the products are exact to 2^-53 and summed over up to 120 volumes / 80000
    # edges.  FP32: z-scores and products to 2^-24, sums of up to 80000 terms of
    # z-scores below ten: window FC to 1e-6 each, which the FCD's second z-scoring
    # (window FC values of spread above 0.1) passes on tenfold.
    tfc, tfcd = (1e-11, 1e-10) if f64 else (5e-6, 2e-5)
    for b in range(B):
        np.testing.assert_allclose(o["fc"][b], oracle_mod.fc_tril(bold[b], bool(exc)), atol=tfc, rtol=0)
        np.testing.assert_allclose(o["fcd"][b], oracle_mod.fcd_tril(bold[b], step, ws, bool(exc)), atol=tfcd, rtol=0)
