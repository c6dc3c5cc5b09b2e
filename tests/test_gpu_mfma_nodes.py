"""The 16-simulation kernel's deal of nodes to waves against the FP64 oracle: one to
four nodes a lane, waves without nodes, a last quad that is not full, both wave
counts, noise that wraps, and FIC restarts (which start the noise again).

Bounds: the FP32 kernels agree with each other within 1e-3 per TR of BOLD on runs of
this length (different orders of the sum over nodes), and with the same FIC trials."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [bnm.PREC_F32, bnm.PREC_BF16X3])
@pytest.mark.parametrize("N,period", [
    (2, 900), (3, 2501), (13, 900), (16, 2501), (17, 1), (33, 900), (50, 2501), (64, 900), (65, 2501), (81, 900),
    (97, 2501), (100, 900), (113, 2501), (125, 900), (128, 2501)])
def test_nodes(oracle_mod, N, period, prec):
    T, B = 2500, 3
    print("case: mfma nodes N", N, "period", period, "precision", prec, flush=True)
    rng = np.random.default_rng(200 + N)
    SC = W.synthetic_sc(N, 0.9 if N < 8 else 0.5, N)
    G = rng.uniform(0.5, 2.0, B)
    wEE, wEI = rng.uniform(0.1, 0.3, (B, N)), rng.uniform(0.1, 0.2, (B, N))
    noise = bnm.make_noise(N, period * 20 * N)
    emp = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40)
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=100, n_vols_remove=2, window_size=6,
                             window_step=3, exc_interhemispheric=0, noise_period_ms=period, max_fic_trials=2,
                             i_sampling_start=200, i_sampling_end=700, precision=prec, kernel=bnm.KERNEL_MFMA,
                             fc_precision=bnm.FC_F32)
    with bnm.Context(cfg) as c:
        c.set_sc(SC)
        c.set_noise(noise)
        c.set_empirical(*emp)
        c.set_params(G, wEE, wEI)
        c.run()
        assert "mfma" in c.kernel_name()
        g = c.outputs()
    r = oracle_mod.run_simulations(SC, G, wEE, wEI, noise_arr=noise, noise_period_ms=period, time_steps=T,
                                   bold_tr=100, n_vols_remove=2, window_size=6, window_step=3, emp_fc=emp[0],
                                   emp_fcd=emp[1], max_fic_trials=2, i_start=200, i_end=700, exc=False)
    rel = max(np.abs(g["bold"][b] - r["bold"][b]).max() / np.abs(r["bold"][b]).max() for b in range(B))
    print("trials", g["fic_trials"], r["fic_trials"], "per-TR BOLD rel", rel, flush=True)
    np.testing.assert_array_equal(g["fic_trials"], r["fic_trials"])
    assert rel <= 1e-3
