"""Large FP32 populations of up to 16 nodes: the tuner times the strict E/I kernel beside
the row-blocked one, and whichever it takes keeps the strict FP32 bound (1e-6 of the
oracle per TR of BOLD on runs of 2.5 s, the same FIC trials)."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,B,offered", [(2, 1025, True), (16, 1025, True), (16, 1024, False), (17, 1100, False)])
def test_tuned_kernel_for_few_nodes(oracle_mod, N, B, offered):
    print("case: tuned kernel, N", N, "simulations", B, flush=True)
    rng = np.random.default_rng(N)
    SC = W.synthetic_sc(N, 0.9, N)
    G, wEE, wEI = rng.uniform(0.5, 2.5, B), rng.uniform(0.1, 0.4, (B, N)), rng.uniform(0.1, 0.3, (B, N))
    kw = dict(time_steps=2500, bold_tr=100, n_vols_remove=2, max_fic_trials=2, noise_period_ms=2501)
    noise = bnm.make_noise(N, 2501 * 20 * N)
    emp = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40)
    cfg = bnm.default_config(nodes=N, n_sims=B, no_fcd=1, exc_interhemispheric=0, i_sampling_start=200,
                             i_sampling_end=700, precision=bnm.PREC_F32, fc_precision=bnm.FC_F32, **kw)
    with bnm.Context(cfg) as c:
        c.set_sc(SC)
        c.set_noise(noise)
        c.set_empirical(*emp)
        c.set_params(G, wEE, wEI)
        c.run()
        print(c.tune_log(), flush=True)
        assert ("split_ei_f32" in c.tune_log()) == offered and "block_f32" in c.tune_log()
        strict = "strict" in c.kernel_name()
        g = c.outputs()
    some = [0, B // 2, B - 1]
    r = oracle_mod.run_simulations(SC, G[some], wEE[some], wEI[some], noise_arr=noise, window_size=6, window_step=3,
                                   emp_fc=emp[0], emp_fcd=emp[1], no_fcd=True, i_start=200, i_end=700, exc=False, **kw)
    if strict:
        np.testing.assert_array_equal(g["fic_trials"][some], r["fic_trials"])
        for i, b in enumerate(some):
            assert np.abs(g["bold"][b] - r["bold"][i]).max() <= 1e-6 * np.abs(r["bold"][i]).max()
