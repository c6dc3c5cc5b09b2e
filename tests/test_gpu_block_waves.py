"""The row-blocked kernel's builds for more than 512 simulations of 65 to 128 nodes
(four waves a SIMD, part of the registers spilled) and those for no more than two or three
waves a SIMD (up to 64 nodes), at the smallest and largest node counts of each slice
length, with FIC restarts.

Bounds: FP32 strict within 1e-6 of the oracle per TR on runs of 2.5 s, the same FIC
trials, wIE to 1e-12; against the build for smaller populations twice that.
"""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu

T, TR, I_END = 2500, 100, 700


@pytest.mark.parametrize("N,B", [(n, 513) for n in (65, 80, 81, 100, 104, 105, 128)] +
                         [(33, 769), (48, 1024), (49, 769), (64, 1024), (33, 1281), (48, 1536), (49, 1281), (64, 1536),
                          (2, 1537), (32, 2048), (17, 2561), (32, 3072)])
def test_large_population_build(oracle_mod, N, B):
    print("case: block kernel, simulations", B, "N", N, flush=True)
    period = 900 if N % 2 else T + 1
    rng = np.random.default_rng(N)
    SC = W.synthetic_sc(N, 0.5, N)
    G = rng.uniform(0.02, 2.5, B)
    wEE, wEI = rng.uniform(0.1, 0.4, (B, N)), rng.uniform(0.1, 0.3, (B, N))
    noise = bnm.make_noise(N, period * 20 * N)
    emp = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40)
    out = {}
    below = 512 if N > 64 else 768 if N > 32 else 1024
    for n in (B, below):
        cfg = bnm.default_config(nodes=N, n_sims=n, time_steps=T, bold_tr=TR, n_vols_remove=2, no_fcd=1,
                                 exc_interhemispheric=0, noise_period_ms=period, max_fic_trials=2, i_sampling_start=200,
                                 i_sampling_end=I_END, precision=bnm.PREC_F32, kernel=bnm.KERNEL_FAST,
                                 fc_precision=bnm.FC_F32)
        with bnm.Context(cfg) as c:
            c.set_sc(SC)
            c.set_noise(noise)
            c.set_empirical(*emp)
            c.set_params(G[:n], wEE[:n], wEI[:n])
            c.run()
            assert c.kernel_name().startswith("block_f32")
            out[n] = c.outputs()
    g, small = out[B], out[below]
    np.testing.assert_array_equal(g["fic_trials"][:below], small["fic_trials"])
    assert g["fic_trials"].max() > 0
    peak = np.abs(g["bold"]).max(axis=(1, 2))
    assert (np.abs(g["bold"][:below] - small["bold"]).max(axis=(1, 2)) <= 2e-6 * peak[:below]).all()
    some = [0, 100, B - 1]
    r = oracle_mod.run_simulations(SC, G[some], wEE[some], wEI[some], noise_arr=noise, noise_period_ms=period,
                                   time_steps=T, bold_tr=TR, n_vols_remove=2, window_size=6, window_step=3,
                                   emp_fc=emp[0], emp_fcd=emp[1], no_fcd=True, max_fic_trials=2, i_start=200,
                                   i_end=I_END, exc=False)
    np.testing.assert_array_equal(g["fic_trials"][some], r["fic_trials"])
    np.testing.assert_allclose(g["wIE_fic"][some], r["wIE_fic"], rtol=0, atol=1e-12)
    for i, b in enumerate(some):
        rel = np.abs(g["bold"][b] - r["bold"][i]).max() / np.abs(r["bold"][i]).max()
        print("sim", b, "trials", r["fic_trials"][i], "per-TR BOLD rel", rel, flush=True)
        assert rel <= 1e-6
    scale = np.abs(r["ext"]).max(axis=(0, 2), keepdims=True)
    assert (np.abs(g["ext"][some] - r["ext"]) <= 1e-5 * scale).all()
