"""The kernel with several workgroups per simulation (N > 256 in FP32, N > 128 in
FP64) against the FP64 oracle at the node counts where its layout can go wrong
(the last workgroup with one node or all of them, partly filled groups and
slices), with FIC restarts, and its fall-back to one workgroup per simulation.

Bounds: FP64 within 1e-9 of the oracle per TR, FP32 strict within 1e-6, the same
FIC trials, wIE to 1e-12.
"""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu

T, TR, I_END = 240, 20, 90


def _check(oracle_mod, prec, N, B, name, period=T + 1, graph=0):
    rng = np.random.default_rng(N)
    SC = W.synthetic_sc(N, 0.9, N)
    G = rng.uniform(0.5, 2.5, B)
    wEE = rng.uniform(0.1, 0.4, (B, N))
    wEI = rng.uniform(0.1, 0.3, (B, N))
    noise = bnm.make_noise(N, period * 20 * N)
    emp_fc = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False))
    emp_fcd = rng.uniform(-0.5, 1.0, 40)
    f64 = prec == bnm.PREC_F64
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=TR, n_vols_remove=2, no_fcd=1,
                             exc_interhemispheric=0, noise_period_ms=period, max_fic_trials=2, i_sampling_start=20,
                             i_sampling_end=I_END, precision=prec, kernel=bnm.KERNEL_AUTO, use_graph=graph,
                             fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32)
    r = oracle_mod.run_simulations(SC, G, wEE, wEI, noise_arr=noise, noise_period_ms=period, time_steps=T,
                                   bold_tr=TR, n_vols_remove=2, window_size=6, window_step=3, emp_fc=emp_fc,
                                   emp_fcd=emp_fcd, no_fcd=True, max_fic_trials=2, i_start=20, i_end=I_END, exc=False)
    with bnm.Context(cfg) as c:
        c.set_sc(SC)
        c.set_noise(noise)
        c.set_empirical(emp_fc, emp_fcd)
        c.set_params(G, wEE, wEI)
        for _ in range(3 if graph else 2):            # (the exchange words are used again)
            c.run()
            assert c.kernel_name().startswith(name)
            g = c.outputs()
            rel = max(np.abs(g["bold"][b] - r["bold"][b]).max() / np.abs(r["bold"][b]).max() for b in range(B))
            print("N", N, "trials", g["fic_trials"], r["fic_trials"], "per-TR BOLD rel", rel, flush=True)
            np.testing.assert_array_equal(g["fic_trials"], r["fic_trials"])
            np.testing.assert_array_equal(g["fic_failed"], r["fic_failed"])
            np.testing.assert_allclose(g["wIE_fic"], r["wIE_fic"], rtol=0, atol=1e-12)
            assert rel <= (1e-9 if f64 else 1e-6)
            scale = np.abs(r["ext"]).max(axis=(0, 2), keepdims=True)
            assert (np.abs(g["ext"] - r["ext"]) <= (1e-9 if f64 else 1e-5) * scale).all()


SIZES = [(bnm.PREC_F32, n, 3) for n in (257, 320, 321, 400, 449, 512)]
SIZES += [(bnm.PREC_F64, n, 3) for n in (129, 160, 193, 200, 256, 257, 320, 400, 512)]
SIZES += [(bnm.PREC_F32, 300, 1), (bnm.PREC_F32, 270, 41), (bnm.PREC_F64, 130, 17)]


@pytest.mark.parametrize("prec,N,B", SIZES, ids=lambda v: str(v))
def test_gang_kernel_matches_oracle(oracle_mod, prec, N, B, monkeypatch):
    print("case: gang kernel precision", prec, "N", N, "B", B, flush=True)
    monkeypatch.setenv("BNM_GANG", "1")
    _check(oracle_mod, prec, N, B, "gang_")


def test_gang_kernel_wrapped_noise_in_a_graph(oracle_mod, monkeypatch):
    monkeypatch.setenv("BNM_GANG", "1")
    _check(oracle_mod, bnm.PREC_F32, 290, 2, "gang_f32", period=70, graph=1)


@pytest.mark.parametrize("prec,N", [(bnm.PREC_F32, 280), (bnm.PREC_F64, 150)], ids=str)
def test_simulations_without_all_workgroups_run_on_one(oracle_mod, prec, N, monkeypatch):
    """With no time to wait no simulation finds its workgroups together; the
    launch that follows runs them all on one workgroup each.  (FP32: the first
    candidate here has the plain update, whose bound on runs this short is the
    same.)"""
    monkeypatch.setenv("BNM_GANG", "1")
    monkeypatch.setenv("BNM_GANG_POLLS", "-1")
    _check(oracle_mod, prec, N, 3, "gang_")


def test_gang_fic_converges(oracle_mod, monkeypatch):
    """Simulations whose FIC comes into band at different trials: the members of
    each agree on the millisecond at which the adjustment ends."""
    monkeypatch.setenv("BNM_GANG", "1")
    N, B, T_, period = 131, 4, 1300, 1301
    rng = np.random.default_rng(3)
    SC = W.synthetic_sc(N, 0.5, 3)
    G = np.array([0.02, 0.3, 0.6, 1.0])
    wEE, wEI = np.full((B, N), 0.21), np.full((B, N), 0.15)
    noise = bnm.make_noise(9, period * 20 * N)
    emp_fc = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False))
    kw = dict(time_steps=T_, bold_tr=100, n_vols_remove=2, max_fic_trials=12, noise_period_ms=period)
    r = oracle_mod.run_simulations(SC, G, wEE, wEI, noise_arr=noise, window_size=6, window_step=3, emp_fc=emp_fc,
                                   emp_fcd=np.zeros(4), no_fcd=True, i_start=400, i_end=1100, exc=False, **kw)
    cfg = bnm.default_config(nodes=N, n_sims=B, no_fcd=1, exc_interhemispheric=0, i_sampling_start=400,
                             i_sampling_end=1100, precision=bnm.PREC_F64, fc_precision=bnm.FC_F64, **kw)
    g = bnm.run_simulations(cfg, SC, G, wEE, wEI, noise=noise, emp_fc=emp_fc, emp_fcd=np.zeros(4))
    print("trials", g["fic_trials"], r["fic_trials"], "failed", g["fic_failed"], r["fic_failed"], flush=True)
    assert not r["fic_failed"].all() and r["fic_trials"].max() > r["fic_trials"].min()
    np.testing.assert_array_equal(g["fic_trials"], r["fic_trials"])
    np.testing.assert_array_equal(g["fic_failed"], r["fic_failed"])
    np.testing.assert_allclose(g["wIE_fic"], r["wIE_fic"], rtol=0, atol=1e-12)
    assert np.abs(g["bold"] - r["bold"]).max() <= 1e-9 * np.abs(r["bold"]).max()


@pytest.mark.parametrize("prec,N,B", [(bnm.PREC_F64, 400, 37), (bnm.PREC_F64, 140, 90), (bnm.PREC_F32, 500, 50)], ids=str)
def test_groups_take_one_simulation_after_the_other(monkeypatch, prec, N, B):
    """More simulations than groups of resident members, with FIC restarts that make
    them end at different times, against one workgroup per simulation."""
    f64 = prec == bnm.PREC_F64
    rng = np.random.default_rng(B)
    SC = W.synthetic_sc(N, 0.9, 1)
    noise = bnm.make_noise(1, 121 * 20 * N)
    emp = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40)
    params = rng.uniform(0.02, 1.5, B), rng.uniform(0.15, 0.25, (B, N)), rng.uniform(0.1, 0.2, (B, N))
    out = {}
    for gang in ("1", "0"):
        print("case: gang groups N", N, "B", B, "gang", gang, flush=True)
        monkeypatch.setenv("BNM_GANG", gang)
        cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=120, bold_tr=10, n_vols_remove=0, no_fcd=1,
                                 exc_interhemispheric=0, noise_period_ms=121, max_fic_trials=2, i_sampling_start=10,
                                 i_sampling_end=40, precision=prec, fc_precision=bnm.FC_F64)
        with bnm.Context(cfg) as c:
            c.set_sc(SC)
            c.set_noise(noise)
            c.set_empirical(*emp)
            c.set_params(*params)
            c.run()
            assert c.kernel_name().startswith("gang") == (gang == "1")
            out[gang] = c.outputs()
    g, r = out["1"], out["0"]
    np.testing.assert_array_equal(g["fic_trials"], r["fic_trials"])
    rel = np.abs(g["bold"] - r["bold"]).max() / np.abs(r["bold"]).max()
    assert rel <= (1e-9 if f64 else 1e-6)
