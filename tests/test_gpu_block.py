"""The row-blocked integration kernel against the FP64 oracle at the sizes where
its layout can go wrong: a partly filled wave (32 nodes), group (4 nodes) or
k-slice, one node more than a slice length holds, the largest of each element
type, and noise arrays that wrap within and after one millisecond.

Bounds: FP64 within 1e-9 of the oracle per TR (rounding differs by a few ulp a
step), FP32 strict within 1e-6 (its bound on runs this short), the same FIC
trials, wIE to 1e-12.
"""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu

T, TR, I_END, B = 2500, 100, 700, 3


def _case(N, period, seed):
    rng = np.random.default_rng(seed)
    SC = W.synthetic_sc(N, 0.9 if N < 8 else 0.5, seed)
    G = rng.uniform(0.5, 2.5, B)
    wEE = rng.uniform(0.1, 0.4, (B, N))
    wEI = rng.uniform(0.1, 0.3, (B, N))
    noise = bnm.make_noise(seed, period * 20 * N)
    emp_fc = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False))
    emp_fcd = rng.uniform(-0.5, 1.0, 40)
    return SC, G, wEE, wEI, noise, emp_fc, emp_fcd


SIZES = [(bnm.PREC_F64, n) for n in (2, 31, 33, 48, 65, 100, 104, 105, 128)]
SIZES += [(bnm.PREC_F32, n) for n in (2, 32, 49, 64, 81, 100, 127, 129, 160, 161, 200, 224, 225, 256)]


@pytest.mark.parametrize("prec,N", SIZES, ids=lambda v: str(v))
@pytest.mark.parametrize("period", [T + 1, 900])
def test_block_kernel_matches_oracle(oracle_mod, prec, N, period):
    print("case: block kernel precision", prec, "N", N, "noise period", period, flush=True)
    _check(oracle_mod, prec, N, period)


def test_block_kernel_one_millisecond_of_noise(oracle_mod):
    _check(oracle_mod, bnm.PREC_F64, 20, 1)


def _check(oracle_mod, prec, N, period):
    SC, G, wEE, wEI, noise, emp_fc, emp_fcd = _case(N, period, 100 + N)
    f64 = prec == bnm.PREC_F64
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=TR, n_vols_remove=2, window_size=6,
                             window_step=3, exc_interhemispheric=0, noise_period_ms=period, max_fic_trials=2,
                             i_sampling_start=200, i_sampling_end=I_END, precision=prec,
                             kernel=bnm.KERNEL_FAST, fc_precision=bnm.FC_F64 if f64 else bnm.FC_F32)
    with bnm.Context(cfg) as c:
        c.set_sc(SC)
        c.set_noise(noise)
        c.set_empirical(emp_fc, emp_fcd)
        c.set_params(G, wEE, wEI)
        c.run()
        assert c.kernel_name().startswith("block_f64" if f64 else "block_f32")
        g = c.outputs()
    r = oracle_mod.run_simulations(SC, G, wEE, wEI, noise_arr=noise, noise_period_ms=period, time_steps=T,
                                   bold_tr=TR, n_vols_remove=2, window_size=6, window_step=3, emp_fc=emp_fc,
                                   emp_fcd=emp_fcd, max_fic_trials=2, i_start=200, i_end=I_END, exc=False)
    rel = max(np.abs(g["bold"][b] - r["bold"][b]).max() / np.abs(r["bold"][b]).max() for b in range(B))
    print("trials", g["fic_trials"], r["fic_trials"], "per-TR BOLD rel", rel, flush=True)
    np.testing.assert_array_equal(g["fic_trials"], r["fic_trials"])
    np.testing.assert_array_equal(g["fic_failed"], r["fic_failed"])
    np.testing.assert_allclose(g["wIE_fic"], r["wIE_fic"], rtol=0, atol=1e-12)
    assert rel <= (1e-9 if f64 else 1e-6)
    scale = np.abs(r["ext"]).max(axis=(0, 2), keepdims=True)
    assert (np.abs(g["ext"] - r["ext"]) <= (1e-9 if f64 else 1e-5) * scale).all()


def test_no_fcd_with_many_windows():
    """no_fcd leaves the configuration's windows out: a context whose window
    settings give hundreds of them keeps no window tables, and FC and cost are
    those of the same run without a window that fits."""
    N, prec = 12, bnm.PREC_F64
    SC, G, wEE, wEI, noise, emp_fc, emp_fcd = _case(N, T + 1, 5)
    out = []
    for window, step in ((4, 1), (4000, 1)):
        cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=5, n_vols_remove=2, window_size=window,
                                 window_step=step, exc_interhemispheric=0, noise_period_ms=T + 1, adjust_fic=0,
                                 no_fcd=1, precision=prec, kernel=bnm.KERNEL_FAST)
        out.append(bnm.run_simulations(cfg, SC, G, wEE, wEI, noise=noise, emp_fc=emp_fc, emp_fcd=emp_fcd))
    np.testing.assert_array_equal(out[0]["fc"], out[1]["fc"])
    np.testing.assert_array_equal(out[0]["corr"], out[1]["corr"])
