"""The 16-simulation kernel against the split kernel, which steps the nodes with the same
FP32 update and adds the coupling up in another order: every node of two workgroups (the
second with one simulation), one to four nodes a lane.

Bounds, per TR of BOLD over 2.5 s.  FP32: the order changes a sum of up to 128 terms by a
few 1e-7 of itself at random from substep to substep, which leaves some 1e-7 of BOLD
(1.2e-7 between the dense FP32 kernels over 30 s); 2e-6.  BF16x3: operands carry 16 bits
(2^-17), those of the SC the same error all the time: 30 times 8e-6 / sqrt(terms) in an
input of about 5, some 1e-5 of BOLD; 1e-4.
"""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,bound", [(bnm.PREC_F32, 2e-6), (bnm.PREC_BF16X3, 1e-4)], ids=str)
@pytest.mark.parametrize("N", [2, 3, 7, 13, 16, 17, 33, 50, 64, 65, 81, 97, 100, 113, 125, 128])
def test_same_as_split(monkeypatch, N, prec, bound):
    T, B = 2500, 17
    print("case: mfma against split, N", N, "precision", prec, flush=True)
    rng = np.random.default_rng(300 + N)
    SC = W.synthetic_sc(N, 0.9 if N < 8 else 0.5, N)
    G = rng.uniform(0.5, 2.0, B)
    wEE, wEI = rng.uniform(0.1, 0.3, (B, N)), rng.uniform(0.1, 0.2, (B, N))
    noise = bnm.make_noise(N, (T + 1) * 20 * N)
    emp = rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40)
    out = []
    for name, p, kernel in (("split_f32", bnm.PREC_F32, bnm.KERNEL_FAST), ("mfma", prec, bnm.KERNEL_MFMA)):
        monkeypatch.setenv("BNM_FAST_LS", "1")
        monkeypatch.setenv("BNM_FAST_KS", "1")
        cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=100, n_vols_remove=2, window_size=6,
                                 window_step=3, exc_interhemispheric=0, noise_period_ms=T + 1, max_fic_trials=2,
                                 i_sampling_start=200, i_sampling_end=700, precision=p, kernel=kernel,
                                 fc_precision=bnm.FC_F32)
        with bnm.Context(cfg) as c:
            c.set_sc(SC)
            c.set_noise(noise)
            c.set_empirical(*emp)
            c.set_params(G, wEE, wEI)
            c.run()
            assert c.kernel_name().startswith(name)
            out.append(c.outputs())
    s, m = out
    np.testing.assert_array_equal(m["fic_trials"], s["fic_trials"])
    peak = np.abs(s["bold"]).max(axis=(1, 2))
    rel = np.abs(m["bold"] - s["bold"]).max(axis=(1, 2)) / peak
    print("per-TR BOLD rel", rel.max(), flush=True)
    assert (rel <= bound).all()
