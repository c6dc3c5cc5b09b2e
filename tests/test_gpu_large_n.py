"""Beyond 512 nodes the tuner times the streaming kernels beside the hybrid ones."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_streaming_kernels_are_timed():
    N, B, T = 520, 2, 5
    print("case: tuner beyond 512 nodes", flush=True)
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=1, n_vols_remove=0, no_fcd=1,
                             noise_period_ms=T + 1, adjust_fic=0, precision=bnm.PREC_F32)
    with bnm.Context(cfg) as c:
        c.set_sc(W.synthetic_sc(N, 0.5, 1))
        c.set_noise(bnm.make_noise(1, (T + 1) * 20 * N))
        n = bnm.n_pairs(N, True)
        c.set_empirical(np.linspace(-0.2, 0.8, n), np.linspace(-0.5, 1.0, 40))
        c.set_params(np.full(B, 1.0), np.full((B, N), 0.2), np.full((B, N), 0.2))
        c.run()
        log = c.tune_log()
    print(log, flush=True)
    assert "stream_f32" in log and "hyb_f32" in log
