"""Simulations that the multi-workgroup kernel did not run, because their workgroups
did not meet, and that one workgroup each ran instead: the same bits as those of the
multi-workgroup kernel, whichever simulations they are, and the others untouched.

BNM_GANG_MARK=n marks every n-th simulation before any workgroup looks.  Sizes: the
smallest and largest of each type and of both row counts (FP64: 256 / 257), a last
workgroup with one node, slices that are not full, FIC restarts, wrapping noise.
"""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("bold", "ext", "wIE_fic", "fic_trials", "fic_failed", "fc", "corr")


def _run(monkeypatch, prec, N, B, mark, period, graph=0):
    monkeypatch.setenv("BNM_GANG", "1")
    monkeypatch.setenv("BNM_GANG_MARK", str(mark))
    rng = np.random.default_rng(N)
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=150, bold_tr=10, n_vols_remove=2, no_fcd=1,
                             exc_interhemispheric=0, noise_period_ms=period, max_fic_trials=2, i_sampling_start=10,
                             i_sampling_end=50, precision=prec, fc_precision=bnm.FC_F64, use_graph=graph)
    with bnm.Context(cfg) as c:
        c.set_sc(W.synthetic_sc(N, 0.9, N))
        c.set_noise(bnm.make_noise(N, period * 20 * N))
        c.set_empirical(rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40))
        c.set_params(rng.uniform(0.02, 1.5, B), rng.uniform(0.15, 0.25, (B, N)), rng.uniform(0.1, 0.2, (B, N)))
        assert c.taken_over() == 0
        for _ in range(3 if graph else 1):
            c.run()
        assert c.kernel_name().startswith("gang")
        return c.taken_over(), c.outputs()


@pytest.mark.parametrize("prec,N", [(bnm.PREC_F32, n) for n in (257, 300, 320, 385, 400, 512)] +
                         [(bnm.PREC_F64, n) for n in (129, 160, 193, 200, 256, 257, 400, 449, 512)], ids=str)
def test_same_bits_on_one_workgroup(monkeypatch, prec, N):
    B = 5
    want = None
    for mark, taken in ((0, 0), (1, B), (2, 3)):
        print("case: gang alone precision", prec, "N", N, "mark", mark, flush=True)
        n, g = _run(monkeypatch, prec, N, B, mark, 151 if N % 2 else 70)
        assert n == taken
        want = want or g
        for k in KEYS:
            np.testing.assert_array_equal(g[k], want[k], err_msg=k)
    assert want["fic_trials"].max() > 0


def test_same_bits_in_a_graph(monkeypatch):
    a = _run(monkeypatch, bnm.PREC_F32, 290, 4, 0, 151)
    b = _run(monkeypatch, bnm.PREC_F32, 290, 4, 3, 151, graph=1)
    assert (a[0], b[0]) == (0, 2)
    for k in KEYS:
        np.testing.assert_array_equal(a[1][k], b[1][k], err_msg=k)


def test_a_launch_waits_once(monkeypatch):
    """A workgroup that never comes is waited for once a launch, not once a simulation:
    with 1024 simulations on 32 groups, 32 simulations a group, a longer patience costs
    its own length, not 32 times that.  (A poll takes between 0.3 and 3 us, so 40000
    polls 12 to 120 ms, and 31 more waits 0.37 s at least.)"""
    N, B, T = 500, 1024, 2
    monkeypatch.setenv("BNM_GANG", "1")
    took = []
    for mark, polls in ((1, 0), (-1, 40000)):
        print("case: gang waits, mark", mark, "polls", polls, flush=True)
        monkeypatch.setenv("BNM_GANG_MARK", str(mark))
        monkeypatch.setenv("BNM_GANG_POLLS", str(polls))
        cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=1, n_vols_remove=0, no_fcd=1,
                                 exc_interhemispheric=0, noise_period_ms=T + 1, adjust_fic=0, analytical_fic=0,
                                 precision=bnm.PREC_F32, fc_precision=bnm.FC_F32)
        with bnm.Context(cfg) as c:
            c.set_sc(W.synthetic_sc(N, 0.9, 1))
            c.set_noise(bnm.make_noise(1, (T + 1) * 20 * N))
            c.set_empirical(np.linspace(-0.2, 0.8, bnm.n_pairs(N, False)), np.linspace(-0.5, 1.0, 40))
            one = np.full((B, N), 0.2)
            c.set_params(np.full(B, 1.0), one, one, None, one)
            ms = []
            for _ in range(3):
                c.run()
                assert c.taken_over() == B
                ms.append(c.timings()["integrate"])
            took.append(min(ms))
    print("integration ms", took, flush=True)
    assert took[1] - took[0] < 300
