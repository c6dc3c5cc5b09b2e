"""Graphs of several populations: small populations are paired before the deal where that
ends sooner, every context runs once, and results are those of the contexts' own runs."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("bold", "ext", "wIE_fic", "fic_trials", "fc", "corr")


def _context(prec, N, B, T):
    rng = np.random.default_rng(N)
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=20, n_vols_remove=1, no_fcd=1,
                             exc_interhemispheric=0, noise_period_ms=100, max_fic_trials=1, i_sampling_start=10,
                             i_sampling_end=60, precision=prec, fc_precision=bnm.FC_F64)
    c = bnm.Context(cfg)
    c.set_sc(W.synthetic_sc(N, 0.9, N))
    c.set_noise(bnm.make_noise(N, 100 * 20 * N))
    c.set_empirical(rng.uniform(-0.2, 0.8, bnm.n_pairs(N, False)), rng.uniform(-0.5, 1.0, 40))
    c.set_params(rng.uniform(0.5, 2.5, B), rng.uniform(0.1, 0.4, (B, N)), rng.uniform(0.1, 0.3, (B, N)))
    return c


def _check(specs):
    ctxs = [_context(*s) for s in specs]
    try:
        eager = []
        for c in ctxs:
            c.run()
            eager.append(c.outputs())
        m = bnm.Multi(ctxs)
        plan = m.plan()
        print("plan:", plan, [c.kernel_name() for c in ctxs], flush=True)
        assert sorted(int(w.split()[0]) for w in plan.split("ctx ")[1:]) == list(range(len(specs)))
        for _ in range(3):
            m.run()
            for c, e in zip(ctxs, eager):
                o = c.outputs()
                for k in KEYS:
                    np.testing.assert_array_equal(o[k], e[k], err_msg=k)
        m.close()
        return plan
    finally:
        for c in ctxs:
            c.close()


def test_small_populations_are_paired_before_the_deal():
    print("case: multi, two small and one large population, FP32", flush=True)
    plan = _check([(bnm.PREC_F32, 68, 128, 600), (bnm.PREC_F32, 100, 128, 600), (bnm.PREC_F32, 200, 128, 300)])
    pair = plan[plan.index("[") + 1:plan.index("]")]
    assert "N=68," in pair and "N=100," in pair and "N=200," not in pair


@pytest.mark.parametrize("specs", [
    [(bnm.PREC_F64, 68, 128, 300), (bnm.PREC_F64, 100, 128, 300), (bnm.PREC_F64, 40, 128, 200)],
    [(bnm.PREC_F32, 64, 256, 300), (bnm.PREC_F32, 30, 256, 300), (bnm.PREC_F32, 100, 256, 300), (bnm.PREC_F32, 20, 256, 300)],
    [(bnm.PREC_F32, 64, 100, 300), (bnm.PREC_F32, 160, 100, 300)]], ids=("f64", "one branch", "two branches"))
def test_every_population_runs_once(specs):
    print("case: multi", specs, flush=True)
    _check(specs)


def test_fp64_populations_that_fill_the_registers_are_not_paired():
    print("case: multi, FP64 beyond 64 nodes", flush=True)
    plan = _check([(bnm.PREC_F64, 68, 256, 200), (bnm.PREC_F64, 100, 256, 200)])
    assert "[" not in plan
