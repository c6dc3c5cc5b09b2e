"""The first context of a process chooses its kernel as later ones do: what the first
launch of a kernel costs is not held against it."""
import os
import re
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import numpy as np
import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W
N, B, T = 41, 2036, 300
noise = bnm.make_noise(1, (T + 1) * 20 * N)
n = bnm.n_pairs(N, False)
for k in range(2):
    cfg = bnm.default_config(nodes=N, n_sims=B, time_steps=T, bold_tr=100, n_vols_remove=0, no_fcd=1, adjust_fic=0,
                             exc_interhemispheric=0, noise_period_ms=T + 1, precision=bnm.PREC_F32)
    with bnm.Context(cfg) as c:
        c.set_sc(W.synthetic_sc(N, 0.4, 1))
        c.set_noise(noise)
        c.set_empirical(np.linspace(-0.2, 0.8, n), np.linspace(-0.5, 1.0, 40))
        c.set_params(np.full(B, 1.0), np.full((B, N), 0.2), np.full((B, N), 0.2))
        c.run()
        print(c.tune_log(), flush=True)
"""


def test_first_context_is_tuned_as_the_second():
    print("case: tuner of a new process", flush=True)
    out = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, env=dict(os.environ, PYTHONPATH=ROOT), check=True,
                         capture_output=True, text=True, timeout=110).stdout
    print(out, flush=True)
    first, second = ({k: float(v) for k, v in re.findall(r"(\w+\([^)]*\))=([\d.]+)ms", line)}
                     for line in out.strip().splitlines()[-2:])
    assert first.keys() == second.keys() and len(first) == 3
    for k in first:
        assert first[k] <= 2 * second[k] + 0.2, k
