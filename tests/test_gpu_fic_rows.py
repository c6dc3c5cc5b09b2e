"""Analytical FIC with the SC's rows through LDS: row and column remainders of its
tiles, each workgroup size, more rows than one pass holds, and an unstable
simulation, against the FP64 oracle."""
import numpy as np
import pytest

import bnm_cuda_amd as bnm
from bnm_cuda_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 255, 256, 257, 300, 513])
def test_rows(oracle_mod, N):
    print("case: analytical fic N", N, flush=True)
    B = 3
    rng = np.random.default_rng(N)
    SC = W.synthetic_sc(N, 0.5, N) if N >= 8 else rng.uniform(0, 0.3, (N, N))
    SC = SC * rng.uniform(0.5, 1.5, SC.shape)          # rows and columns differ
    G = np.array([0.0, 1.3, 2.4])
    wEE, wEI = rng.uniform(0.1, 0.4, (B, N)), rng.uniform(0.1, 0.4, (B, N))
    wEI[2, N // 2] = -3.0                               # no fixed point or a negative wIE
    w, unstable = bnm.analytical_fic(SC, G, wEE, wEI)
    for b in range(B):
        wo, uo = oracle_mod.analytical_fic(SC, G[b], wEE[b], wEI[b])
        assert bool(unstable[b]) == bool(uo)
        want = np.ones(N) if uo else wo
        # The same expressions in the same order: equal to a few roundings, except
        # where another rounding of exp lets the root search (interval 1e-3) stop a
        # step earlier or later.
        rel = np.abs(w[b] - want) / np.abs(want)
        assert np.median(rel) <= 1e-12 and rel.max() <= 5e-3, (b, np.median(rel), rel.max())
