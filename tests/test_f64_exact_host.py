"""The FP64 update of the row-blocked and multi-workgroup kernels is as exact as the
reference's order of operations (CPU, against 128-bit arithmetic).

`tests/host_model/f64_exact.cpp` builds pool.hpp and math64.hpp on the host.

* Functions, over the ranges that the model reaches, in ulp: a result that is
  rounded once from an argument that is exact to half an ulp of the result is
  within 1; each further rounding of the result's size adds a half.  exp: 1.5
  (1 + m, and m), log: 1, pow: 2 (exp of a rounded argument, and the correction),
  1 - exp: 3 (both terms, up to 2.3 times the difference, and the difference).
* Runs of 6 nodes: rms errors of S_E and BOLD no larger than those of the
  reference's order on the same inputs.  Both are sums of some 1e5 independent
  roundings of eight parameter sets; the quotient of two such rms values varies by
  well under a quarter.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
INC = os.path.join(HERE, "host_model")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("f64") / "f64_exact")
    subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-I", INC, "-o", out,
                    os.path.join(INC, "f64_exact.cpp"), "-lquadmath"], check=True)
    return out


def _values(exe, *args):
    text = subprocess.run([exe, *args], check=True, capture_output=True, text=True, timeout=300).stdout
    print(text)
    return {k: float(v) for k, v in (line.split() for line in text.splitlines())}


def test_functions_within_ulps(exe):
    v = _values(exe, "functions")
    bound = dict(exp=1.5, log=1.0, log_near_1=1.0, pow=2.0, one_minus_exp=3.0, one_minus_exp_small=3.0)
    assert set(v) == set(bound)
    for k, b in bound.items():
        assert v[k] <= b, k


def test_edge_values(exe):
    """Infinite, undefined and far values end as they do in the reference's order (NaN
    BOLD, hence the largest cost; an infinite rate), not in other finite values."""
    assert _values(exe, "edges") == dict(edges=0)


def test_runs_no_less_exact_than_the_reference_order(exe):
    v = _values(exe, "runs", "3000", "8")
    assert v["S_kernels"] <= 1.25 * v["S_reference"]
    assert v["BOLD_kernels"] <= 1.25 * v["BOLD_reference"]
