"""Launches that deal the Jacobian's columns out to replicas: that they do, and
every output against whole sums per lane."""
import numpy as np
import pytest

from test_gpu_replica_columns import DEALT
from test_gpu_term_records import run

pytestmark = pytest.mark.gpu

# replicas of each case of DEALT: two past one wave per SIMD; four where the
# coefficients leave LDS for two waves per CU (n = 10, 660 coefficients)
REPLICAS = [4 if monomials == 0 else 2 for _, _, monomials, _, _, _ in DEALT]
# the same on the generic instance: n = 11, 858 coefficients
CASES = list(zip(DEALT, REPLICAS)) + [((11, 11, 0, 64, 700, 1), 4)]


@pytest.mark.parametrize("case,replicas", CASES)
def test_columns_are_dealt(hcx_mod, gpu, case, replicas):
    from hcx import workloads
    hcx = hcx_mod
    n, quadratic, monomials, K, waves, specialize = case
    sysf = hcx.System.synthetic(n, 2 * n, num_quadratic=quadratic, monomials=monomials, seed=41 + n)
    p0 = workloads.random_cn(43 + n, 2 * n)
    start = workloads.seed_start_roots(sysf, p0, K, 47)
    prob = hcx.Problem.from_system(sysf, start, p0=p0)
    count = max(1, waves * (64 // n) // len(start))
    b = hcx.Batch(prob, count, target_params=workloads.targets(2 * n, count, seed=53))
    a, shape = run(hcx, prob, b, specialize=specialize)
    w, whole = run(hcx, prob, b, specialize=specialize, replicas=1)
    print(f"[n={n}] {shape}", flush=True)
    assert (shape["dealt"], shape["replicas"]) == (1, replicas)
    assert (whole["dealt"], whole["replicas"]) == (0, 1)
    assert ((a["flags"] & hcx.FLAG_REFINED) != 0).mean() > 0.9
    for key in ("flags", "steps", "newton", "refine", "t_final", "dt_final", "roots", "residual"):
        assert np.array_equal(a[key], w[key], equal_nan=True), key
    prob.close()
