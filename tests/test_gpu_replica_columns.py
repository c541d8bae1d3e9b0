"""Replica lane groups that share columns: the evaluation dealt out by columns
(launches past one wave per SIMD) and the solve's columns dealt out (any
number of replicas), at sizes on and beside the instances' edges."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(hcx, prob, batch, **kw):
    import torch
    r = hcx.track(prob, batch, hcx.default_opts(precision=0, **kw))
    torch.cuda.synchronize()
    return r.to_host()


# n, quadratic equations (the rest cubic), monomials, start roots, lanes' waves
# at one replica, specialised: n = 9, 12 and 16 with their remainders of two and
# four replicas, a cubic one, generic ones below and above 8, and one of 660
# coefficients, whose LDS takes four replicas at this size (at 300 waves four
# replicas split its term sums, which rounds differently)
DEALT = [(3, 3, 10, 8, 1060, 1), (5, 5, 11, 16, 1100, 1), (9, 9, 15, 64, 1100, 1), (12, 12, 18, 64, 1050, 1),
         (16, 16, 22, 40, 1100, 1), (10, 10, 0, 64, 700, 1), (6, 3, 14, 32, 1100, 1), (7, 7, 13, 32, 1100, 1),
         (11, 11, 17, 32, 1040, 1), (9, 9, 15, 64, 1100, 0)]


@pytest.mark.parametrize("n,quadratic,monomials,K,waves,specialize", DEALT)
def test_dealt_columns_equal_whole_sums(hcx_mod, gpu, n, quadratic, monomials, K, waves, specialize):
    """Each column is summed whole, in the order of one replica: every output
    of the launch equals that of replicas = 1 bit for bit."""
    from hcx import workloads
    hcx = hcx_mod
    sysf = hcx.System.synthetic(n, 2 * n, num_quadratic=quadratic, monomials=monomials, seed=41 + n)
    p0 = workloads.random_cn(43 + n, 2 * n)
    start = workloads.seed_start_roots(sysf, p0, K, 47)
    prob = hcx.Problem.from_system(sysf, start, p0=p0)
    count = max(1, waves * (64 // n) // len(start))
    b = hcx.Batch(prob, count, target_params=workloads.targets(2 * n, count, seed=53))
    a = _solve(hcx, prob, b, specialize=specialize)
    w = _solve(hcx, prob, b, specialize=specialize, replicas=1)
    print(f"[n={n}] {count * len(start)} paths, refined {int(((a['flags'] & 4) != 0).sum())}", flush=True)
    for key in ("flags", "steps", "newton"):
        assert (a[key] == w[key]).all(), key
    both_nan = np.isnan(a["roots"]) & np.isnan(w["roots"])
    assert ((a["roots"] == w["roots"]) | both_nan).all()
    prob.close()


@pytest.mark.parametrize("n,replicas", [(2, 8), (3, 4), (7, 2), (8, 8), (11, 4), (13, 2), (16, 4), (17, 2), (31, 2),
                                        (32, 2)])
def test_split_solve_sizes(hcx_mod, gpu, n, replicas):
    """Columns of the solve over R replicas, with n on and off multiples of R:
    the split sums round differently, so refined roots agree to 1e-10 relative
    (the refinement's contraction leaves an error of a few units of rounding
    times the condition of the root), and the same paths refine."""
    from hcx import workloads
    hcx = hcx_mod
    k = 2 * n
    sysf = hcx.System.synthetic(n, k, num_quadratic=n, monomials=0 if n <= 3 else n + 6, seed=61 + n)
    p0 = workloads.random_cn(67 + n, k)
    start = workloads.seed_start_roots(sysf, p0, min(2 ** n, 16), 71)
    prob = hcx.Problem.from_system(sysf, start, p0=p0)
    b = hcx.Batch(prob, 4, target_params=workloads.targets(k, 4, seed=73))
    one = _solve(hcx, prob, b, replicas=1)
    rep = _solve(hcx, prob, b, replicas=replicas)
    ok = (one["flags"] & hcx.FLAG_REFINED) != 0
    assert (ok == ((rep["flags"] & hcx.FLAG_REFINED) != 0)).all()
    assert ok.mean() > 0.5
    err = np.abs(one["roots"][ok] - rep["roots"][ok]).max(axis=1) / np.maximum(
        1.0, np.abs(one["roots"][ok]).max(axis=1))
    print(f"[n={n} R={replicas}] refined {int(ok.sum())} of {len(ok)}, max rel diff {err.max():.2e}", flush=True)
    assert err.max() <= 1e-10
    prob.close()
