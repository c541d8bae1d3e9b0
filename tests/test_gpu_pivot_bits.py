"""The pivot search of the FP64 solve compares whole magnitudes: candidates
whose keys share all but the last bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def near_tie(hcx, n, at, m):
    """The rows x_at + x_at+1 = 0 and c x_at + c x_at+1 = 0 with c = 1 + m 2^-52,
    and x_i = 1 for the others, started on the solution, constant in t: every
    right-hand side is exactly 0.  With the larger magnitude c as pivot, 1 / c
    rounds to 1 - m 2^-52 and the other row's second entry becomes
    1 - (1 - m 2^-52)(1 + m 2^-52) = m^2 2^-104 in one fused operation, and
    the solve returns 0.  With the earlier and smaller 1 as pivot it is c - c * 1 = 0,
    a zero pivot column."""
    c = 1.0 + m * 2.0 ** -52
    mons = [(at, at, 1.0), (at, at + 1, 1.0), (at + 1, at, c), (at + 1, at + 1, c)]
    for i in range(n):
        if i not in (at, at + 1):
            mons += [(i, i, 1.0), (i, None, -1.0)]
    exps = np.array([[int(v == w) for w in range(n)] for _, v, _ in mons], dtype=np.int32)
    sysf = hcx.System.from_monomials(exps, [q[0] for q in mons])
    start = np.ones((8, n), dtype=np.complex128)
    start[:, at:at + 2] = 0
    prob = hcx.Problem.from_system(sysf, start, with_affine=False)
    hx = np.zeros((len(mons) + 1, 2), dtype=np.complex128)
    hx[:, 0] = [q[2] for q in mons] + [1]
    return prob, hx


# n with an instance of their own (8 and 16: lane groups of a power of two, 30:
# of 32 lanes) and generic ones; instances of 8 paths each: few (replicas share
# the solve's columns), more than a wave per SIMD, and a full GPU
@pytest.mark.parametrize("n", [3, 5, 7, 8, 12, 16, 18, 30, 32])
@pytest.mark.parametrize("m", [1, 16, 31])
def test_larger_later_candidate(hcx_mod, gpu, n, m):
    import torch
    hcx = hcx_mod
    for at in (0, n - 2):
        prob, hx = near_tie(hcx, n, at, m)
        for waves, kw in ((1, {}), (1, dict(replicas=1)), (1100, {}), (2100, dict(replicas=1))):
            count = max(1, waves * (64 // n) // 8)
            b = hcx.Batch(prob, count, coeffs_hx=np.tile(hx, (count, 1, 1)),
                          coeffs_ht=np.zeros((count, len(hx), 1), dtype=np.complex128))
            r = hcx.track(prob, b, hcx.default_opts(precision=0, **kw))
            torch.cuda.synchronize()
            g = r.to_host()
            assert (g["flags"] & hcx.FLAG_REFINED).all(), (n, at, waves, kw, g["flags"][:4])
            assert not (g["flags"] & hcx.FLAG_SINGULAR).any()
            assert (g["roots"] == prob.start_sols[0]).all()
        prob.close()
