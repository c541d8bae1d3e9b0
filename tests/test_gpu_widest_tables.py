"""The most coefficients that a lane group's LDS holds: c(t) of one path fills a
CU's 160 KiB up to the padding."""
import numpy as np
import pytest

from test_gpu_parity import compare
from test_gpu_term_records import homotopy, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coefficients", [10189, 10190, 10191])
def test_widest_tables(hcx_mod, oracle_mod, gpu, coefficients):
    """n = 17, cubic, one group per wave: the x slots, the pivot keys and
    16 bytes for each coefficient (its 10,191 leave 224 bytes)."""
    hcx, oracle = hcx_mod, oracle_mod
    n = 17
    system, start, hx, ht = homotopy(hcx, n, 3, 600, 4, 1, 5)
    exps, eq = system.monomials()
    # the first equations lose cross terms until the number is met
    drop, left = np.zeros(len(eq), dtype=bool), len(eq) - coefficients
    for j in np.nonzero((exps > 0).sum(axis=1) > 1)[0][:left]:
        drop[j] = True
    system = hcx.System.from_monomials(exps[~drop], eq[~drop])
    keep = np.append(~drop, True)
    hx, ht = hx[:, keep].copy(), ht[:, keep].copy()
    assert system.info["num_coeffs"] == coefficients
    prob = hcx.Problem.from_system(system, start, with_affine=False)
    b = hcx.Batch(prob, 1, coeffs_hx=hx, coeffs_ht=ht)
    hxi, hti = system.tables()
    o = oracle.OracleProblem(n, coefficients, hxi, hti, 1).track(start, hx, ht, threads=4)
    for precision in (0, 1):
        g, _ = run(hcx, prob, b, precision=precision)
        compare(hcx, oracle, g, o, f"C={coefficients} precision={precision}", exact_flags=precision == 0)
    prob.close()
