"""The forms in which the kernels hold a problem's term records (compact
records in LDS, full records in LDS or in global memory) against the oracle, at
the edges of the compact ones."""
import ctypes
import itertools

import numpy as np
import pytest

from test_gpu_parity import ROOT_TOL, compare, rel_err

pytestmark = pytest.mark.gpu


def launch_shape(hcx):
    """Of this thread's latest launch (LaunchShape in hcx_internal.hpp)."""
    s = (ctypes.c_int * 7)()
    hcx.lib().hcx_internal_launch_shape(s)
    return dict(zip(("replicas", "dealt", "waves_per_block", "blocks", "pass_blocks", "specialized",
                     "record_bytes"), s))


def homotopy(hcx, n, degree, monomials, K, instances, seed):
    """Straight lines from gamma_i (x_i^degree - 1) to random coefficients:
    system, start roots, tables of the instances."""
    rng = np.random.default_rng([n, degree, seed])
    exps, eq = [], []
    for i in range(n):
        rows = [tuple([0] * n)] + [tuple(degree if v == w else 0 for v in range(n)) for w in range(n)]
        while len(rows) < monomials:
            e = np.bincount(rng.integers(0, n, rng.integers(1, degree + 1)), minlength=n)
            if tuple(e) not in rows:
                rows.append(tuple(e))
        exps += rows
        eq += [i] * len(rows)
    exps, eq = np.array(exps, dtype=np.int32), np.array(eq, dtype=np.int32)
    gamma = np.exp(2j * np.pi * rng.random(n))
    g = np.where(exps.any(axis=1), np.where(exps[np.arange(len(eq)), eq] == degree, gamma[eq], 0), -gamma[eq])
    f = (rng.standard_normal((instances, len(eq))) + 1j * rng.standard_normal((instances, len(eq)))) / np.sqrt(2)
    hx = np.zeros((instances, len(eq) + 1, 2), dtype=np.complex128)
    hx[:, :-1, 0], hx[:, :-1, 1], hx[:, -1, 0] = g, f - g, 1
    picks = itertools.islice(itertools.product(range(degree), repeat=n), K)
    start = np.exp(2j * np.pi * np.array(list(picks)) / degree)
    return hcx.System.from_monomials(exps, eq), start, hx, hx[:, :, 1:].copy()


def scaled_problem(hcx, system, start, scalar, at=0):
    """Equation `at` multiplied by an integer in the scalars of its terms."""
    hxi, hti = (t.copy() for t in system.tables())
    hxi[at, ..., 0] *= scalar
    hti[at, ..., 0] *= scalar
    return hcx.Problem(system.info["num_vars"], system.info["num_coeffs"], hxi, hti, start), hxi, hti


def run(hcx, prob, b, **kw):
    import torch
    r = hcx.track(prob, b, hcx.default_opts(**kw))
    shape = launch_shape(hcx)
    torch.cuda.synchronize()
    return r.to_host(), shape


@pytest.mark.parametrize("n,degree", [(4, 3), (5, 4), (8, 3), (12, 3)])
@pytest.mark.parametrize("scalar,fits", [(10922, True), (8191, True), (-8192, True), (32768, False)])
def test_scalars_of_compact_records(hcx_mod, oracle_mod, gpu, n, degree, scalar, fits):
    """Scalars of up to 16 bits (the derivative multiplies them by up to the
    degree) keep the instance of the size; wider ones run the generic one."""
    hcx, oracle = hcx_mod, oracle_mod
    system, start, hx, ht = homotopy(hcx, n, degree, n + 5, 16, 6, 1)
    fits = fits and abs(scalar) * degree < 32768 + (scalar < 0)
    prob, hxi, hti = scaled_problem(hcx, system, start, scalar, at=n - 1)
    b = hcx.Batch(prob, len(hx), coeffs_hx=hx, coeffs_ht=ht)
    op = oracle.OracleProblem(n, system.info["num_coeffs"], hxi, hti, 1)
    o = op.track(start, hx, ht, threads=8)
    for kw in (dict(precision=0, replicas=1), dict(precision=0), dict(precision=1)):
        g, shape = run(hcx, prob, b, **kw)
        # mixed precision has no instance of its own at degree 4
        assert shape["specialized"] == (1 if fits and not (kw["precision"] and degree > 3) else 0), (kw, shape)
        compare(hcx, oracle, g, o, f"n={n} d={degree} s={scalar} {kw}", exact_flags=False)
    assert ((o["flags"] & hcx.FLAG_REFINED) != 0).mean() > 0.5
    prob.close()


# a step control that leaves no path to a rounding: the roots of FP64, of mixed
# precision and of the oracle are the same ones
STEADY = dict(dt0=0.02, corr_tol=1e-10, max_steps=2000)


def against_oracle(hcx, oracle, n, degree, scalar, seed, records, launches):
    """Runs the launches (waves at one replica, options) of copies of four
    instances; records(shape, options) checks the form that each took."""
    system, start, hx, ht = homotopy(hcx, n, degree, n + 5, 8, 4, seed)
    prob, hxi, hti = scaled_problem(hcx, system, start, scalar)
    op = oracle.OracleProblem(n, system.info["num_coeffs"], hxi, hti, 1)
    o = op.track(start, hx, ht, threads=8, **STEADY)
    assert ((o["flags"] & hcx.FLAG_REFINED) != 0).mean() > 0.5
    P = len(o["flags"])
    for waves, kw in launches:
        copies = max(1, waves * (64 // max(n, kw.get("lanes_per_path", 0))) // P)
        b = hcx.Batch(prob, 4 * copies, coeffs_hx=np.tile(hx, (copies, 1, 1)), coeffs_ht=np.tile(ht, (copies, 1, 1)))
        g, shape = run(hcx, prob, b, **STEADY, **kw)
        records(shape, kw)
        first = {k: v[:P] for k, v in g.items() if k not in ("inst_done", "batch_start")}
        label = f"n={n} d={degree} s={scalar} {waves} {kw} {shape}"
        if kw.get("precision"):
            # a path that FP64 loses may arrive by another step sequence; those that it follows arrive at its roots
            both = (o["flags"] & hcx.FLAG_REFINED) != 0
            more = ((first["flags"] & hcx.FLAG_REFINED) != 0) & ~both
            print(f"[{label}] oracle {both.sum()}, more {more.sum()}", flush=True)
            assert ((first["flags"][both] & hcx.FLAG_REFINED) != 0).all(), label
            assert (rel_err(first["roots"][both], o["roots"][both]) <= ROOT_TOL).all(), label
        else:
            compare(hcx, oracle, first, o, label, exact_flags=False)
        for key in ("flags", "steps", "newton", "roots"):
            assert np.array_equal(np.tile(first[key].T, copies).T, g[key], equal_nan=True), key
    prob.close()


LAUNCHES = [(1, dict(replicas=1)), (1, dict(replicas=2)), (1, {}), (2100, dict(replicas=1)), (1, dict(precision=1))]


@pytest.mark.parametrize("n,degree", [(2, 5), (3, 6), (5, 5), (8, 6), (9, 5), (16, 6), (17, 5)])
@pytest.mark.parametrize("scalar", [1, -21845])
def test_compact_records_of_degree_5_and_6(hcx_mod, oracle_mod, gpu, n, degree, scalar):
    """Records in LDS with three words of variables, scalars of up to 18 bits;
    n on both sides of the generic instances' widths."""
    def records(shape, kw):
        assert shape["record_bytes"] > 0 and not shape["specialized"], (kw, shape)
    against_oracle(hcx_mod, oracle_mod, n, degree, scalar, 2, records, LAUNCHES)


@pytest.mark.parametrize("n,degree,scalar", [(5, 2, 100), (12, 2, 100), (6, 3, 1 << 18), (10, 3, 1 << 18),
                                             (7, 4, 1 << 18), (20, 2, 100), (3, 6, 1 << 18), (8, 5, 1 << 18)])
def test_full_records(hcx_mod, oracle_mod, gpu, n, degree, scalar):
    """Scalars that no compact form of the degree holds: full records, copied to
    LDS by the latency instances and in global memory else."""
    def records(shape, kw):
        few = not kw.get("precision") and shape["blocks"] * shape["waves_per_block"] < 1000
        assert not shape["specialized"]
        if few and n <= 10:  # beyond, the groups' coefficients may leave no room for the records
            assert shape["record_bytes"] > 0 and shape["record_bytes"] % 16 == 0, (kw, shape)
        if not few:
            assert shape["record_bytes"] == 0, (kw, shape)
    against_oracle(hcx_mod, oracle_mod, n, degree, scalar, 3, records, LAUNCHES)
