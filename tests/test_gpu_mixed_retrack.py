"""The FP64 pass of mixed-precision launches: escalated paths take part in the
comparison of roots that finds paths which jumped onto another path's root."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# x^3 = f(t) with f on the line from 1 to F1.  At this first step FP64
# prediction follows a path to the cube root it belongs to, and Newton from the
# unpredicted point takes path 0 to the root of path 1.
F1 = -2.0 + 0.3125j
OPTS = dict(dt0=0.1, max_corr=8)
# An offset whose FP32 spacing (16) exceeds the derivative of f: it cancels in
# H (every sum of it and F1 is exact), and in FP32 the derivative of f goes with
# it.
D = 1.5 * 2.0 ** 27 * (1 + 1j)


def jump_and_escalate(hcx, n):
    """Two paths of one instance: path 0 starts at 1 and jumps in FP32 (its
    predictor sees no motion); path 1 starts at exp(2 pi i / 3) with y = 1e20
    off its constant 2, which Newton in FP64 mends at once and whose square
    exceeds FP32.  Variables x, y, w = 0, v = 1, the rest 0."""
    mons = [  # equation, exponents, c(0), c(1) - c(0)
        (0, {0: 3}, 1, 0), (0, {}, -D - 1, D - (F1 - 1)), (0, {3: 1}, D, -D),
        (0, {1: 2, 2: 1}, 1, 0), (0, {2: 1}, -4, 0),
        (1, {1: 1}, 1, 0), (1, {}, -2, 0), (2, {2: 1}, 1, 0), (3, {3: 1}, 1, 0), (3, {}, -1, 0)]
    mons += [(i, {i: 1}, 1, 0) for i in range(4, n)]
    exps = np.array([[e.get(v, 0) for v in range(n)] for _, e, _, _ in mons], dtype=np.int32)
    sysf = hcx.System.from_monomials(exps, [m[0] for m in mons])
    hx = np.array([[m[2], m[3]] for m in mons] + [[1, 0]], dtype=np.complex128)
    ht = np.array([[m[3]] for m in mons] + [[0]], dtype=np.complex128)
    start = np.zeros((2, n), dtype=np.complex128)
    start[:, 0] = 1, np.exp(2j * np.pi / 3)
    start[:, 1] = 2, 1e20
    start[:, 3] = 1
    prob = hcx.Problem.from_system(sysf, start, with_affine=False)
    return prob, hcx.Batch(prob, 1, coeffs_hx=hx, coeffs_ht=ht)


@pytest.mark.parametrize("n", [5, 7, 18, 30])
def test_jump_onto_root_of_escalated_path(hcx_mod, gpu, n):
    """Sizes with an instance of their own (5, 30) and generic ones: both roots
    of FP64 are found."""
    import torch
    hcx = hcx_mod
    prob, b = jump_and_escalate(hcx, n)
    r = {p: hcx.track(prob, b, hcx.default_opts(precision=p, **OPTS)) for p in (0, 1)}
    torch.cuda.synchronize()
    f, m = r[0].to_host(), r[1].to_host()
    root = abs(F1) ** (1 / 3) * np.exp(1j * np.angle(F1) / 3)
    for g in (f, m):
        print(f"[n={n}] flags {g['flags']}, x {g['roots'][:, 0]}", flush=True)
        assert (g["flags"] & hcx.FLAG_REFINED).all()
        # a cube root of F1 from two roundings of its size
        assert np.abs(g["roots"][:, 0] - root * np.exp([0, 2j * np.pi / 3])).max() < 1e-14
    # path 1 failed in FP32 and path 0 was found on its root
    assert (m["flags"] & hcx.FLAG_ESCALATED).all()
    assert hcx.collect(r[1], hcx.default_opts())["unique"] == 2
    prob.close()


@pytest.mark.parametrize("n,waves", [(7, 1100), (12, 1100), (18, 700)])
def test_batch_without_a_path_for_fp32(hcx_mod, gpu, n, waves):
    """Coefficients beyond FP32: the FP64 pass tracks the whole batch, on as
    many waves as the batch has (its LDS lets a CU hold at least four, n = 18
    three), with the results of an FP64 launch bit for bit."""
    import ctypes
    import torch
    from hcx import workloads
    hcx = hcx_mod
    k, K = 2 * n, 32
    sysf = hcx.System.synthetic(n, k, num_quadratic=n, monomials=n + 6, seed=3 + n)
    p0 = workloads.random_cn(5 + n, k)
    start = workloads.seed_start_roots(sysf, p0, K, 7)
    count = waves * (64 // n) // K
    hx, ht = zip(*(sysf.param_homotopy_coeffs(p0, p) for p in workloads.targets(k, count, seed=11)))
    hx, ht = np.array(hx), np.array(ht)
    hx[:, :-1] *= 1e39
    ht[:, :-1] *= 1e39
    prob = hcx.Problem.from_system(sysf, start, with_affine=False)
    b = hcx.Batch(prob, count, coeffs_hx=hx, coeffs_ht=ht)
    f = hcx.track(prob, b, hcx.default_opts(precision=0, replicas=1))
    m = hcx.track(prob, b, hcx.default_opts(precision=1))
    shape = (ctypes.c_int * 7)()
    hcx.lib().hcx_internal_launch_shape(shape)
    torch.cuda.synchronize()
    f, m = f.to_host(), m.to_host()
    ok = (f["flags"] & hcx.FLAG_REFINED) != 0
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    needed = -(-len(ok) // (64 // n))
    print(f"[n={n}] {len(ok)} paths, {int(ok.sum())} refined, pass on {shape[4]} blocks of {needed}", flush=True)
    assert ok.mean() > 0.9
    assert shape[4] >= min(needed, (3 if n > 16 else 4) * cus)
    assert (m["flags"] == (f["flags"] | hcx.FLAG_ESCALATED)).all()
    for key in ("steps", "newton", "refine", "t_final", "roots"):
        assert np.array_equal(m[key], f[key], equal_nan=True), key
    prob.close()


def test_captured_retrack(hcx_mod, gpu):
    """Both rounds of the pass in a captured launch of two types: every replay
    gives the eager launch's results."""
    import torch
    hcx = hcx_mod
    problems, batches = zip(*(jump_and_escalate(hcx, n) for n in (5, 7)))
    opts = hcx.default_opts(precision=1, **OPTS)
    eager = [r.to_host() for r in hcx.track_multi(problems, batches, opts)]
    assert all((e["flags"] & hcx.FLAG_ESCALATED).all() for e in eager)
    graph = hcx.Graph(problems, batches, opts)
    for _ in range(4):
        for r in graph.results:
            r.flags.zero_()
            r.roots.zero_()
        hcx.track_multi(problems, batches, opts)
        replay = graph.launch()
        torch.cuda.synchronize()
        for r, e in zip(replay, eager):
            g = r.to_host()
            for key in ("flags", "steps", "newton", "refine", "roots"):
                assert np.array_equal(g[key], e[key], equal_nan=True), key
    graph.close()
    for p in problems:
        p.close()
