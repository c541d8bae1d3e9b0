"""waves_per_cu of launches whose blocks hold several waves: a request is met to
the wave, and results do not depend on it."""
import numpy as np
import pytest

from test_gpu_term_records import launch_shape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision,replicas", [(12, 1, 0), (16, 0, 1)])
def test_requested_waves(hcx_mod, gpu, n, precision, replicas):
    """n = 12 in mixed precision runs seven waves per CU in one block, n = 16
    five to eight; a block of r waves fits wherever a larger one does, so every
    smaller number can be had exactly."""
    import torch
    from hcx import workloads
    hcx = hcx_mod
    k, K = 2 * n, 64
    sysf = hcx.System.synthetic(n, k, num_quadratic=n, monomials=20, seed=7 + n)
    p0 = workloads.random_cn(9 + n, k)
    prob = hcx.Problem.from_system(sysf, workloads.seed_start_roots(sysf, p0, K, 11), p0=p0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    count = 9 * cus * (64 // n) // prob.num_tracks + 1
    b = hcx.Batch(prob, count, target_params=workloads.targets(k, count, seed=13))

    def run(request):
        r = hcx.track(prob, b, hcx.default_opts(precision=precision, replicas=replicas, waves_per_cu=request))
        s = launch_shape(hcx)
        torch.cuda.synchronize()
        return r.to_host(), s

    full, shape = run(0)
    waves = shape["waves_per_block"] * shape["blocks"] // cus
    print(f"[n={n}] {waves} waves per CU in blocks of {shape['waves_per_block']}", flush=True)
    assert shape["waves_per_block"] > 4
    for request in list(range(1, waves + 1)) + list(range(-waves, 0)):
        g, s = run(request)
        want = request if request > 0 else max(waves + request, 1)
        assert s["waves_per_block"] * s["blocks"] == want * cus, (request, s)
        for key in ("flags", "steps", "roots"):
            assert np.array_equal(g[key], full[key], equal_nan=True), (request, key)
    prob.close()


def test_tuned_density(hcx_mod, gpu):
    """The autotuner's candidate of half the density is half of what runs, and a
    stored density is met."""
    import torch
    from hcx import workloads
    hcx = hcx_mod
    n, k = 12, 24
    sysf = hcx.System.synthetic(n, k, num_quadratic=n, monomials=20, seed=19)
    p0 = workloads.random_cn(21, k)
    prob = hcx.Problem.from_system(sysf, workloads.seed_start_roots(sysf, p0, 64, 11), p0=p0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    count = 9 * cus * 5 // prob.num_tracks + 1
    b = hcx.Batch(prob, count, target_params=workloads.targets(k, count, seed=13))
    opts = hcx.default_opts(precision=1)
    hcx.track(prob, b, opts)
    full = launch_shape(hcx)
    for density in (3, 2):
        assert hcx.lib().hcx_problem_set_launch_shape(prob.handle, n, 1, density) == 0
        hcx.track(prob, b, opts)
        s = launch_shape(hcx)
        assert s["waves_per_block"] * s["blocks"] == density * cus, s
    best = hcx.autotune(prob, b, opts)
    waves = full["waves_per_block"] * full["blocks"] // cus
    print(f"[tuned] {best}, {waves} waves per CU", flush=True)
    assert best["waves_per_cu"] in (0, waves // 2)
    prob.close()
