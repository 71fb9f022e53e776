"""Contexts with a scratch limit (lra_ctx_create's hbm_budget): what succeeded on the paths that
need the least scratch succeeds under the same limit on the faster ones."""
import contextlib

import numpy as np
import pytest

from test_gpu_kernels import host

pytestmark = pytest.mark.gpu

STEP = 32 << 10


@contextlib.contextmanager
def limited(gpu, budget):
    """The package's context replaced by one with a scratch limit of `budget` bytes."""
    import torch
    dev = torch.cuda.current_device()
    plain = gpu._lib.Context.get(dev)
    ctx = gpu._lib.Context(dev, budget)
    gpu._lib.Context._ctx[dev] = ctx
    try:
        yield
        torch.cuda.synchronize()
    finally:
        gpu._lib.Context._ctx[dev] = plain
        ctx.close()


def smallest_budget(gpu, call, most=1 << 30):
    """The smallest limit (to STEP bytes) under which a fresh context runs `call`."""
    lo, hi = 0, most // STEP
    while hi - lo > 1:
        mid = (lo + hi) // 2
        try:
            with limited(gpu, mid * STEP):
                call()
            hi = mid
        except gpu.LraError as e:
            assert "budget" in str(e), e
            lo = mid
    return hi * STEP


def spectrum(m, n, fall, seed):
    """A matrix with singular values exp(-fall i)."""
    rng = np.random.default_rng(seed)
    r = min(m, n)
    U, _ = np.linalg.qr(rng.standard_normal((m, r)))
    V, _ = np.linalg.qr(rng.standard_normal((n, r)))
    return (U * np.exp(-fall * np.arange(r))) @ V.T


@pytest.mark.parametrize("m,n,fall,rtol,env", [
    # orders 520 (rejected) and 1032 on the register grid or in blocks, one after the other
    (1500, 1500, 0.015, 1e-4, {"LRA_QRCP_PAIR": "0"}),
    (1400, 1300, 0.02, 1e-7, {"LRA_QRCP_GLOBAL": "1"})])  # every round in HBM
def test_blocks_fit_where_single_steps_did(gpu, monkeypatch, m, n, fall, rtol, env):
    """The smallest limit that holds a slowly decaying idfact without blocks of pivoted-QR steps
    holds it with them, and gives the same ID."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    A = gpu.to_device(spectrum(m, n, fall, 5))
    run = lambda: gpu.idfact(A, rtol=rtol, seed=4)
    V1 = run()  # (products tuned without a limit)
    monkeypatch.setenv("LRA_QG_BLOCK", "0")
    V0 = run()
    budget = smallest_budget(gpu, run)
    monkeypatch.delenv("LRA_QG_BLOCK")
    assert V1.k == V0.k > 500
    with limited(gpu, budget):
        V = run()
    assert V.k == V0.k and np.array_equal(host(V.sk), host(V0.sk))


def direct_id(gpu):
    """An ID without a sketch, and the smallest limit that holds it."""
    B = gpu.to_device(spectrum(700, 900, 0.05, 2))
    call = lambda: gpu.idfact(B, rtol=1e-9, sketch="none")
    k = call().k
    return call, k, smallest_budget(gpu, call)


def test_narrow_product_leaves_room(gpu):
    """A product with few columns whose tiled form takes no scratch (1024 x 64, K = 512, beta = 1)
    leaves a limited context's room to the call that follows."""
    import torch
    call, k, budget = direct_id(gpu)
    rng = np.random.default_rng(3)
    A, B, C = (np.asfortranarray(rng.standard_normal(s)) for s in ((1024, 512), (512, 64), (1024, 64)))
    ref = A @ B + C
    with limited(gpu, budget):
        Cd = gpu.to_device(C).clone().t().contiguous().t()
        gpu.dgemm(A, B, "n", "n", 1.0, Cd, 1.0)
        assert call().k == k
    bound = 2.3e-16 * 520 * (np.abs(A) @ np.abs(B) + np.abs(C))
    assert (np.abs(host(Cd) - ref) <= bound).all()


@pytest.mark.parametrize("m,n", [(600, 40000), (2000, 9000)])
def test_snorm_leaves_room(gpu, m, n):
    """snorm under a limit keeps to the partial sums of 256-column chunks, as many as about four
    blocks of 256 rows per CU ask for: an ID that fits beside them still fits after it."""
    import torch
    call, k, budget = direct_id(gpu)
    g = torch.Generator(device="cuda").manual_seed(1)
    A = torch.randn((n, m), generator=g, device="cuda", dtype=torch.float64).t()
    ref = gpu.snorm(A, snorm_niter=4, rtol=0.0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rt = -(-m // 256)
    chunks = min(-(-n // 256), -(-4 * cus // rt))
    with limited(gpu, budget + 8 * (n + m + 65 + chunks * m)):
        got = gpu.snorm(A, snorm_niter=4, rtol=0.0)
        assert call().k == k
    assert abs(got - ref) <= 1e-12 * ref


def test_odd_sketch_takes_no_larger_partials(gpu):
    """The tuner's candidates for a sketch with an odd leading dimension take no more K ranges
    (their partial sums are the scratch) than the generic tiles': 16 at 531 x 2048, K = 8193."""
    import torch
    m, n, order = 8193, 2048, 531
    g = torch.Generator(device="cuda").manual_seed(2)
    A = torch.randn((n, m), generator=g, device="cuda", dtype=torch.float64).t()
    with limited(gpu, 8 * (order * (m + 1) + 16 * order * n) + (1 << 16)):
        B = host(gpu.sketch("left", "n", A, order, seed=3))
    Om, Ah = host(gpu.gaussian(order, m, 3, 0)), host(A)
    assert (np.abs(B - Om @ Ah) <= 2.3e-16 * (m + 4) * (np.abs(Om) @ np.abs(Ah))).all()


def test_refused_workspace_leaves_no_error(gpu):
    """A workspace that the device cannot give is an error of that call alone."""
    import torch
    L = gpu._lib.load()
    ctx = gpu.context()
    A, out = torch.ones(1000, device="cuda", dtype=torch.float64), torch.empty(64, device="cuda", dtype=torch.float64)
    p = gpu._ptr
    order = 1 << 40  # Omega: 8 PiB
    st = L.lra_sketch_gaussian(ctx.h, 0, 0, 1000, 1, p(A), 1000, order, None, 1, 0, 0, p(out), order)
    assert st == 2, L.lra_last_error()
    assert L.lra_gaussian_fill(ctx.h, 1, 0, 64, 1, p(out), 64) == 0, L.lra_last_error()
    torch.cuda.synchronize()
    assert torch.isfinite(out).all()
