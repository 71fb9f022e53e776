"""snorm / snormdiff on the GPU (test/snorm.jl:12-25 bounds) and the ID error through
snormdiff against numpy's 2-norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def test_snorm_reference_cases(gpu):
    rng = np.random.default_rng(0)
    rtol = 100 * EPS
    A = rng.random((20, 10))
    nrm = np.linalg.norm(A, 2)
    assert abs(gpu.snorm(A) - nrm) <= rtol * nrm
    A = rng.random((10, 10)); A = A + A.T
    nrm = np.linalg.norm(A, 2)
    assert abs(gpu.snorm(A) - nrm) <= rtol * nrm
    B = rng.random((10, 10))
    nrm = np.linalg.norm(A - B, 2)
    assert abs(gpu.snormdiff(A, B) - nrm) <= rtol * nrm


def test_snorm_large_gap(gpu):
    rng = np.random.default_rng(1)
    U, _ = np.linalg.qr(rng.standard_normal((3000, 50)))
    V, _ = np.linalg.qr(rng.standard_normal((2000, 50)))
    s = np.concatenate([[10.0], np.linspace(5, 1, 49)])  # gap large enough for 32 steps
    A = np.asfortranarray((U * s) @ V.T)
    assert abs(gpu.snorm(A) - 10.0) <= 1e-10


def test_snormdiff_id_matches_dense(gpu, orc):
    A = orc.hilbert(600)
    V = gpu.idfact(A, seed=2, rtol=1e-9)
    E = A[:, V.rd.cpu().numpy() - 1] - A[:, V.sk.cpu().numpy() - 1] @ V.T.cpu().numpy()
    ref = np.linalg.norm(E, 2)
    got = gpu.snormdiff(A, V, snorm_niter=200, rtol=1e-12)
    assert abs(got - ref) <= 1e-3 * ref + 1e-14


@pytest.mark.parametrize("m,n,k,pad", [
    (1, 1, 0, 0), (2, 3, 1, 0), (33, 70, 9, 1), (512, 100, 17, 0), (513, 99, 16, 0),
    (514, 4100, 33, 0),    # two row blocks of the products
    (1023, 30, 7, 1), (1024, 31, 7, 0),  # a wave per column, and a block
    (1026, 4097, 40, 1),   # odd leading dimension: 8-byte loads
    (700, 600, 600, 2),    # k = n: no T
    (20000, 17, 5, 0),     # tall; the iterate fits one block
    (40, 17000, 30, 0),    # the iterate longer than one block holds
])
def test_snormdiff_id_edges(gpu, m, n, k, pad):
    """snormdiff(A, V) and snorm(A - F) after a fixed number of steps from a given vector against
    the same power iteration in numpy.  Products are sums of at most m + n terms; their
    rounding reaches the estimate relative to |A| / |A - F|, bounded here by 1e3."""
    import torch
    rng = np.random.default_rng(m + n)
    A = np.zeros((m + pad, n))
    A[:m] = rng.standard_normal((m, n))
    Ad = torch.from_numpy(np.ascontiguousarray(A.T)).cuda().t()[:m]
    perm = rng.permutation(n)
    sk, rd = perm[:k], perm[k:]
    T = rng.standard_normal((k, n - k)) * 0.1
    V = gpu.IDPackedV(torch.from_numpy(sk + 1).cuda(), torch.from_numpy(rd + 1).cuda(),
                      gpu.to_device(np.asfortranarray(T)) if T.size else gpu.empty_colmajor(k, 0))
    x0 = rng.standard_normal(n)
    E = A[:m].copy()
    E[:, rd] -= A[:m][:, sk] @ T
    E[:, sk] = 0.0
    for what, M in (("diff", E), ("norm", A[:m])):
        x, s = x0.copy(), 1.0
        for _ in range(6):
            x = x / np.linalg.norm(x)
            x = M.T @ (M @ x)
            s = np.sqrt(np.linalg.norm(x))
            if s == 0:
                break
        if what == "diff":
            if k == 0:
                continue
            got = gpu.snormdiff(Ad, V, x0=x0, snorm_niter=6, rtol=0.0)
        else:
            got = gpu.snorm(Ad, x0=x0, snorm_niter=6, rtol=0.0)
        # (a 1 x 1 matrix is Hermitian: |A| itself, the same value)
        assert abs(got - s) <= 1e3 * 2.3e-16 * (m + n) ** 0.5 * max(s, 1e-300) + 1e-14 * (k == n), \
            (what, got, s)


def test_snorm_stops_with_the_reference(gpu):
    """The estimate is the one at which the reference's loop stops: the first step with
    |s - t| <= max(atol, t rtol), here after 1, 2, ... steps of a batch and in later batches."""
    rng = np.random.default_rng(8)
    U, _ = np.linalg.qr(rng.standard_normal((60, 60)))
    W, _ = np.linalg.qr(rng.standard_normal((50, 50)))
    A = np.asfortranarray((U[:, :50] * np.linspace(1.0, 0.05, 50)) @ W.T)
    x0 = rng.standard_normal(50)
    steps = []
    for rtol in (0.5, 0.1, 3e-2, 1e-2, 3e-3, 1e-3, 3e-4):
        x, s, t, it = x0.copy(), 1.0, 0.0, 0
        while s > 0 and abs(s - t) > t * rtol and it < 32:
            x = x / np.linalg.norm(x)
            x = A.T @ (A @ x)
            t, s, it = s, np.sqrt(np.linalg.norm(x)), it + 1
        steps.append(it)
        got = gpu.snorm(A, x0=x0, rtol=rtol)
        assert abs(got - s) <= 1e-13 * s, (rtol, it, got, s)
    assert min(steps) <= 4 and max(steps) > 4, steps
    assert gpu.snorm(A, x0=x0, snorm_niter=0) == 1.0
    assert gpu.snorm(A, x0=x0, atol=1.0) == 1.0
    assert gpu.snorm(np.zeros((4, 3)), x0=np.ones(3)) == 0.0
