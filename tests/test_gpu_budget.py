"""Scratch memory that cannot be had."""
import pytest

pytestmark = pytest.mark.gpu


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
