"""The global-memory pivoted QR (sketches beyond the register-resident kernel): forced on the
oracle cases, against the register-resident kernel on the same sketch, and end to end on a
wide matrix whose adaptive rounds outgrow the register-resident kernel."""
import numpy as np
import pytest

from test_gpu_kernels import first_mismatch_ok, graded, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,rtol", [(40, 300, 1e-12), (72, 3000, 1e-10), (264, 2500, 1e-13),
                                      (12, 5, 0.0), (33, 700, 1e-6), (700, 400, 1e-12),
                                      (1032, 3000, 1e-10), (2056, 2500, 1e-12),
                                      (3500, 1200, 1e-12), (6000, 300, 1e-12)])
@pytest.mark.parametrize("fused", ["1", "0"])
def test_global_qrcp_vs_oracle(gpu, orc, monkeypatch, m, n, rtol, fused):
    """Both forms of the HBM path: one fused launch per step (columns in place, permuted at
    the end) and the two launches per step (LRA_QG_FUSED=0)."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    monkeypatch.setenv("LRA_QG_FUSED", fused)
    B = graded(m, n, m * 7 + n, decay=0.85 if m < 100 else 0.95)
    print(f"global geqp3_adap m={m} n={n} rtol={rtol} fused={fused}", flush=True)
    Bf, p_o, tau_o, k_o, gap = orc.geqp3_adap(B, -1, 0.0, rtol, 32, want_gap=True)
    Bd = gpu.to_device(B)
    p_g, tau_g, k_g = gpu.geqp3_adap(Bd, -1, 0.0, rtol, 32)
    torch.cuda.synchronize()
    p_g, tau_g, Bg = host(p_g), host(tau_g), host(Bd)
    ok, i = first_mismatch_ok(p_g, p_o, gap)
    assert ok, f"pivot mismatch at step {i} with gap {gap[i]}"
    if i == len(p_g):
        assert k_g == k_o
        kk = min(k_o, min(m, n))
        R_g, R_o = np.triu(Bg[:kk, :]), np.triu(Bf[:kk, :])
        assert np.abs(R_g - R_o).max() <= 1e-10 * np.abs(R_o).max()


def test_global_matches_register_kernel(gpu, monkeypatch):
    """The same 520 x 8192 sketch through both engines: same rank and pivots."""
    import torch
    B = graded(520, 8192, 11, decay=0.97)
    B1, B2 = gpu.to_device(B), gpu.to_device(B)
    p1, _, k1 = gpu.geqp3_adap(B1, -1, 0.0, 1e-10, 32)
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    p2, _, k2 = gpu.geqp3_adap(B2, -1, 0.0, 1e-10, 32)
    torch.cuda.synchronize()
    assert k1 == k2
    assert np.array_equal(host(p1)[:k1], host(p2)[:k2])
    R1, R2 = np.triu(host(B1)[:k1]), np.triu(host(B2)[:k2])
    assert np.abs(R1 - R2).max() <= 1e-10 * np.abs(R1).max()


@pytest.mark.parametrize("m,n,rtol,rank", [(2056, 3000, 1e-10, -1), (1032, 2600, 0.0, 700),
                                            (700, 5000, 1e-13, -1), (5000, 900, 1e-12, -1)])
def test_fused_matches_two_launch_form(gpu, monkeypatch, m, n, rtol, rank):
    """The fused HBM steps against the two-launch form on the same sketch: the same rank, the
    same pivots, R to rounding, and each reflector and tau to rounding amplified by the
    condition of its step, |R(0,0)| / |R(j,j)| (the two forms sum norms and dot products in
    different orders; graded columns, so no near ties); rank 700 ends inside a block
    (700 = 21 blocks of 32 + 28 steps)."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    B = graded(m, n, m + 3 * n, decay=0.97)
    out = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("LRA_QG_FUSED", fused)
        print(f"fused vs two-launch m={m} n={n} rtol={rtol} rank={rank} fused={fused}", flush=True)
        Bd = gpu.to_device(B)
        p, tau, k = gpu.geqp3_adap(Bd, rank, 0.0, rtol, 32)
        torch.cuda.synchronize()
        out[fused] = (host(p), host(tau), k, host(Bd))
    (p1, t1, k1, B1), (p0, t0, k0, B0) = out["1"], out["0"]
    assert k1 == k0
    assert np.array_equal(p1, p0)
    kk = min(k1, m, n)
    scale = np.abs(B0[:kk]).max()
    assert np.abs(np.triu(B1[:kk]) - np.triu(B0[:kk])).max() <= 1e-11 * scale
    cond = np.abs(B0[0, 0]) / np.abs(np.diag(B0[:kk, :kk]))
    dv = np.abs(np.tril(B1[:, :kk], -1) - np.tril(B0[:, :kk], -1)).max(axis=0)
    assert np.all(dv <= 1e-12 * cond), int(np.argmax(dv / cond))
    assert np.all(np.abs(t1[:kk] - t0[:kk]) <= 1e-12 * cond)


def test_wide_matrix_beyond_register_kernel(gpu, orc):
    """400 x 16384 with rank ~380 at rtol 1e-12: the order-264 and order-520 rounds no longer
    fit the register-resident kernel (16384 columns), so they run on the global path; checked
    against the oracle with the same Omegas."""
    rng = np.random.default_rng(3)
    m, n, r = 400, 16384, 390
    U, _ = np.linalg.qr(rng.standard_normal((m, r)))
    V, _ = np.linalg.qr(rng.standard_normal((n, r)))
    s = 10.0 ** (-14 * np.arange(r) / (r - 1))
    A = np.asfortranarray((U * s) @ V.T)

    class DeviceOmega:
        def gaussian(self, rnd, rows, cols):
            return np.asfortranarray(gpu.gaussian(rows, cols, 4, rnd).cpu().numpy())

    V_g = gpu.idfact(A, rtol=1e-12, seed=4)
    V_o = orc.idfact("n", A, orc.LRAOptions().copy(rtol=1e-12), rand=DeviceOmega())
    print(f"wide: k={V_g.k} oracle k={V_o.k} rounds={V_g.rounds}", flush=True)
    assert V_g.rounds == V_o.rounds and V_g.rounds >= 4
    assert V_g.k == V_o.k
    first_bad = next((i for i, (a, b) in enumerate(zip(host(V_g.sk), V_o.sk)) if a != b), None)
    if first_bad is not None:
        assert V_o.gap[first_bad] < 1e-10
    e_g = np.linalg.norm(A[:, host(V_g.rd) - 1] - A[:, host(V_g.sk) - 1] @ host(V_g.T), 2)
    e_o = np.linalg.norm(A[:, V_o.rd - 1] - A[:, V_o.sk - 1] @ V_o.T, 2)
    assert e_g <= 10 * max(e_o, 1e-15)


def test_slow_decay_orders_1032_to_2600(gpu, orc):
    """3000 x 2600 with sigma_i = exp(-0.011 (i-1)): at rtol 1e-10 the rank is about 2090, so
    the adaptive rounds run to order 2056 (rejected, k reaches its target 2048) and then the
    whole 2600 columns; the orders 1032, 2056 and 2600 run on the global path.  Checked against
    the oracle with the same Omegas: rounds, rank (within one step: the diagonal falls by 1.1%
    per step near the threshold), pivots up to the first near-tie, error within 10x."""
    rng = np.random.default_rng(8)
    m, n = 3000, 2600
    U, _ = np.linalg.qr(rng.standard_normal((m, n)))
    V, _ = np.linalg.qr(rng.standard_normal((n, n)))
    s = np.exp(-0.011 * np.arange(n))
    A = np.asfortranarray((U * s) @ V.T)
    del U, V

    class DeviceOmega:
        def gaussian(self, rnd, rows, cols):
            return np.asfortranarray(gpu.gaussian(rows, cols, 2, rnd).cpu().numpy())

    print("slow decay 3000x2600: gpu idfact", flush=True)
    V_g = gpu.idfact(A, rtol=1e-10, seed=2)
    print(f"gpu k={V_g.k} rounds={V_g.rounds}; oracle", flush=True)
    V_o = orc.idfact("n", A, orc.LRAOptions().copy(rtol=1e-10), rand=DeviceOmega())
    print(f"oracle k={V_o.k} rounds={V_o.rounds}", flush=True)
    assert V_g.rounds == V_o.rounds == 8
    assert abs(V_g.k - V_o.k) <= 1 and 2048 <= V_o.k < n
    sk_g = host(V_g.sk)
    first_bad = next((i for i, (a, b) in enumerate(zip(sk_g, V_o.sk)) if a != b), None)
    if first_bad is not None:
        assert V_o.gap[first_bad] < 1e-10, (first_bad, V_o.gap[first_bad])
    e_g = np.linalg.norm(A[:, host(V_g.rd) - 1] - A[:, sk_g - 1] @ host(V_g.T), 2)
    e_o = np.linalg.norm(A[:, V_o.rd - 1] - A[:, V_o.sk - 1] @ V_o.T, 2)
    assert e_g <= 10 * max(e_o, 1e-15)
    assert e_g <= 1e3 * 1e-10


def _edge_matrix(kind, m, n, seed):
    rng = np.random.default_rng(seed)
    B = graded(m, n, seed, decay=0.99)
    if kind == "ties":          # every column of the same norm, many exactly equal
        B = np.asfortranarray(np.tile(rng.standard_normal((m, 4)), (1, (n + 3) // 4))[:, :n])
    elif kind == "lowrank":     # rank 37 exactly: zero residuals after 37 steps
        B = np.asfortranarray(rng.standard_normal((m, 37)) @ rng.standard_normal((37, n)))
    elif kind == "zeros":       # zero columns among the others
        B[:, ::3] = 0.0
    elif kind == "cliff":       # columns whose norm falls by 1e6 within a block
        u = rng.standard_normal((m, 5))
        B = np.asfortranarray(u @ rng.standard_normal((5, n)) + 1e-6 * rng.standard_normal((m, n)))
    elif kind == "huge":        # outside the range of the blocks: single steps
        B = np.asfortranarray(B * 1e148)
    elif kind == "tiny":
        B = np.asfortranarray(B * 1e-148)
    elif kind == "slow":        # 16-step blocks, norms recomputed (early dlaqps block ends)
        U, _ = np.linalg.qr(rng.standard_normal((m, min(m, n))))
        V, _ = np.linalg.qr(rng.standard_normal((n, min(m, n))))
        B = np.asfortranarray((U * np.exp(-0.03 * np.arange(min(m, n)))) @ V.T)
    elif kind == "steep":       # the pivots' own norms fall far enough to end dlaqps blocks
        U, _ = np.linalg.qr(rng.standard_normal((m, min(m, n))))
        V, _ = np.linalg.qr(rng.standard_normal((n, min(m, n))))
        B = np.asfortranarray((U * np.exp(-0.3 * np.arange(min(m, n)))) @ V.T)
    return B


@pytest.mark.parametrize("kind,m,n,rtol,rank", [
    ("graded", 40, 9, 0.0, -1), ("graded", 17, 300, 0.0, -1), ("slow", 700, 500, 1e-13, -1),
    ("slow", 1040, 700, 1e-9, -1), ("slow", 2100, 333, 1e-7, 200), ("slow", 3100, 260, 1e-7, -1),
    ("slow", 5000, 140, 0.0, 77), ("slow", 530, 1300, 1e-8, 33), ("ties", 200, 600, 0.0, 40),
    ("lowrank", 300, 700, 1e-10, -1), ("zeros", 300, 301, 1e-9, -1), ("cliff", 400, 640, 1e-9, -1),
    ("steep", 100, 60, 1e-8, -1), ("steep", 64, 200, 1e-7, -1), ("steep", 90, 75, 1e-9, -1),
    ("steep", 1100, 81, 1e-8, -1), ("huge", 300, 400, 1e-8, -1), ("tiny", 300, 400, 1e-8, -1)])
def test_blocks_match_single_steps(gpu, monkeypatch, kind, m, n, rtol, rank):
    """Blocks of steps against one launch per step on the same matrix: the same rank and pivots,
    all n positions (the columns past the rank included), R and the reflectors to rounding times
    the condition of their step.  Where columns tie or have no residual left, any order is a
    pivoted QR: there the product Q R is compared with the permuted matrix instead."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    B = _edge_matrix(kind, m, n, m + 5 * n)
    out = {}
    for block in ("1", "0"):
        monkeypatch.setenv("LRA_QG_BLOCK", block)
        print(f"blocks {kind} m={m} n={n} rtol={rtol} rank={rank} block={block}", flush=True)
        Bd = gpu.to_device(B).clone().t().contiguous().t()
        p, tau, k = gpu.geqp3_adap(Bd, rank, 0.0, rtol, 32)
        torch.cuda.synchronize()
        out[block] = (host(p), host(tau), k, host(Bd))
    (p1, t1, k1, B1), (p0, t0, k0, B0) = out["1"], out["0"]
    assert k1 == k0
    if kind in ("ties", "lowrank", "cliff"):
        assert np.array_equal(np.sort(p1), np.arange(1, n + 1))
        kk = k1
        V = np.tril(B1[:, :kk], -1) + np.eye(m, kk)
        X = np.zeros((m, n))
        X[:kk] = np.triu(B1[:kk])
        for j in range(kk - 1, -1, -1):
            X -= t1[j] * np.outer(V[:, j], V[:, j] @ X)
        E = X - B[:, p1 - 1]
        d = np.abs(np.diag(B1)[:kk])
        assert (d[1:] <= d[:-1] * (1 + 1e-7)).all()  # (the downdated norms' accuracy)
        tail = max(rtol * d[0] * np.sqrt(n * max(1, min(m, n) - kk)), 1e-12 * d[0])
        rest = 0.0 if kk < min(m, n) and rank >= 0 else np.linalg.norm(E[:, kk:], axis=0).max()
        assert np.abs(E[:, :kk]).max() <= 1e-12 * d[0] and rest <= 10 * tail
        return
    assert np.array_equal(p1, p0)
    kk = min(k1, m, n)
    scale = np.abs(B0[:kk]).max()
    assert np.abs(np.triu(B1[:kk]) - np.triu(B0[:kk])).max() <= 1e-11 * scale
    cond = np.abs(B0[0, 0]) / np.abs(np.diag(B0[:kk, :kk]))
    dv = np.abs(np.tril(B1[:, :kk], -1) - np.tril(B0[:, :kk], -1)).max(axis=0)
    assert np.all(dv <= 1e-12 * cond), int(np.argmax(dv / cond))
    assert np.all(np.abs(t1[:kk] - t0[:kk]) <= 1e-12 * cond)


def test_blocks_nan_column(gpu, monkeypatch):
    """A NaN column is never a pivot, in either form, and the others are factored alike."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    B = _edge_matrix("slow", 400, 300, 3)
    B[7, 11] = np.nan
    got = []
    for block in ("1", "0"):
        monkeypatch.setenv("LRA_QG_BLOCK", block)
        Bd = gpu.to_device(B).clone().t().contiguous().t()
        p, _, k = gpu.geqp3_adap(Bd, 60, 0.0, 1e-9, 32)
        torch.cuda.synchronize()
        got.append((host(p), k))
    assert got[0][1] == got[1][1] == 60
    assert np.array_equal(got[0][0][:60], got[1][0][:60]) and 12 not in got[0][0][:60]


@pytest.mark.parametrize("m,n", [(1040, 3758), (700, 9000), (530, 20000)])
def test_blocks_repeat_their_bits(gpu, monkeypatch, m, n):
    """Blocks of steps choose the same pivots and give the same bits each time, with 4, 16 and more
    positions a thread in the selection of their candidates (its norms in registers, or re-read)."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    rng = np.random.default_rng(m)
    B = rng.standard_normal((m, n)) * np.exp(-0.02 * np.arange(m))[:, None]
    ref = None
    for _ in range(6):
        Bd = gpu.to_device(np.asfortranarray(B))
        p, tau, k = gpu.geqp3_adap(Bd, -1, 0.0, 1e-7, 32)
        torch.cuda.synchronize()
        got = (host(p), host(tau)[:k], host(Bd))  # (tau past the rank is not written)
        ref = ref or got
        assert k == len(ref[1]) and k > 300
        for what, a, b in zip(("pivots", "tau", "factors"), got, ref):
            assert np.array_equal(a, b), (what, np.argwhere(a != b)[:4])


@pytest.mark.parametrize("m,n", [(8192, 264), (5000, 520), (4096, 200)])
def test_tall_sketches_take_single_steps(gpu, monkeypatch, m, n):
    """Sketches on which a block of steps costs more than the steps it holds (tall, with few columns)
    run in single steps: the bits of LRA_QG_BLOCK=0."""
    import torch
    monkeypatch.setenv("LRA_QRCP_GLOBAL", "1")
    rng = np.random.default_rng(m)
    B = (rng.standard_normal((m, n)) * np.exp(-0.01 * np.arange(n))) @ rng.standard_normal((n, n))
    out = []
    for block in (None, "0"):
        if block:
            monkeypatch.setenv("LRA_QG_BLOCK", block)
        Bd = gpu.to_device(np.asfortranarray(B))
        p, tau, k = gpu.geqp3_adap(Bd, 100, 0.0, 0.0, 32)
        torch.cuda.synchronize()
        out.append((k, host(p), host(tau)[:k], host(Bd)))
    assert out[0][0] == out[1][0] == 100
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("m,n,fall,rtol,env,opts", [
    (900, 700, 0.03, 1e-7, {"LRA_QRCP_GLOBAL": "1"}, {}),
    # rounds of 24, 48, ... columns: their stops and dlaqps blocks end inside blocks of 16
    (900, 800, 0.02, 1e-5, {"LRA_QRCP_GLOBAL": "1"}, {"nb": 24}),
    (700, 1200, 0.1, 1e-9, {"LRA_QRCP_GLOBAL": "1"}, {"nb": 40}),
    # orders 520 and 1032 that fit the register-resident grid, foreseen to fall slowly: there in
    # blocks or (LRA_QG_BLOCK=0) in that grid
    (1500, 1500, 0.015, 1e-4, {"LRA_QRCP_PAIR": "0"}, {}),
    (1300, 1900, 0.012, 1e-3, {"LRA_QRCP_PAIR": "0"}, {"nb": 36})])
@pytest.mark.parametrize("block", ["", "1"])
def test_blocks_in_adaptive_rounds(gpu, monkeypatch, m, n, fall, rtol, env, opts, block):
    """An adaptive ID in blocks and in single steps: rounds that are stopped at their target or at the
    rank inside a block, whose later steps are taken back.  The same rounds, rank, skeleton and order of the
    redundant columns, T to rounding (relative to its largest entry; R11's condition 1 / rtol)."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(m + n)
    r = min(m, n)
    U, V = (np.linalg.qr(rng.standard_normal((d, r)))[0] for d in (m, n))
    A = gpu.to_device((U * np.exp(-fall * np.arange(r))) @ V.T)
    out = []
    for b in (block, "0"):
        monkeypatch.setenv("LRA_QG_BLOCK", b)
        W = gpu.idfact(A, rtol=rtol, seed=6, **opts)
        out.append(((W.k, W.rounds), host(W.sk), host(W.rd), host(W.T)))
    (k1, s1, r1, T1), (k0, s0, r0, T0) = out
    assert k1 == k0 and k1[0] > 100
    assert np.array_equal(s1, s0) and np.array_equal(r1, r0)
    assert np.abs(T1 - T0).max() <= 1e-14 / rtol * np.abs(T0).max()


@pytest.mark.parametrize("m,n,fall,rtol", [(2999, 2999, 0.1, 1e-8), (4500, 4200, 0.2, 1e-8),
                                           (3000, 2500, 0.09, 1e-4), (5000, 4100, 0.03, 1e-3)])
def test_rounds_alone_and_in_pairs(gpu, monkeypatch, m, n, fall, rtol):
    """Which rounds share a launch (by size, or alone where a rejected round foresees the next one to
    be accepted) changes no result: the same ID as with every round alone, T to rounding."""
    rng = np.random.default_rng(m)
    r = min(m, n, 400)
    U, V = (np.linalg.qr(rng.standard_normal((d, r)))[0] for d in (m, n))
    A = gpu.to_device((U * np.exp(-fall * np.arange(r))) @ V.T)
    out = []
    for pair in ("1", "0"):
        monkeypatch.setenv("LRA_QRCP_PAIR", pair)
        W = gpu.idfact(A, rtol=rtol, seed=6)
        out.append(((W.k, W.rounds), host(W.sk), host(W.rd), host(W.T)))
    (k1, s1, r1, T1), (k0, s0, r0, T0) = out
    assert k1 == k0 and k1[0] > 32
    assert np.array_equal(s1, s0) and np.array_equal(r1, r0)
    assert np.abs(T1 - T0).max() <= 1e-13 / rtol * np.abs(T0).max()
