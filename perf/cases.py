"""Workloads of the framework through its public entry points, for timing and comparing.

Kinds of case (`kind`), each with the sizes users bring:

  id       idfact(trans, A): matrices with sigma_i = exp(-decay (i-1)) and a noise floor
           below rtol, 200 to 8192 per side, square or tall, served at rtol 1e-6 or 1e-10
           (Gaussian sketch, adaptive rounds)
  srft     idfact with the SRFT sketch at a fixed rank on a tall matrix
  batched  one planned launch over many uneven far-field kernel blocks (C ABI, packed outputs)
  psvd     psvdfact of tall matrices;  pqr  pqrfact;  pheig  pheigfact of symmetric matrices
  zid      idfact of a ComplexF64 matrix
  apply    an ID's products with blocks of vectors, A X and A' Y
  errnorm  snormdiff(A, V): the spectral error of an ID, checked after a factorization
  sketch   the Gaussian sketch alone, at each precision the options offer
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
F64 = torch.float64


def package():
    name = "lowrankapprox_jl_amd"
    if name not in sys.modules:
        pkg = os.path.join(ROOT, "lowrankapprox.jl_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------------------- the cases

def listed():
    return [
        # one small request of a stream: rank 17, accepted in the first round; the time
        # is launches and latency
        {"name": "id_1024", "kind": "id", "m": 1024, "n": 1024, "decay": 0.7, "rtol": 1e-6,
         "trans": "n"},
        # a served request with odd sides, skeleton rows (trans c), rank 231
        {"name": "id_2999x1777_c", "kind": "id", "m": 2999, "n": 1777, "decay": 0.05,
         "rtol": 1e-6, "trans": "c"},
        # the throughput workload: 8192 x 8192, rtol 1e-10, rank 434
        {"name": "id_8192", "kind": "id", "m": 8192, "n": 8192,
         "decay": 9.0 * math.log(10.0) / 433.0, "rtol": 1e-10, "trans": "n"},
        # the slowest of the served distribution: rank 1152, sketches of 1032 and 2056 rows
        {"name": "id_3758_slow", "kind": "id", "m": 3758, "n": 3758, "decay": 0.01,
         "rtol": 1e-6, "trans": "n"},
        # the bandwidth-bound sketch: rank 300 of a tall matrix at order 310
        {"name": "srft_65536x4096", "kind": "srft", "m": 65536, "n": 4096, "decay": 0.025,
         "rank": 300, "over": 10},
        # the same on a row count with no power of two in it that the transform could use
        {"name": "srft_65000x4000", "kind": "srft", "m": 65000, "n": 4000, "decay": 0.025,
         "rank": 300, "over": 10},
        # thousands of off-diagonal kernel blocks of uneven sizes, planned once
        {"name": "batched_4096", "kind": "batched", "blocks": 4096, "rtol": 1e-8},
        # a served psvdfact request (tall), rank 231
        {"name": "psvd_5689x2048", "kind": "psvd", "m": 5689, "n": 2048, "decay": 0.05,
         "rtol": 1e-6},
        # the complex element type
        {"name": "zid_2048", "kind": "zid", "m": 2048, "n": 2048, "decay": 0.05, "rtol": 1e-6},
        # products of an ID with 64 vectors, both directions
        {"name": "apply_8192", "kind": "apply", "m": 8192, "n": 8192, "k": 436, "nrhs": 64},
        # the error check after an ID of the throughput workload's size
        {"name": "errnorm_8192", "kind": "errnorm", "m": 8192, "n": 8192, "k": 436},
        # a mixed-precision sketch
        {"name": "sketch_f32", "kind": "sketch", "m": 8192, "n": 8192, "order": 136,
         "trans": "n", "precision": "f32"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _logu(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["id", "id", "id", "id", "srft", "batched", "psvd", "pqr", "pheig", "zid",
                       "apply", "errnorm", "sketch"])
    m = _logint(rng, 200, 8192)
    n = m if rng.random() < 0.5 else _logint(rng, 200, m)
    if kind == "id":
        rtol = rng.choice([1e-6, 1e-6, 1e-10])
        # ranks up to 1152, as in the listed cases
        decay = _logu(rng, -math.log(10 * rtol) / 1151.0, 1.0)
        return {"kind": kind, "m": m, "n": n, "decay": decay, "rtol": rtol,
                "trans": rng.choice(["n", "c"])}
    if kind == "srft":
        rank = rng.randint(40, 300)
        return {"kind": kind, "m": _logint(rng, 4096, 60000), "n": _logint(rng, 512, 3500),
                "decay": _logu(rng, 0.02, min(0.2, 13.8 / rank)), "rank": rank,
                "over": rng.choice([8, 10])}
    if kind == "batched":
        return {"kind": kind, "blocks": _logint(rng, 64, 2048), "rtol": 1e-8}
    if kind in ("psvd", "pqr", "zid"):
        top = 2048 if kind == "zid" else 6000
        m = _logint(rng, 200, top)
        n = _logint(rng, 100, min(m, 3001))
        return {"kind": kind, "m": m, "n": n,
                "decay": _logu(rng, 0.05 if kind != "pqr" else 0.02, 0.3), "rtol": 1e-6}
    if kind == "pheig":
        return {"kind": kind, "m": _logint(rng, 200, 3001), "decay": _logu(rng, 0.08, 0.3),
                "rtol": 1e-6}
    if kind == "apply":
        return {"kind": kind, "m": m, "n": n, "k": _logint(rng, 10, min(n // 2, 436)),
                "nrhs": _logint(rng, 1, 256)}
    if kind == "errnorm":
        return {"kind": kind, "m": m, "n": n, "k": _logint(rng, 10, min(n // 2, 436))}
    return {"kind": kind, "m": m, "n": n, "order": _logint(rng, 16, min(520, m, n)),
            "trans": rng.choice(["n", "c"]),
            "precision": rng.choice(["f64", "f32", "bf16x3", "bf16"])}


# ------------------------------------------------------------------------------- the inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=F64):
    return torch.randn(*shape, dtype=dtype, device=DEV, generator=g)


def _decaying(case, seed, dtype=F64):
    """m x n column-major: Gaussian factors around a spectrum sigma_i = exp(-decay (i-1)) for
    the rank's values, and a noise floor that starts at rtol / 10 and decays on to 1e-17."""
    m, n = case["m"], case.get("n", case["m"])
    g = _gen(seed)
    sig = _spectrum(case, min(m, n))
    r = len(sig)
    U, V = _randn(g, m, r, dtype=dtype), _randn(g, n, r, dtype=dtype)
    return (V @ (U * (sig / math.sqrt(m * n))).mH).t()


def _spectrum(case, most):
    r = min(most, int(math.ceil(17 * math.log(10) / case["decay"])) + 1)
    sig = torch.exp(-case["decay"] * torch.arange(r, dtype=F64, device=DEV))
    k = _rank(case)
    if "rtol" in case and k < r:
        sig[k:] = 0.1 * case["rtol"] * sig[:r - k]
    return sig


def _sizes(case):
    """Uneven block sizes round(64 16^U)."""
    rng = np.random.default_rng(case["blocks"])
    return np.rint(64 * 16.0 ** rng.random((case["blocks"], 2))).astype(int)


def _blocks(case, seed):
    """Off-diagonal blocks 1 / |x_i - y_j|, x in the unit cube and y in the cube three to the
    right."""
    mn = _sizes(case)
    g = _gen(seed)
    X = torch.rand(int(mn[:, 0].sum()), 3, device=DEV, dtype=F64, generator=g)
    Y = torch.rand(int(mn[:, 1].sum()), 3, device=DEV, dtype=F64, generator=g)
    Y[:, 0] += 3.0
    out, i, j = [], 0, 0
    for m, n in mn.tolist():
        out.append(torch.cdist(Y[j:j + n], X[i:i + m]).reciprocal_().t())
        i, j = i + m, j + n
    return out


def _known_id(case, seed, noise):
    """A = C [I T] P' + noise and the ID's parts, known without factoring."""
    m, n, k = case["m"], case["n"], case["k"]
    g = _gen(seed)
    perm = torch.randperm(n, device=DEV, generator=g)
    sk, rd = perm[:k].contiguous(), perm[k:].contiguous()
    Ct = _randn(g, k, m) * (torch.exp(-0.05 * torch.arange(k, dtype=F64, device=DEV))[:, None])
    Tt = _randn(g, n - k, k) * 0.3
    At = None
    if noise:
        At = _randn(g, n, m) * noise
        At[sk] += Ct
        At[rd] += Tt @ Ct
        Ct = At[sk].contiguous()
    return At, Ct, Tt, sk, rd


def _spd_like(case, seed):
    """n x n symmetric with eigenvalues of both signs decaying as exp(-decay i)."""
    n = case["m"]
    g = _gen(seed)
    lam = _spectrum(case, n) / n
    U = _randn(g, n, len(lam))
    lam[1::3] *= -1.0
    A = (U * lam) @ U.T
    return (0.5 * (A + A.T)).t()


def prepare(case, seed):
    lra, kind = package(), case["kind"]
    if kind in ("id", "pqr", "psvd", "srft"):
        return {"case": case, "seed": seed, "A": _decaying(case, seed)}
    if kind == "zid":
        return {"case": case, "seed": seed, "A": _decaying(case, seed, torch.complex128)}
    if kind == "pheig":
        return {"case": case, "seed": seed, "A": _spd_like(case, seed)}
    if kind == "batched":
        return _Batch(case, _blocks(case, seed), seed)
    if kind == "apply":
        _, Ct, Tt, sk, rd = _known_id(case, seed, 0.0)
        g = _gen(seed + (1 << 20))
        F = lra.ID(Ct.t(), lra.IDPackedV(sk + 1, rd + 1, Tt.t()))
        return {"case": case, "F": F, "X": _randn(g, case["nrhs"], case["n"]).t(),
                "Y": _randn(g, case["nrhs"], case["m"]).t()}
    if kind == "errnorm":
        At, _, Tt, sk, rd = _known_id(case, seed, 1e-6)
        x0 = np.random.default_rng(seed).standard_normal(case["n"])
        return {"case": case, "A": At.t(), "V": lra.IDPackedV(sk + 1, rd + 1, Tt.t()), "x0": x0}
    g = _gen(seed)
    return {"case": case, "seed": seed, "A": _randn(g, case["n"], case["m"]).t()}


class _Batch:
    """A plan over blocks whose factors land in packed arrays, as an H-matrix code keeps them."""

    def __init__(self, case, blocks, seed):
        lra = package()
        L = lra._lib
        self.case, self.blocks, self.lib = case, blocks, L.load()
        nb = len(blocks)
        m = np.array([b.shape[0] for b in blocks], dtype=np.int64)
        n = np.array([b.shape[1] for b in blocks], dtype=np.int64)
        ldt = np.minimum(n, 72)
        at = np.concatenate([[0], np.cumsum(n)])
        att = np.concatenate([[0], np.cumsum(n * ldt)])
        self.k = np.zeros(nb, dtype=np.int64)
        self.sk = torch.zeros(int(at[-1]), dtype=torch.int64, device=DEV)
        self.rd = torch.zeros(int(at[-1]), dtype=torch.int64, device=DEV)
        self.T = torch.zeros(int(att[-1]), dtype=F64, device=DEV)
        self.ldt, self.at, self.att, self.m, self.n = ldt, at, att, m, n
        arr = ctypes.c_void_p * nb
        opts = lra.LRAOptions(rtol=case["rtol"], seed=seed, pqrfact_retval="t").to_c()
        A = arr(*[b.data_ptr() for b in blocks])
        sk = arr(*[self.sk.data_ptr() + 8 * int(o) for o in at[:-1]])
        rd = arr(*[self.rd.data_ptr() + 8 * int(o) for o in at[:-1]])
        T = arr(*[self.T.data_ptr() + 8 * int(o) for o in att[:-1]])
        self.ctx = lra.context()
        self.h = ctypes.c_void_p()
        cast = lambda v: ctypes.cast(v, ctypes.c_void_p)  # noqa: E731
        L.check(self.lib.lra_idfact_batched_plan(
            self.ctx.h, nb, m.ctypes.data, n.ctypes.data, cast(A), m.ctypes.data,
            ctypes.byref(opts), cast(sk), cast(rd), cast(T), ldt.ctypes.data,
            ctypes.byref(self.h)), "lra_idfact_batched_plan")
        self.check = L.check

    def run(self):
        left = ctypes.c_int64(0)
        self.check(self.lib.lra_idfact_batched_launch(self.h), "lra_idfact_batched_launch")
        self.check(self.lib.lra_idfact_batched_finish(self.h, self.k.ctypes.data,
                                                      ctypes.byref(left)),
                   "lra_idfact_batched_finish")
        return {"k": self.k, "sk": self.sk, "rd": self.rd, "T": self.T}

    def __del__(self):
        if self.h:
            self.lib.lra_idfact_batched_plan_destroy(self.h)


def run(state):
    if isinstance(state, _Batch):
        return state.run()
    lra, case = package(), state["case"]
    kind = case["kind"]
    if kind in ("id", "zid"):
        V = lra.idfact(case.get("trans", "n"), state["A"], rtol=case["rtol"], seed=state["seed"])
        return {"sk": V.sk, "rd": V.rd, "T": V.T}
    if kind == "srft":
        V = lra.idfact(state["A"], sketch="srft", rank=case["rank"], sketchfact_adap=False,
                       sketchfact_srft_samp=(1, case["over"]), rtol=1e-12, seed=state["seed"])
        return {"sk": V.sk, "rd": V.rd, "T": V.T}
    if kind == "pqr":
        F = lra.pqrfact(state["A"], rtol=case["rtol"], seed=state["seed"])
        return {"Q": F.Q, "R": F.R, "p": F.p}
    if kind == "psvd":
        F = lra.psvdfact(state["A"], rtol=case["rtol"], seed=state["seed"])
        return {"U": F.U, "S": F.S, "Vt": F.Vt}
    if kind == "pheig":
        F = lra.pheigfact(state["A"], rtol=case["rtol"], seed=state["seed"])
        return {"values": F.values, "vectors": F.vectors}
    if kind == "apply":
        return {"AX": state["F"].apply(state["X"]), "AtY": state["F"].apply(state["Y"], "c")}
    if kind == "errnorm":
        return np.float64(lra.snormdiff(state["A"], state["V"], x0=state["x0"]))
    return lra.sketch("left", case["trans"], state["A"], case["order"],
                      precision=case["precision"], seed=state["seed"])


# ------------------------------------------------------- what a pass needs, and its tolerance

def _rank(case):
    """The rank that rtol finds (the spectrum's values above 10 rtol)."""
    if "rank" in case:
        return case["rank"]
    most = min(case["m"], case.get("n", case["m"]))
    return max(1, min(int(0.8 * most), int(-math.log(10 * case["rtol"]) / case["decay"] + 1e-9) + 1))


def _id_work(m, n, k, nt, cplx=1):
    """One read of the matrix, one sketch of k + 8 rows, its pivoted QR to step k and the solve
    for T (a complex multiply-add is four real ones)."""
    ell = k + 8
    qr = 4.0 * (ell * nt * k - (ell + nt) * k * k / 2.0 + k ** 3 / 3.0)
    return {"bytes": 8.0 * cplx * (m * n + k * (nt - k)),
            "flops": (4 if cplx == 2 else 1) * (2.0 * ell * m * n + qr + float(k) * k * (nt - k))}


def work(case):
    kind = case["kind"]
    if kind == "batched":
        # ranks are about 33
        per = [_id_work(m, n, min(33, n), n) for m, n in _sizes(case).tolist()]
        return {k: sum(w[k] for w in per) for k in per[0]}
    m, n = case["m"], case.get("n", case["m"])
    if kind in ("id", "zid"):
        return _id_work(m, n, _rank(case), n if case.get("trans", "n") == "n" else m,
                        2 if kind == "zid" else 1)
    if kind == "srft":
        w = _id_work(m, n, case["rank"], n)
        ell = case["rank"] + case["over"]
        return {"bytes": w["bytes"], "flops": w["flops"] - 2.0 * ell * m * n
                + 2.5 * m * n * math.log2(ell)}
    if kind in ("pqr", "psvd", "pheig"):
        k = _rank(case)
        w = _id_work(m, n, k, n)
        qr = 4.0 * m * k * k  # the skeleton's QR and Q
        extra = k * k * n if kind == "pqr" else qr * n / m + 16.0 * k ** 3 + 2.0 * (m + n) * k * k
        if kind == "pheig":
            qr = 0.0
        return {"bytes": 8.0 * (m * n + k * (m + n)), "flops": w["flops"] + qr + extra}
    k = case.get("k", 0)
    if kind == "apply":
        r = case["nrhs"]
        return {"bytes": 2 * 8.0 * (m * k + k * (n - k) + r * (m + n)),
                "flops": 4.0 * r * (m * k + k * (n - k))}
    if kind == "errnorm":
        # 32 steps of the power iteration, each one product with A and one with A'
        return {"bytes": 32 * 2 * 8.0 * (m * n + m * k + k * (n - k)),
                "flops": 32 * 4.0 * (m * n + m * k + k * (n - k))}
    q = n if case["trans"] == "n" else m
    return {"bytes": 8.0 * (m * n + case["order"] * q), "flops": 2.0 * case["order"] * m * n}


def tolerance(case):
    """About four times the difference measured from the 64-bit form below, whose sums run in
    another order.  Factors of an ill-conditioned skeleton differ by its condition, 1/rtol,
    times the rounding of the sketch."""
    kind = case["kind"]
    if kind in ("id", "zid"):
        return {"rel": 5e-6 if case["rtol"] < 1e-9 else 3e-9, "differ": 0.0}
    if kind == "srft":
        return {"rel": 1e-15 * math.exp(case["decay"] * case["rank"]) + 1e-11, "differ": 0.0}
    if kind == "batched":
        return {"rel": 1e-7, "differ": 0.0}
    if kind in ("pqr", "psvd", "pheig"):
        return {"rel": 1e-9, "differ": 0.0}
    if kind == "apply":
        return {"rel": 1.5e-14}
    if kind == "errnorm":
        return {"rel": 1e-10}
    return {"rel": {"f64": 2e-14, "f32": 2.5e-6, "bf16x3": 2.5e-6, "bf16": 1e-2}[case["precision"]]}


# ----------------------------------------------------------- the same results in plain 64 bits

M32 = 0xFFFFFFFF


def _philox(pair, stream, seed, c3x=0):
    """Philox4x32-10 at counters `pair` (int64): four 32-bit words in int64."""
    c0, c1 = pair & M32, pair >> 32
    c2 = torch.full_like(pair, stream & M32)
    c3 = torch.full_like(pair, ((stream >> 32) & M32) ^ c3x)
    k0, k1 = seed & M32, (seed >> 32) & M32
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        h0, h1 = (p0 >> 32) & M32, (p1 >> 32) & M32
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, p1 & M32, h0 ^ c3 ^ k1, p0 & M32
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c0, c1, c2, c3


def _normals(count, stream, seed):
    """Normals #0 .. count-1 of a stream (Box-Muller on 53-bit uniforms)."""
    x = _philox(torch.arange((count + 1) // 2, dtype=torch.int64, device=DEV), stream, seed)
    u1 = (((x[0] << 21) | (x[1] >> 11)).to(F64) + 1.0) * 2.0 ** -53
    u2 = ((x[2] << 21) | (x[3] >> 11)).to(F64) * 2.0 ** -53
    rad = torch.sqrt(-2.0 * torch.log(u1))
    z = torch.stack([rad * torch.cos(2 * math.pi * u2), rad * torch.sin(2 * math.pi * u2)], 1)
    return z.reshape(-1)[:count]


def _omega(rows, cols, stream, seed):
    return _normals(rows * cols, stream, seed).reshape(cols, rows).t()


def _pqr_steps(B, n, rtol, nb, stop_after, rank=-1):
    """Pivoted QR of G matrices at once (G x ell x N, zero beyond n[g] columns), with the
    reference's blocks of nb steps (a block also ends where a column norm fell by sqrt(tol3z)
    since it was last computed), its stop rule at block ends and its column swaps.  Returns
    (permutation, rank, R)."""
    G, ell, N = B.shape
    B = B.clone()
    lastrk = torch.clamp(n, max=ell)
    kmax = lastrk if rank < 0 else torch.clamp(lastrk, max=rank)
    top = int(kmax.max())
    drop = math.sqrt(1.0536712127723509e-08)
    perm = torch.arange(N, device=DEV).expand(G, N).clone()
    vn = torch.linalg.vector_norm(B, dim=1)
    vn2 = vn.clone()
    ptol = rtol * vn.max(1).values
    g = torch.arange(G, device=DEV)
    j0 = torch.zeros(G, dtype=torch.int64, device=DEV)
    jb = torch.clamp(kmax, max=nb)
    k = torch.full((G,), -1, dtype=torch.int64, device=DEV)
    diag = torch.zeros(G, top, dtype=F64, device=DEV)
    for s in range(top):
        live = k < 0
        c = torch.where(live, vn[:, s:].argmax(1) + s, s)
        for t in (perm, vn, vn2):
            a, b = t[:, s].clone(), t[g, c]
            t[g, c] = a
            t[:, s] = b
        a, b = B[:, :, s].clone(), B[g, :, c]
        B[g, :, c] = a
        B[:, :, s] = b
        x = B[:, s:, s]
        alpha, xn = x[:, 0].clone(), torch.linalg.vector_norm(x[:, 1:], dim=1)
        nrm = torch.hypot(alpha.abs(), xn)
        ph = torch.where(alpha == 0, torch.ones_like(alpha), alpha / alpha.abs())
        v = x.clone()
        v[:, 0] = alpha + ph * nrm
        vv = (v.abs() ** 2).sum(1)
        f = torch.where(vv > 0, 2.0 / vv, torch.zeros_like(vv))
        w = torch.einsum("gi,gij->gj", v.conj(), B[:, s:, s + 1:])
        B[:, s:, s + 1:] -= (f[:, None] * v)[:, :, None] * w[:, None, :]
        B[:, s, s] = -ph * nrm
        B[:, s + 1:, s] = 0
        diag[:, s] = nrm
        new = torch.linalg.vector_norm(B[:, s + 1:, s + 1:], dim=1)
        low = (new <= drop * vn2[:, s + 1:]) & (vn[:, s + 1:] > 0) & (s + 1 < lastrk)[:, None]
        vn[:, s + 1:] = new
        vn2[:, s + 1:] = torch.where(low, new, vn2[:, s + 1:])
        end = live & (low.any(1) | (s - j0 + 1 == jb) | (s + 1 == kmax))
        small = diag[:, :s + 1] <= ptol[:, None]
        inside = torch.arange(s + 1, device=DEV)[None, :] >= j0[:, None]
        first = torch.where(small & inside, torch.arange(s + 1, device=DEV), N).min(1).values
        k = torch.where(end & small[:, s], first, k)
        k = torch.where(end & (k < 0) & (s + 1 == kmax), kmax, k)
        if stop_after > 0 and s + 1 >= stop_after:
            k = torch.where(end & (k < 0), s + 1, k)
        go = end & (k < 0)
        j0 = torch.where(go, s + 1, j0)
        jb = torch.where(go, torch.clamp(kmax - s - 1, max=nb), jb)
        if s % 8 == 7 and bool((k >= 0).all()):
            break
    return perm, k, B


def _solve_T(R, k, n):
    return torch.linalg.solve_triangular(R[:k, :k], R[:k, k:n], upper=True)


def _id_exact(A, rtol, seed, sketch=None, rank=-1):
    """(sk, rd, T) of A through the adaptive rounds (orders 40, 72, 136, ...), or one round of
    `sketch` at a fixed rank."""
    m, N = A.shape
    n = torch.tensor([N], device=DEV)
    target, rnd = 32, 0
    while True:
        if sketch is not None:
            B = sketch
        elif A.is_complex():
            z = _normals(2 * (target + 8) * m, rnd, seed).reshape(m, target + 8, 2)
            B = torch.view_as_complex(z).t() @ A
        else:
            B = _omega(target + 8, m, rnd, seed) @ A
        perm, k, R = _pqr_steps(B[None], n, rtol, 32, 0 if sketch is not None else target, rank)
        k = int(k[0])
        if sketch is not None or k < target:
            p = perm[0] + 1
            return p[:k], p[k:], _solve_T(R[0], k, N)
        target, rnd = 2 * target, rnd + 1


def _srft_exact(A, ell, seed):
    m = A.shape[0]
    x = _philox(torch.arange(m + ell, dtype=torch.int64, device=DEV), 0, seed, 0x5bd1e995)
    d = torch.where((x[0][:m] >> 31) > 0, 1.0, -1.0).to(F64)
    f = ((x[0][m:] * m + ((x[1][m:] * m) >> 32)) >> 32)
    B = torch.empty(ell, A.shape[1], dtype=F64, device=DEV)
    for j in range(0, A.shape[1], 256):
        Z = torch.fft.fft(d[:, None] * A[:, j:j + 256], dim=0)[f[0::2]]
        B[0::2, j:j + 256] = Z.real
        B[1::2, j:j + 256] = Z.imag[:ell // 2]
    return B


def _batch_exact(case, seed):
    blocks = _blocks(case, seed)
    sizes = np.array([b.shape[1] for b in blocks])
    ldt = np.minimum(sizes, 72)
    at = np.concatenate([[0], np.cumsum(sizes)])
    att = np.concatenate([[0], np.cumsum(sizes * ldt)])
    ks = np.zeros(len(blocks), dtype=np.int64)
    sk = torch.zeros(int(at[-1]), dtype=torch.int64, device=DEV)
    rd = torch.zeros_like(sk)
    T = torch.zeros(int(att[-1]), dtype=F64, device=DEV)
    top = max(b.shape[0] for b in blocks)
    left = [int(b) for b in np.argsort(sizes, kind="stable")]
    for rnd, target in ((0, 32), (1, 64)):
        om, again = _omega(target + 8, top, rnd, seed), []
        for q in range(0, len(left), 128):
            ids = left[q:q + 128]
            n = torch.tensor([sizes[b] for b in ids], device=DEV)
            B = torch.zeros(len(ids), target + 8, int(n.max()), dtype=F64, device=DEV)
            for i, b in enumerate(ids):
                B[i, :, :sizes[b]] = om[:, :blocks[b].shape[0]] @ blocks[b]
            perm, k, R = _pqr_steps(B, n, case["rtol"], 32, target)
            for i, b in enumerate(ids):
                kk, nn = int(k[i]), int(sizes[b])
                if kk >= target:
                    again.append(b)
                    continue
                ks[b] = kk
                sk[at[b]:at[b] + kk] = perm[i, :kk] + 1
                rd[at[b]:at[b] + nn - kk] = perm[i, kk:nn] + 1
                t = T[att[b]:att[b] + ldt[b] * (nn - kk)].reshape(nn - kk, int(ldt[b]))
                t[:, :kk] = _solve_T(R[i], kk, nn).t()
        left = again
    for b in left:
        s, r, t = _id_exact(blocks[b], case["rtol"], seed)
        kk, nn = len(s), int(sizes[b])
        ks[b] = kk
        sk[at[b]:at[b] + kk], rd[at[b]:at[b] + nn - kk] = s, r
        T[att[b]:att[b] + ldt[b] * (nn - kk)].reshape(nn - kk, int(ldt[b]))[:, :kk] = t.t()
    return {"k": ks, "sk": sk, "rd": rd, "T": T}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        return _batch_exact(case, seed)
    if kind in ("id", "zid"):
        A = _decaying(case, seed, torch.complex128 if kind == "zid" else F64)
        A = A if case.get("trans", "n") == "n" else A.mH
        return dict(zip(("sk", "rd", "T"), _id_exact(A, case["rtol"], seed)))
    if kind == "srft":
        A = _decaying(case, seed)
        B = _srft_exact(A, case["rank"] + case["over"], seed)
        return dict(zip(("sk", "rd", "T"), _id_exact(A, 1e-12, seed, B, case["rank"])))
    if kind in ("pqr", "psvd"):
        A = _decaying(case, seed)
        sk, rd, T = _id_exact(A, case["rtol"], seed)
        Q, R = np.linalg.qr(A[:, sk - 1].cpu().numpy())
        R = torch.from_numpy(R).to(DEV)
        W = torch.cat([R, R @ T], 1)
        if kind == "pqr":
            return {"Q": torch.from_numpy(Q), "R": W, "p": torch.cat([sk, rd])}
        S = np.linalg.svd(W.cpu().numpy(), compute_uv=False)
        # singular vectors carry the sign that the method gives them
        return {"U": None, "S": S[:max(1, int((S > case["rtol"] * S[0]).sum()))], "Vt": None}
    if kind == "pheig":
        A = _spd_like(case, seed)
        sk, rd, T = _id_exact(A, case["rtol"], seed)
        V = torch.cat([torch.eye(len(sk), dtype=F64, device=DEV), T], 1)
        R = np.linalg.qr(V.t().cpu().numpy(), mode="r")
        C = R @ A[sk - 1][:, sk - 1].cpu().numpy() @ R.T
        w = np.linalg.eigvalsh(0.5 * (C + C.T))
        return {"values": w[np.abs(w) > case["rtol"] * np.abs(w).max()], "vectors": None}
    if kind == "apply":
        _, Ct, Tt, sk, rd = _known_id(case, seed, 0.0)
        g = _gen(seed + (1 << 20))
        X, Y = _randn(g, case["nrhs"], case["n"]).t(), _randn(g, case["nrhs"], case["m"]).t()
        W = Ct @ Y
        Z = torch.empty(case["n"], case["nrhs"], dtype=F64, device=DEV)
        Z[sk], Z[rd] = W, Tt @ W
        return {"AX": Ct.t() @ (X[sk] + Tt.t() @ X[rd]), "AtY": Z}
    if kind == "errnorm":
        At, _, Tt, sk, rd = _known_id(case, seed, 1e-6)
        E = At[rd] - Tt @ At[sk]  # the skeleton's columns have no error
        x = np.random.default_rng(seed).standard_normal(case["n"])
        x = torch.from_numpy(x).to(DEV)
        s = 1.0
        for _ in range(32):
            x = x / x.norm()
            y = E.t() @ x[rd]
            x = torch.zeros_like(x)
            x[rd] = E @ y
            s = float(x.norm().sqrt())
        return np.float64(s)
    g = _gen(seed)
    A = _randn(g, case["n"], case["m"]).t()
    A = A if case["trans"] == "n" else A.t()
    return _omega(case["order"], A.shape[0], 0, seed) @ A
