"""The work that programs give this library, as cases that can be timed.

Each case is one call sequence of a user's program through the public entry
points of ``tmv_amd``: matrix products, LU solves, the mixed-precision solve,
batches of small systems and their products, a differentiated batched solve,
complex solves and least squares by QR.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call,
``run(state)`` is one pass, ``work(case)`` the bytes and operations that a
pass cannot do without and ``exact(case, seed)`` its outputs in 64 bits.

Matrices that a pass overwrites (factors in place) are copied from the
state first: a program keeps A for its residuals and for the next step.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tmv_amd

_TYPES = {"f64": torch.float64, "f32": torch.float32,
          "c128": torch.complex128, "c64": torch.complex64}
_BYTES = {"f64": 8, "f32": 4, "c128": 16, "c64": 8}


def listed():
    return [
        # The smallest configuration: one product of a program that works
        # with matrices of a few hundred rows; launch and latency count.
        {"name": "gemm_f64_512", "kind": "gemm", "dtype": "f64", "m": 512, "n": 512, "k": 512,
         "a_rm": False, "b_rm": False},
        # The large product whose share of the FP64 peak is quoted.
        {"name": "gemm_f64_8192", "kind": "gemm", "dtype": "f64", "m": 8192, "n": 8192, "k": 8192,
         "a_rm": False, "b_rm": False},
        # An ordinary single-precision product: ragged sizes, A row-major
        # (A^T B of a column-major A, as in normal equations).
        {"name": "gemm_f32_ragged", "kind": "gemm", "dtype": "f32", "m": 3001, "n": 1777, "k": 2500,
         "a_rm": True, "b_rm": False},
        # x = b/A for one right-hand side: the small LU solve.
        {"name": "solve_f64_512", "kind": "solve", "dtype": "f64", "n": 512, "nrhs": 1,
         "trans": False},
        # The large LU solve with a few right-hand sides, pivoting exercised.
        {"name": "solve_f64_8192x16", "kind": "solve", "dtype": "f64", "n": 8192, "nrhs": 16,
         "trans": False},
        # Single precision, ragged, many right-hand sides, solved with the
        # transposed factors (b % A).
        {"name": "solve_f32_3001x64", "kind": "solve", "dtype": "f32", "n": 3001, "nrhs": 64,
         "trans": True},
        # The headline: FP32 factors and FP64 refinement of a dense system
        # with singular values spread over four decades.
        {"name": "mixed_16384", "kind": "mixed", "n": 16384, "nrhs": 1, "kappa": 1e4},
        # Thousands of independent small systems of mixed sizes, factored and
        # solved in one call (a finite-element or filter bank step).
        {"name": "batch_solve_f64_20000", "kind": "batch_solve", "dtype": "f64", "count": 20000,
         "nmin": 8, "nmax": 128, "rmax": 4},
        # The products that go with such a batch, in single precision.
        {"name": "batch_gemm_f32_20000", "kind": "batch_gemm", "dtype": "f32", "count": 20000,
         "nmin": 8, "nmax": 128},
        # A training step through a batched solve: factor, solve, adjoint
        # (the gradients of both operands).
        {"name": "train_f64_512x256", "kind": "train", "dtype": "f64", "count": 512, "n": 256,
         "nrhs": 1},
        # A complex LU solve (a frequency-domain system).
        {"name": "solve_c128_1000x4", "kind": "zsolve", "dtype": "c128", "n": 1000, "nrhs": 4,
         "trans": False},
        # Least squares by QR, the division of a matrix that is not square.
        {"name": "qr_f64_2000x500", "kind": "qr", "dtype": "f64", "m": 2000, "n": 500, "nrhs": 3},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "solve", "solve", "mixed", "batch_solve", "batch_gemm",
                       "train", "zsolve", "qr"])
    real = rng.choice(["f64", "f32"])
    if kind == "gemm":
        return {"kind": kind, "dtype": real, "m": _log(rng, 32, 8192), "n": _log(rng, 32, 8192),
                "k": _log(rng, 32, 8192), "a_rm": rng.random() < 0.4, "b_rm": rng.random() < 0.4}
    if kind == "solve":
        return {"kind": kind, "dtype": real, "n": _log(rng, 64, 8192), "nrhs": _log(rng, 1, 64),
                "trans": rng.random() < 0.4}
    if kind == "mixed":
        n = _log(rng, 512, 12000)
        return {"kind": kind, "n": n, "nrhs": _log(rng, 1, 16) if n <= 6000 else 1,
                "kappa": rng.choice([1e2, 1e3, 1e4])}
    if kind in ("batch_solve", "batch_gemm"):
        lo = _log(rng, 8, 64)
        case = {"kind": kind, "dtype": real, "count": _log(rng, 300, 20000), "nmin": lo,
                "nmax": _log(rng, lo, 128)}
        if kind == "batch_solve":
            case["rmax"] = rng.randint(1, 4)
        return case
    if kind == "train":
        return {"kind": kind, "dtype": real, "count": _log(rng, 32, 512), "n": _log(rng, 16, 256),
                "nrhs": rng.randint(1, 4)}
    if kind == "zsolve":
        return {"kind": kind, "dtype": rng.choice(["c128", "c64"]), "n": _log(rng, 64, 2000),
                "nrhs": _log(rng, 1, 16), "trans": rng.random() < 0.4}
    m = _log(rng, 128, 4000)
    return {"kind": kind, "dtype": real, "m": m, "n": _log(rng, 32, max(32, min(1000, m // 2))),
            "nrhs": _log(rng, 1, 16)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (int(seed) + 1))
    return g


def _uniform(g, *shape, dtype):
    """Entries uniform in [-1, 1] (real and imaginary parts for complex)."""
    if dtype.is_complex:
        part = torch.float64 if dtype == torch.complex128 else torch.float32
        return torch.view_as_complex(_uniform(g, *shape, 2, dtype=part))
    return torch.rand(*shape, generator=g, dtype=dtype, device="cuda").mul_(2).sub_(1)


def _normal(g, *shape, dtype):
    if dtype.is_complex:
        part = torch.float64 if dtype == torch.complex128 else torch.float32
        return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=part, device="cuda"))
    return torch.randn(*shape, generator=g, dtype=dtype, device="cuda")


def _matrix(g, m, n, dtype, row_major=False):
    t = _uniform(g, m, n, dtype=dtype) if row_major else _uniform(g, n, m, dtype=dtype).t()
    return t


def _square(g, n, dtype):
    """A square system, column-major.  Real double precision: uniform
    entries, whatever condition that gives.  Single precision and complex: n
    added on the diagonal, the equations then put in a random order, so that
    the system is well conditioned, every column needs an interchange and
    which one does not depend on how the size of a complex number is taken."""
    A = _uniform(g, n, n, dtype=dtype).t()
    if dtype != torch.float64:
        A.diagonal().add_(n)
        A = tmv_amd.colmajor(A[torch.randperm(n, generator=g, device="cuda")])
    return A


def _spread(g, n, kappa):
    """A = U diag(s) V^T, column-major, s log-spaced from 1 to 1/kappa in a
    random order, U and V orthogonal: cosine transforms with rows in random
    order and random signs."""
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    C = torch.cos((math.pi / n) * torch.outer(i + 0.5, i)).mul_(math.sqrt(2.0 / n))
    C[:, 0] *= math.sqrt(0.5)
    s = torch.logspace(0.0, -math.log10(kappa), n, dtype=torch.float64, device="cuda")
    s = s[torch.randperm(n, generator=g, device="cuda")]

    def rows():
        sign = torch.randint(0, 2, (n, 1), generator=g, device="cuda").double().mul_(2).sub_(1)
        return C[torch.randperm(n, generator=g, device="cuda")] * sign

    U = rows().mul_(s)
    V = rows()
    return (V @ U.t()).t()          # (U V^T) with unit stride down its columns


def _sizes(case):
    """The sizes of a batch: part of the case, the same for every seed."""
    r = np.random.RandomState(case["count"] * 131 + case["nmin"] * 7 + case["nmax"])
    ns = r.randint(case["nmin"], case["nmax"] + 1, size=case["count"]).astype(np.int32)
    nrhs = r.randint(1, case.get("rmax", 1) + 1, size=case["count"]).astype(np.int32)
    return ns, nrhs


def _by_size(ns, widths=None):
    """(n, width, indices) of the systems that share both."""
    widths = ns if widths is None else widths
    for n, w in sorted(set(zip(ns.tolist(), widths.tolist()))):
        yield n, w, np.nonzero((ns == n) & (widths == w))[0]


def _offsets(counts):
    return np.concatenate([[0], np.cumsum(counts.astype(np.int64))[:-1]])


def _blocks(off, size, device="cuda"):
    """Flat positions of blocks of `size` entries: one row per block."""
    return torch.as_tensor(off, device=device)[:, None] + torch.arange(size, device=device)


def _batch_matrices(g, ns, dtype):
    """Packed column-major blocks: uniform entries and n on the diagonal, the
    equations of each system in a random order."""
    flat = _uniform(g, int((ns.astype(np.int64) ** 2).sum()), dtype=dtype)
    off = _offsets(ns.astype(np.int64) ** 2)
    for n, _, who in _by_size(ns):
        order = torch.rand(len(who), n, generator=g, device="cuda").argsort(dim=1)
        at = torch.as_tensor(off[who], device="cuda")[:, None] + order + n * torch.arange(n, device="cuda")
        flat[at.reshape(-1)] += n       # column j's large entry sits in row order[j]
    return flat


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    dtype = _TYPES[case.get("dtype", "f64")]
    st = {"case": dict(case)}
    if kind == "gemm":
        st["A"] = _matrix(g, case["m"], case["k"], dtype, case["a_rm"])
        st["B"] = _matrix(g, case["k"], case["n"], dtype, case["b_rm"])
    elif kind in ("solve", "zsolve"):
        st["A"] = _square(g, case["n"], dtype)
        st["b"] = _normal(g, case["nrhs"], case["n"], dtype=dtype).t()
    elif kind == "mixed":
        st["A"] = _spread(g, case["n"], case["kappa"])
        st["b"] = _normal(g, case["nrhs"], case["n"], dtype=dtype).t()
    elif kind == "qr":
        st["A"] = _matrix(g, case["m"], case["n"], dtype)
        st["b"] = _normal(g, case["nrhs"], case["m"], dtype=dtype).t()
    elif kind == "batch_solve":
        ns, nrhs = _sizes(case)
        st["A"] = _batch_matrices(g, ns, dtype)
        st["b"] = _normal(g, int((ns.astype(np.int64) * nrhs).sum()), dtype=dtype)
        st["batch"] = tmv_amd.Batch(ns, nrhs, dtype=dtype)
        st["plan"] = tmv_amd.BatchPlan(st["batch"])
    elif kind == "batch_gemm":
        ns, _ = _sizes(case)
        total = int((ns.astype(np.int64) ** 2).sum())
        st["A"] = tmv_amd.Batch(ns, dtype=dtype, A=_uniform(g, total, dtype=dtype))
        st["B"] = tmv_amd.Batch(ns, dtype=dtype, A=_uniform(g, total, dtype=dtype))
        st["C"] = tmv_amd.Batch(ns, dtype=dtype)
    else:
        ns = np.full(case["count"], case["n"], dtype=np.int32)
        nrhs = np.full(case["count"], case["nrhs"], dtype=np.int32)
        nb = case["count"] * case["n"] * case["nrhs"]
        st["A"] = _batch_matrices(g, ns, dtype)
        st["b"] = _normal(g, nb, dtype=dtype)
        st["fact"] = tmv_amd.Batch(ns, nrhs, dtype=dtype)
        st["grad"] = tmv_amd.Batch(ns, nrhs, dtype=dtype)
        st["w"] = tmv_amd.Batch(ns, nrhs, dtype=dtype, A=st["grad"].A,
                                B=_normal(g, nb, dtype=dtype))
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemm":
        return tmv_amd.gemm(st["A"], st["B"])
    if kind == "solve":
        lu, x = st["A"].clone(), st["b"].clone()
        piv, info = tmv_amd.getrf(lu)
        tmv_amd.getrs(lu, piv, x, trans=case["trans"])
        return {"lu": lu, "piv": piv, "info": info, "x": x}
    if kind == "zsolve":
        lu, x = st["A"].clone(), st["b"].clone()
        piv, info = tmv_amd.getrf_complex(lu)
        tmv_amd.getrs_complex(lu, piv, x, trans=case["trans"])
        return {"lu": lu, "piv": piv, "info": info, "x": x}
    if kind == "mixed":
        # refined to what a double-precision solve gives
        x, info = tmv_amd.gesv_mixed(st["A"], st["b"], tol=1e-14)
        return {"x": x, "converged": info["converged"]}
    if kind == "qr":
        qr, x = st["A"].clone(), st["b"].clone()
        beta = tmv_amd.geqrf(qr)
        tmv_amd.geqrs(qr, beta, x)
        return {"qr": qr, "beta": beta, "x": x}
    if kind == "batch_solve":
        bt = st["batch"]
        bt.A.copy_(st["A"])
        bt.B.copy_(st["b"])
        info = tmv_amd.gesv_batched(st["plan"], bt)
        return {"lu": bt.A, "piv": bt.P, "info": info, "x": bt.B}
    if kind == "batch_gemm":
        a, b, c = st["A"], st["B"], st["C"]
        tmv_amd.gemm_batched(a.d_n, a.d_n, a.d_n, a.pA, b.pA, c.pA, dtype=a.dtype)
        return c.A
    fact, grad = st["fact"], st["grad"]
    fact.A.copy_(st["A"])
    fact.B.copy_(st["b"])
    info = tmv_amd.getrf_batched(fact)
    tmv_amd.getrs_batched(fact)
    tmv_amd.gesv_adjoint_batched(fact, fact, st["w"], grad, grad)
    return {"lu": fact.A, "piv": fact.P, "info": info, "x": fact.B, "grad_b": grad.B,
            "grad_a": grad.A}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    es = _BYTES[case.get("dtype", "f64")]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind in ("solve", "zsolve", "mixed"):
        n, r = case["n"], case["nrhs"]
        wide = 4 if kind == "zsolve" else 1
        lu = 1 if kind == "mixed" else 2
        return {"bytes": es * (lu * n * n + 2 * n * r) + (0 if kind == "mixed" else 8 * n),
                "flops": wide * (2 * n ** 3 / 3 + 2 * n * n * r)}
    if kind == "qr":
        m, n, r = case["m"], case["n"], case["nrhs"]
        return {"bytes": es * (2 * m * n + 2 * m * r + n),
                "flops": 2 * m * n * n - 2 * n ** 3 / 3 + r * (4 * m * n - n * n)}
    if kind in ("batch_solve", "batch_gemm"):
        ns, nrhs = (v.astype(np.float64) for v in _sizes(case))
        if kind == "batch_gemm":
            return {"bytes": float(es * 3 * (ns ** 2).sum()), "flops": float(2 * (ns ** 3).sum())}
        return {"bytes": float((es * (2 * ns ** 2 + 2 * ns * nrhs) + 8 * ns + 4).sum()),
                "flops": float((2 * ns ** 3 / 3 + 2 * ns * ns * nrhs).sum())}
    c, n, r = case["count"], case["n"], case["nrhs"]
    # A read, its factors and grad A written; b, w read, x and grad b written
    return {"bytes": c * (es * (3 * n * n + 4 * n * r) + 8 * n),
            "flops": c * (2 * n ** 3 / 3 + 6 * n * n * r)}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits, by torch alone
# ---------------------------------------------------------------------------

def _wide(t):
    return t.to(torch.complex128 if t.is_complex() else torch.float64)


def _lu_solve(A, b, trans):
    """(factors, solution) on the host, whose LAPACK pivots by the largest
    entry."""
    b = b.cpu()
    lu, piv = torch.linalg.lu_factor(A.cpu())
    if trans:                                   # A^T x = b: the conjugate of A^H conj(x) = conj(b)
        x = torch.linalg.lu_solve(lu, piv, b.conj().resolve_conj(), adjoint=True)
        return lu, x.conj().resolve_conj()
    return lu, torch.linalg.lu_solve(lu, piv, b)


def _exact_batch(ns, nrhs, A, b):
    """(flat factors, flat solutions) of packed systems."""
    A, b = A.cpu(), b.cpu()
    ns64 = ns.astype(np.int64)
    offa, offb = _offsets(ns64 ** 2), _offsets(ns64 * nrhs)
    lu, x = torch.empty_like(A), torch.empty_like(b)
    for n, r, who in _by_size(ns, nrhs):
        ia, ib = _blocks(offa[who], n * n, "cpu"), _blocks(offb[who], n * r, "cpu")
        M = A[ia].view(len(who), n, n).transpose(1, 2)
        f, s = _lu_solve(M, b[ib].view(len(who), r, n).transpose(1, 2), False)
        lu[ia] = f.transpose(1, 2).reshape(len(who), n * n)
        x[ib] = s.transpose(1, 2).reshape(len(who), n * r)
    return lu, x


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "gemm":
        return _wide(st["A"]) @ _wide(st["B"])
    if kind in ("solve", "zsolve"):
        lu, x = _lu_solve(_wide(st["A"]), _wide(st["b"]), case["trans"])
        return {"lu": lu, "piv": None, "info": None, "x": x}
    if kind == "mixed":
        return {"x": torch.linalg.solve(st["A"], st["b"]), "converged": None}
    if kind == "qr":
        qr, beta = torch.geqrf(_wide(st["A"]).cpu())
        n = case["n"]
        x = torch.ormqr(qr, beta, _wide(st["b"]).cpu(), left=True, transpose=True)
        x[:n] = torch.linalg.solve_triangular(qr[:n].triu(), x[:n], upper=True)
        return {"qr": qr, "beta": beta, "x": x}
    if kind == "batch_solve":
        ns, nrhs = _sizes(case)
        lu, x = _exact_batch(ns, nrhs, _wide(st["A"]), _wide(st["b"]))
        return {"lu": lu, "piv": None, "info": None, "x": x}
    if kind == "batch_gemm":
        ns, _ = _sizes(case)
        off = _offsets(ns.astype(np.int64) ** 2)
        A, B = _wide(st["A"].A), _wide(st["B"].A)
        C = torch.empty_like(A)
        for n, _, who in _by_size(ns):
            at = _blocks(off[who], n * n)
            # packed column-major blocks read row-major are the transposes: C^T = B^T A^T
            C[at] = torch.bmm(B[at].view(-1, n, n), A[at].view(-1, n, n)).view(-1, n * n)
        return C
    c, n, r = case["count"], case["n"], case["nrhs"]
    A = _wide(st["A"]).cpu().view(c, n, n).transpose(1, 2)
    b = _wide(st["b"]).cpu().view(c, r, n).transpose(1, 2)
    w = _wide(st["w"].B).cpu().view(c, r, n).transpose(1, 2)
    lu, piv = torch.linalg.lu_factor(A)
    x = torch.linalg.lu_solve(lu, piv, b)
    gb = torch.linalg.lu_solve(lu, piv, w, adjoint=True)
    # grad A = -grad b x^T; its transpose, row-major, is the packed column-major block
    ga = -(x @ gb.transpose(1, 2))
    return {"lu": lu.transpose(1, 2).reshape(-1), "piv": None, "info": None,
            "x": x.transpose(1, 2).reshape(-1), "grad_b": gb.transpose(1, 2).reshape(-1),
            "grad_a": ga.reshape(-1)}
