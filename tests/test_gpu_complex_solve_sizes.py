"""Complex solves above 2048 rows, where the vector in LDS takes several turns
of the workgroup, up to its largest order (4096), and above it, where column
sweeps in memory take over.

The factors are made, not computed: a unit lower and an upper triangle with
off-diagonal entries of at most 1 / n, so that both are well conditioned (their
inverses' norms are below e), and a random interchange list; B is formed from a
known X.  Bar: a substitution's forward error, n eps for each of the two
triangles and the product that formed B, with a factor 2 for complex
arithmetic: 6 n eps |X|."""
import numpy as np
import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n,nrhs,dtype", [
    (2050, 1, torch.complex128), (3001, 2, torch.complex64), (4095, 2, torch.complex128),
    (4096, 3, torch.complex128), (4096, 1, torch.complex64), (4097, 3, torch.complex128),
    (4097, 1, torch.complex64)])
def test_complex_solve_sizes(dev, n, nrhs, dtype, trans):
    print(f"complex solve n {n} nrhs {nrhs} {dtype} trans {trans}", flush=True)
    part = torch.float64 if dtype == torch.complex128 else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(n)
    g = np.random.default_rng(n)
    LU = torch.view_as_complex(torch.rand(n, n, 2, generator=gen, dtype=part, device="cuda") * 2 - 1)
    LU = (LU * (0.7 / n)).t()                        # column-major
    LU.diagonal().copy_(torch.from_numpy(np.exp(2j * np.pi * g.random(n)) * (1 + g.random(n))))
    piv = np.array([g.integers(k, n) for k in range(n)], dtype=np.int64)
    X = torch.from_numpy(g.uniform(-1, 1, (n, nrhs)) + 1j * g.uniform(-1, 1, (n, nrhs)))
    wide = LU.to(torch.complex128).contiguous()
    L, U = torch.tril(wide, -1) + torch.eye(n, dtype=torch.complex128, device="cuda"), torch.triu(wide)
    del wide

    def permuted(v, order):
        v = v.cpu().numpy().copy()
        for k in order:
            v[[k, piv[k]]] = v[[piv[k], k]]
        return torch.from_numpy(v).cuda()

    if trans:                                        # A^T = U^T L^T P
        B = U.t().contiguous() @ (L.t().contiguous() @ permuted(X, range(n)))
    else:                                            # A = P^-1 L U
        B = permuted(L @ (U @ X.cuda()), range(n - 1, -1, -1))
    x = tmv_amd.colmajor(B.to(dtype))
    tmv_amd.getrs_complex(LU, torch.from_numpy(piv).cuda(), x, trans=trans)
    err = (x.cpu().to(torch.complex128) - X).abs().max().item()
    assert err <= 6 * n * torch.finfo(part).eps * X.abs().max().item(), err


@pytest.mark.parametrize("n", [2050, 4096, 4097])
def test_complex_solve_singular(dev, n):
    """A zero on U's diagonal met by a non-zero entry is reported."""
    LU = torch.eye(n, dtype=torch.complex128, device="cuda").t()
    LU[n // 2, n // 2] = 0
    piv = torch.arange(n, device="cuda")
    x = torch.zeros(n, 1, dtype=torch.complex128, device="cuda")
    x[0] = 1
    tmv_amd.getrs_complex(LU, piv, x)
    assert x[0].item() == 1 and x[1:].abs().max().item() == 0
    x[n // 2] = 1
    with pytest.raises(tmv_amd.TmvxError):
        tmv_amd.getrs_complex(LU, piv, x)


@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n", [5, 40, 600, 2100, 4097])
def test_complex_zero_entry_takes_no_part(dev, n, trans, dtype):
    """A zero entry is skipped by the substitution: Inf and NaN in its column
    of the factors (or, transposed, its row) do not matter, and a zero on U's
    diagonal there is not reported.  Same bar as above."""
    g = np.random.default_rng(n)
    h = n // 2
    LU = ((g.uniform(-1, 1, (n, n)) + 1j * g.uniform(-1, 1, (n, n))) * (0.7 / n)).astype(np.complex64)
    np.fill_diagonal(LU, 1 + g.random(n))
    B = np.zeros((n, 2), np.complex128)
    if trans:
        B[h] = (1, -2j)             # U^T x = b: zero before row h
        clean = LU.copy()
        LU[: h, h:] = np.nan
        LU[0, 0] = 0
        clean[: h, h:] = 0
    else:
        B[h] = (1, -2j)             # L: row h alone; U: nothing below it
        LU[h + 1:, h] = 0
        clean = LU.copy()
        LU[1:, 0] = np.inf
        LU[: n - 1, n - 1] = np.nan
        LU[n - 1, n - 1] = 0
        clean[1:, 0] = clean[: n - 1, n - 1] = 0
        clean[n - 1, n - 1] = 1
    L, U = np.tril(clean, -1).astype(np.complex128) + np.eye(n), np.triu(clean).astype(np.complex128)
    print(f"complex zeros n {n} trans {trans} {dtype}", flush=True)
    x = tmv_amd.colmajor(torch.from_numpy(B).to(dtype).cuda())
    tmv_amd.getrs_complex(tmv_amd.colmajor(torch.from_numpy(LU).to(dtype).cuda()),
                          torch.arange(n, device="cuda"), x, trans=trans)
    X = x.cpu().numpy().astype(np.complex128)
    back = L @ (U @ X) if not trans else U.T @ (L.T @ X)
    part = torch.float64 if dtype == torch.complex128 else torch.float32
    assert np.abs(back - B).max() <= 6 * n * torch.finfo(part).eps * np.abs(B).max()
