"""GEMM loads: several stages in flight, 16-byte loads at any element alignment,
rows clamped at the edge of the matrix.

Every configuration, at the edges of its tiles and stages (the first stages, the
last one short, one row or column past a tile), with odd leading dimensions and
bases.  What lies between the columns (rows m .. ld-1) is NaN and must not reach
C.  Bar: k eps |A||B| per entry (the error of a sum of k products).
"""
import ctypes

import pytest
import torch

import tmv_amd

pytestmark = pytest.mark.gpu

MN = [(1, 1), (31, 33), (64, 130), (129, 67), (257, 96)]
KS = [1, 3, 16, 17, 64, 95, 160, 289]


def operand(rows, cols, rm, pad, shift, dt, gen):
    """rows x cols in row- or column-major storage, NaN between its vectors."""
    ln, nv = (cols, rows) if rm else (rows, cols)
    ld = ln + pad
    buf = torch.full((shift + nv * ld + 8,), float("nan"), dtype=dt)
    v = buf[shift:shift + nv * ld].view(nv, ld)
    v[:, :ln] = torch.rand(nv, ln, dtype=dt, generator=gen) * 2 - 1
    val = v[:, :ln].double()
    return buf.cuda(), ld, (val if rm else val.t())


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("layouts", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (3, 1)])
def test_gemm_edges_every_config(dt, layouts, pad, shift):
    L = tmv_amd.lib()
    eb = 8 if dt == torch.float64 else 4
    fn = L.tmvx_gemm_cfg_f64 if eb == 8 else L.tmvx_gemm_cfg_f32
    eps = torch.finfo(dt).eps
    la, lb = layouts
    gen = torch.Generator().manual_seed(5)
    for m, n in MN:
        for k in KS:
            A, lda, a = operand(m, k, la, pad, shift, dt, gen)
            B, ldb, b = operand(k, n, lb, pad, shift, dt, gen)
            ref = (a @ b).cuda()
            bar = ((k + 2) * eps) * (a.abs() @ b.abs()).cuda() + eps * ref.abs()
            for cfg in range(L.tmvx_gemm_config_count(eb)):
                C = torch.full((n, m), float("nan"), dtype=dt, device="cuda")
                rc = fn(cfg, la, lb, m, n, k, 1.0, A.data_ptr() + shift * eb, lda,
                        B.data_ptr() + shift * eb, ldb, 0.0, C.data_ptr(), m,
                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
                assert rc == 0
                d = (C.t().double() - ref).abs()
                assert bool((d <= bar).all()), (cfg, m, n, k)


@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
@pytest.mark.parametrize("layouts", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_bits_do_not_depend_on_the_tile(dt, layouts):
    """Every configuration adds an entry's products in the same order, so a
    factorisation may take another tile beside a panel than alone."""
    L = tmv_amd.lib()
    eb = 8 if dt == torch.float64 else 4
    fn = L.tmvx_gemm_cfg_f64 if eb == 8 else L.tmvx_gemm_cfg_f32
    la, lb = layouts
    gen = torch.Generator().manual_seed(6)
    for m, n, k in ((130, 257, 256), (300, 200, 289), (64, 64, 31), (1100, 1030, 256)):
        A, lda, _ = operand(m, k, la, 0, 0, dt, gen)
        B, ldb, _ = operand(k, n, lb, 0, 0, dt, gen)
        C0 = (torch.rand(n, m, dtype=dt, generator=gen) * 2 - 1).cuda()
        first = None
        for cfg in range(L.tmvx_gemm_config_count(eb)):
            C = C0.clone()
            rc = fn(cfg, la, lb, m, n, k, -1.0, A.data_ptr(), lda, B.data_ptr(), ldb, 1.0,
                    C.data_ptr(), m, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            assert rc == 0
            if first is None:
                first = C
            assert torch.equal(C, first), (cfg, m, n, k)
