"""GEMM dispatch at the edges of its tiles, through the device entry points:
integer operands, so every product and partial sum is exact in any order and
the result is compared bit for bit with the int64 product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def operands(torch, rows, cols, ld, offset, seed, dtype):
    """An integer matrix at a given row stride and element offset."""
    vals = np.random.default_rng(seed).integers(-8, 9, (rows, cols))
    buf = torch.full((offset + rows * ld,), 7.0, dtype=dtype, device="cuda")
    view = buf[offset:].view(rows, ld)[:, :cols]
    view.copy_(torch.tensor(vals, dtype=dtype))
    return vals, view


def check(torch, fn, dtype, cdtype, m, n, k, ta, tb, pad, offset, beta):
    va, A = operands(torch, *((k, m) if ta == "T" else (m, k)), (m if ta == "T" else k) + pad, offset, 1, dtype)
    vb, B = operands(torch, *((n, k) if tb == "T" else (k, n)), (k if tb == "T" else n) + pad, offset, 2, dtype)
    vc, C = operands(torch, m, n, n + pad, offset, 3, cdtype)
    fn(A, B, C, alpha=2.0, beta=beta, transa=ta, transb=tb)
    want = 2 * ((va.T if ta == "T" else va) @ (vb.T if tb == "T" else vb)) + int(beta) * vc
    np.testing.assert_array_equal(C.cpu().numpy().astype(np.int64), want)


# fewer 64 x 64 tiles than CUs: the split-k kernel, its three tiles, k below
# and above one chunk a wave, partial chunks, aligned and unaligned rows
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad,offset", [(1, 1, 48, 0, 0), (17, 15, 49, 1, 1), (100, 100, 100, 0, 0),
                                              (33, 70, 391, 3, 1), (256, 256, 64, 0, 0), (500, 500, 500, 0, 0),
                                              (1024, 64, 1024, 0, 0), (2000, 48, 1000, 2, 2)])
def test_split_k_exact(lmx_gpu, m, n, k, pad, offset, ta, tb):
    import torch
    check(torch, lmx_gpu.dgemm_dev, torch.float64, torch.float64, m, n, k, ta, tb, pad, offset, 3.0)
    check(torch, lmx_gpu.sgemm_dev, torch.float32, torch.float32, m, n, k, ta, tb, pad, offset, 0.0)


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("n,k", [(1, 64), (33, 100), (300, 777), (700, 49)])
def test_split_k_lower_tiles_exact(lmx_gpu, n, k, trans):
    import torch
    va, A = operands(torch, *((k, n) if trans == "T" else (n, k)), n if trans == "T" else k, 0, 4, torch.float64)
    C = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    lmx_gpu.syrk_dev(A, C, trans=trans)
    np.testing.assert_array_equal(C.cpu().numpy().astype(np.int64), va.T @ va if trans == "T" else va @ va.T)


# BF16 tiles of 128 and 256 (at least 100 tiles of 128), remainders in m, n
# and k; the last two shapes are not aligned for 16-byte vectors
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad", [(1288, 1304, 8, 0), (1288, 1280, 200, 8), (3080, 3000, 136, 0),
                                       (3072, 3072, 64, 16), (1288, 1304, 72, 4), (1290, 1301, 67, 0)])
def test_bf16_large_tiles_exact(lmx_gpu, m, n, k, pad, ta, tb):
    import torch
    check(torch, lmx_gpu.gemm_bf16_dev, torch.bfloat16, torch.float32, m, n, k, ta, tb, pad, 0, 3.0 if pad else 0.0)


# FP64 products on the wave-by-wave kernel (at least 140 tiles of 64 x 128):
# k below, at and past one chunk's multiples, unaligned rows, ragged edges
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad,offset", [(1153, 1025, 64, 0, 0), (1100, 1030, 65, 1, 1), (640, 1800, 100, 0, 0),
                                              (1999, 1001, 79, 2, 0), (1280, 1281, 96, 0, 1)])
def test_fp64_direct_exact(lmx_gpu, m, n, k, pad, offset, ta, tb):
    import torch
    check(torch, lmx_gpu.dgemm_dev, torch.float64, torch.float64, m, n, k, ta, tb, pad, offset, 3.0 if pad else 0.0)
