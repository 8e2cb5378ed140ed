"""Which kernel a product takes, by the timing family it is counted in, and
its exact result (integer operands) on both sides of the rule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def family(lmx, call):
    """The families among `gemm` (large tiles) and `gemm64` that call() used."""
    lmx.kernel_timing(True)
    try:
        lmx.kernel_timing_reset()
        call()
        return [f for f in ("gemm", "gemm64") if lmx.kernel_timing_get(f)[0] > 0]
    finally:
        lmx.kernel_timing(False)


# 64 x 64 tiles where 64 x 128 would multiply padding or fill a round of the
# 256 CUs badly: few columns, 129 - 192 columns, a grid just past a round, a
# small k; the wave-by-wave kernel where its tiles divide the output well
@pytest.mark.parametrize("m,n,k,tb,pad,want", [
    (16384, 1, 64, "N", 0, "gemm64"), (9001, 16, 300, "N", 1, "gemm64"), (30000, 64, 128, "N", 0, "gemm64"),
    (9000, 192, 256, "N", 0, "gemm64"), (17000, 50, 100, "T", 1, "gemm64"), (6000, 320, 500, "N", 0, "gemm64"),
    (1500, 1500, 64, "N", 0, "gemm64"),
    # a round of 64 x 64 tiles or less: the split-k kernel
    (16, 16, 8192, "N", 0, "gemm64"), (33, 300, 8000, "T", 1, "gemm64"), (500, 500, 2000, "N", 1, "gemm64"),
    (2000, 1000, 777, "N", 0, "gemm"), (4096, 1024, 512, "N", 1, "gemm"), (8192, 256, 256, "N", 0, "gemm")])
@pytest.mark.parametrize("ta", ["N", "T"])
def test_fp64_tiles(lmx_gpu, m, n, k, tb, pad, want, ta):
    import torch

    def operand(rows, cols, seed):
        v = torch.tensor(np.random.default_rng(seed).integers(-8, 9, (rows, cols)).astype(float), device="cuda")
        return torch.nn.functional.pad(v, (0, pad))[:, :cols]

    A = operand(*((k, m) if ta == "T" else (m, k)), 1)
    B = operand(*((n, k) if tb == "T" else (k, n)), 2)
    C = torch.empty(m, n, dtype=torch.float64, device="cuda")
    assert family(lmx_gpu, lambda: lmx_gpu.dgemm_dev(A, B, C, transa=ta, transb=tb)) == [want]
    a, b = A.cpu().numpy(), B.cpu().numpy()
    np.testing.assert_array_equal(C.cpu().numpy(), (a.T if ta == "T" else a) @ (b.T if tb == "T" else b))


# deep enough for the BF16 tiles of 128 (the first two) and 256, with remainders
# in m, n and k
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad,beta", [(1288, 1304, 2056, 0, 0.0), (1160, 2440, 2120, 8, 3.0),
                                            (3080, 3000, 1032, 0, 3.0), (2568, 4104, 904, 16, 0.0)])
def test_bf16_large_tiles_exact(lmx_gpu, m, n, k, pad, beta, ta, tb):
    import torch

    def operand(rows, cols, seed, dtype):
        v = torch.tensor(np.random.default_rng(seed).integers(-8, 9, (rows, cols)), device="cuda").to(dtype)
        return torch.nn.functional.pad(v, (0, pad))[:, :cols]

    A = operand(*((k, m) if ta == "T" else (m, k)), 1, torch.bfloat16)
    B = operand(*((n, k) if tb == "T" else (k, n)), 2, torch.bfloat16)
    C = operand(m, n, 3, torch.float32)
    a, b, c = A.double().cpu().numpy(), B.double().cpu().numpy(), C.double().cpu().numpy()
    lmx_gpu.gemm_bf16_dev(A, B, C, alpha=2.0, beta=beta, transa=ta, transb=tb)
    want = 2 * ((a.T if ta == "T" else a) @ (b.T if tb == "T" else b)) + beta * c
    np.testing.assert_array_equal(C.cpu().numpy().astype(float), want)
