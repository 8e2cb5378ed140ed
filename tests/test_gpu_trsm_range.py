"""Small triangular solves whose rows' elements differ in scale by more than
the range of a number: as substitution gives them, exactly (powers of two)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pairs(n, big, diag, b_first, b_second):
    """A lower triangle of independent pairs [[1, 0], [big, diag]] (a last odd
    row alone) and its right-hand side."""
    L, b = np.eye(n), np.full(n, b_first)
    for i in range(0, n - 1, 2):
        L[i + 1, i], L[i + 1, i + 1], b[i + 1] = big, diag, b_second
    return L, b


# (big, diag, b of the first row, b of the second, x of the second):
# big / diag overflows; big / diag is lost below the range
CASES = [(2.0 ** 665, 2.0 ** -465, 1.0, 2.0 ** 665, 0.0),
         (2.0 ** 665, 2.0 ** -465, 0.0, 2.0 ** -465, 1.0),
         (2.0 ** -665, 2.0 ** 465, 2.0 ** 1000, 3 * 2.0 ** 335, 2.0 ** -129)]


@pytest.mark.parametrize("uplo,trans", [("L", "N"), ("L", "T"), ("U", "N"), ("U", "T")])
@pytest.mark.parametrize("n,nrhs", [(2, 1), (63, 4), (64, 2), (100, 1), (130, 3)])
@pytest.mark.parametrize("case", CASES)
def test_rows_of_mixed_scale(lmx_gpu, case, n, nrhs, uplo, trans):
    big, diag, b1, b2, x2 = case
    L, b = pairs(n, big, diag, b1, b2)
    x = np.full(n, b1)
    x[1::2] = x2
    if (uplo == "U") != (trans == "T"):  # an upper system: the lower one reversed
        L, b, x = L[::-1, ::-1], b[::-1], x[::-1]
    T = np.ascontiguousarray(L.T if trans == "T" else L)
    B = np.ascontiguousarray(b[:, None] * 2.0 ** -np.arange(nrhs))
    X = lmx_gpu.trsm(T, B, uplo, trans, "N")
    np.testing.assert_array_equal(X, x[:, None] * 2.0 ** -np.arange(nrhs))


@pytest.mark.parametrize("n", [2, 64, 100])
def test_mixed_solve_of_rows_of_mixed_scale(lmx_gpu, n):
    # big / diag beyond FP32: the FP32 factor's solve has to stay finite, or
    # the refinement gives up and factors again in FP64
    L, b = pairs(n, 2.0 ** 83, 2.0 ** -50, 1.0, 2.0 ** 83)
    A, b = np.ascontiguousarray(L[::-1, ::-1]), b[::-1].copy()
    X, info = lmx_gpu.gesv_mixed(A, b[:, None])
    x = np.ones(n)
    x[1::2] = 0.0
    np.testing.assert_array_equal(np.asarray(X).reshape(n), x[::-1])
    assert info.fell_back == 0
