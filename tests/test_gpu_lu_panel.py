"""The LU panel kernel at the edges of its workgroups (512 rows) and panels
(32 columns): exact factors of matrices whose pivots chain from column to
column, LAPACK's pivots on general ones, and rows of infinities."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16
SIZES = [1, 31, 33, 64, 127, 129, 511, 513, 545, 1025, 1537]


def chained(n, kind):
    """Integer matrices with |l_ij| <= 1 exact: a unit lower triangle of 0 / 1
    and an upper one of powers of two, rows permuted."""
    rng = np.random.default_rng(n)
    L = np.tril(rng.integers(0, 2, (n, n)).astype(float), -1) * (rng.random((n, n)) < 4.0 / n) + np.eye(n)
    # rows of L scaled to magnitudes below one half keep the planted pivots
    L = np.tril(L, -1) * 0.5 + np.eye(n)
    U = np.triu(rng.integers(-1, 2, (n, n)) * (rng.random((n, n)) < 4.0 / n), 1) + 4.0 * np.eye(n)
    perm = {"cyclic": np.roll(np.arange(n), 1), "reversed": np.arange(n)[::-1],
            "random": rng.permutation(n)}[kind]
    A = np.empty((n, n))
    A[perm] = L @ U
    return A, L, U, perm


@pytest.mark.parametrize("kind", ["cyclic", "reversed", "random"])
@pytest.mark.parametrize("n", SIZES)
def test_chained_pivots_exact(lmx_gpu, n, kind):
    A, L, U, perm = chained(n, kind)
    want = np.tril(L, -1) + U
    LU, ipiv, info = lmx_gpu.getrf(A)
    assert info == 0
    np.testing.assert_array_equal(lmx_gpu.swaps_to_perm(ipiv), perm)
    np.testing.assert_array_equal(LU, want)
    LU32, ipiv32, _ = lmx_gpu.sgetrf(A)
    np.testing.assert_array_equal(ipiv32, ipiv)
    np.testing.assert_array_equal(LU32.astype(float), want)


@pytest.mark.parametrize("n", SIZES)
def test_general_pivots_vs_lapack(lmx_gpu, n):
    A = np.random.default_rng(3 * n).uniform(-1, 1, (n, n))
    LU, ipiv, info = lmx_gpu.getrf(A)
    ref, piv = scipy.linalg.lu_factor(A)
    assert info == 0
    np.testing.assert_array_equal(ipiv, piv)
    # backward error of the factors: |PA - LU| <= 4 n eps (|L||U|)
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    R = A[lmx_gpu.swaps_to_perm(ipiv)] - L @ U
    assert np.all(np.abs(R) <= 4 * n * EPS * (np.abs(L) @ np.abs(U)))


@pytest.mark.parametrize("special", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("row,col", [(0, 3), (5, 0), (31, 31), (7, 7), (12, 20)])
def test_infinities_and_nan_as_unblocked_elimination(lmx_gpu, special, row, col):
    # one panel: every element sees the terms of the unblocked elimination, so
    # the special values end where its updates take them, and finished rows
    # and columns keep theirs
    n = 32
    A = np.random.default_rng(row + 40 * col).integers(-4, 5, (n, n)).astype(float)
    A[row, col] = special
    W = A.copy()
    piv = np.zeros(n, int)
    with np.errstate(all="ignore"):
        for j in range(n):
            p = j  # rawPivotSearch: strict >, from row j
            if not np.isnan(W[j, j]):
                for i in range(j + 1, n):
                    if abs(W[i, j]) > abs(W[p, j]):
                        p = i
            piv[j] = p
            W[[j, p]] = W[[p, j]]
            if W[j, j] != 0:
                W[j + 1:, j] /= W[j, j]
                W[j + 1:, j + 1:] -= np.outer(W[j + 1:, j], W[j, j + 1:])
    LU, ipiv, _ = lmx_gpu.getrf(A)
    np.testing.assert_array_equal(ipiv, piv)
    np.testing.assert_array_equal(np.isnan(LU), np.isnan(W))
    np.testing.assert_array_equal(np.isinf(LU), np.isinf(W))


@pytest.mark.parametrize("special", [np.inf, np.nan])
@pytest.mark.parametrize("n,row,col", [(545, 0, 3), (545, 540, 0), (1100, 5, 5), (1100, 700, 17), (1100, 1099, 31)])
def test_special_values_over_several_workgroups(lmx_gpu, special, n, row, col):
    # the first panel (32 columns, 512 rows a workgroup) against the unblocked
    # elimination of the same columns, in the final order of the rows
    A = np.random.default_rng(row + 40 * col).integers(-4, 5, (n, n)).astype(float)
    A[row, col] = special
    LU, ipiv, _ = lmx_gpu.getrf(A)
    W = A[:, :32].copy()
    with np.errstate(all="ignore"):
        for j in range(32):
            p = j
            if not np.isnan(W[j, j]):
                best = np.where(np.isnan(W[j:, j]), -1.0, np.abs(W[j:, j]))
                p = j + int(np.argmax(best))  # the lowest row of the largest
            assert ipiv[j] == p
            W[[j, p]] = W[[p, j]]
            if W[j, j] != 0:
                W[j + 1:, j] /= W[j, j]
                W[j + 1:, j + 1:] -= np.outer(W[j + 1:, j], W[j, j + 1:])
    for j in range(32, n):
        W[[j, ipiv[j]]] = W[[ipiv[j], j]]
    np.testing.assert_array_equal(np.isnan(LU[:, :32]), np.isnan(W))
    np.testing.assert_array_equal(np.isinf(LU[:, :32]), np.isinf(W))


@pytest.mark.parametrize("pad", [1, 2])
@pytest.mark.parametrize("n", [129, 545, 1025])
def test_chained_pivots_with_row_strides(lmx_gpu, n, pad):
    # rows that do not start on 16-byte boundaries, and a stride
    import torch
    A, L, U, perm = chained(n, "random")
    buf = torch.full((n * (n + pad) + 1,), 7.0, dtype=torch.float64, device="cuda")
    dA = buf[1:].view(n, n + pad)[:, :n]
    dA.copy_(torch.tensor(A))
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    lmx_gpu.getrf_dev(dA, ipiv, info)
    np.testing.assert_array_equal(lmx_gpu.swaps_to_perm(ipiv.cpu().numpy()), perm)
    np.testing.assert_array_equal(dA.cpu().numpy(), np.tril(L, -1) + U)
    assert bool((buf[1:].view(n, n + pad)[:, n:] == 7.0).all())
