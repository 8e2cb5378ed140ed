"""Triangular solves of small orders (one workgroup): every flag at the edges
of its 64-row blocks and of its range, against scipy's substitution."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu
EPS = 2.220446049250313e-16


def triangle(n, uplo, diag, seed):
    rng = np.random.default_rng(seed)
    T = rng.uniform(-1, 1, (n, n)) / max(n, 1)
    T = np.tril(T, -1) if uplo == "L" else np.triu(T, 1)
    # what lies in the other triangle, and a unit diagonal, is not read
    other = np.full((n, n), np.nan)
    T = T + np.where((np.tri(n, k=-1, dtype=bool) if uplo == "U" else np.tri(n, k=-1, dtype=bool).T), other, 0.0)
    np.fill_diagonal(T, np.nan if diag == "U" else rng.uniform(1, 2, n) * rng.choice([-1, 1], n))
    return T


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("diag", ["N", "U"])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (63, 3), (64, 4), (65, 1), (129, 2), (500, 4), (768, 1), (769, 1), (768, 5)])
def test_small_solves(lmx_gpu, n, nrhs, uplo, trans, diag):
    T = triangle(n, uplo, diag, n)
    B = np.random.default_rng(n + 1).uniform(-1, 1, (n, nrhs))
    X = lmx_gpu.trsm(T, B, uplo, trans, diag)
    M = np.nan_to_num(T, nan=0.0)
    if diag == "U":
        np.fill_diagonal(M, 1.0)
    want = scipy.linalg.solve_triangular(M, B, lower=uplo == "L", trans=trans)
    Op = M.T if trans == "T" else M
    # backward error of a substitution, row by row: (n + 4) eps |T||x|
    assert np.all(np.abs(Op @ X - B) <= 2 * (n + 4) * EPS * (np.abs(Op) @ np.abs(X) + np.abs(B)))
    assert np.all(np.abs(X - want) <= 1e-12 * np.abs(want).max())


@pytest.mark.parametrize("scale", [1e-200, 1e200])
def test_diagonals_beyond_the_reciprocals_range(lmx_gpu, scale):
    n = 100
    T = triangle(n, "L", "N", 5)
    M = np.nan_to_num(T, nan=0.0) * scale
    B = np.random.default_rng(6).uniform(-1, 1, (n, 2)) * scale
    X = lmx_gpu.trsm(M, B, "L", "N", "N")
    want = scipy.linalg.solve_triangular(M / scale, B / scale, lower=True)
    assert np.all(np.abs(X - want) <= 1e-12 * np.abs(want).max())


def test_two_solves_in_place_with_strides(lmx_gpu):
    import torch
    n, nrhs = 200, 3
    rng = np.random.default_rng(9)
    A = rng.uniform(-1, 1, (n, n)) + np.eye(n) * 20
    B = rng.uniform(-1, 1, (n, nrhs))
    dA = torch.tensor(np.pad(A, ((0, 0), (0, 7))), device="cuda")[:, :n]
    dB = torch.tensor(np.pad(B, ((0, 0), (0, 2)), constant_values=5.0), device="cuda")
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    lmx_gpu.gesv_dev(dA, ipiv, dB[:, :nrhs], info)
    X = dB.cpu().numpy()
    np.testing.assert_array_equal(X[:, nrhs:], 5.0)
    assert np.abs(X[:, :nrhs] - np.linalg.solve(A, B)).max() <= 1e-13
