"""A NaN anywhere in a block of columns reaches its column's norm and the
reported backward error, whichever row or column it stands in."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 8, 9, 16, 17, 70])
@pytest.mark.parametrize("n,row", [(1, 0), (40, 0), (40, 5), (40, 31), (40, 39), (300, 130)])
def test_scaled_residual_of_a_single_nan(lmx_gpu, n, row, k):
    rng = np.random.default_rng(n + k)
    A = rng.uniform(-1, 1, (n, n)) + 4 * np.eye(n)
    X = rng.uniform(-1, 1, (n, k))
    B = A @ X
    col = (3 * k) // 4
    B[row, col] = np.nan  # one element of one column; its residual alone is NaN
    eta = np.asarray(lmx_gpu.scaled_residual_linear(A, X, B))
    assert np.isnan(eta[col])
    assert np.all(np.delete(eta, col) <= 1)  # the others' are untouched


@pytest.mark.parametrize("precision", ["PREC_F32", "PREC_BF16"])
@pytest.mark.parametrize("k,col", [(1, 0), (9, 4), (64, 0), (70, 10)])
def test_mixed_solve_reports_a_nan_column(lmx_gpu, k, col, precision):
    n = 100
    rng = np.random.default_rng(k)
    A = rng.uniform(-1, 1, (n, n)) + 4 * np.sqrt(n) * np.eye(n)
    B = rng.uniform(-1, 1, (n, k))
    B[17, col] = np.nan
    X = np.zeros((n, k))
    ri = lmx_gpu.RefineInfo()
    lib = lmx_gpu.raw()
    lib.lmx_dgesv_mixed(getattr(lmx_gpu, precision), n, k, A.ctypes.data, n, B.ctypes.data, k, X.ctypes.data, k,
                        ctypes.byref(ri))
    assert np.isnan(ri.backward_error)
