"""Factorisations of singular and of non-finite blocks: refused with the block and the
column of the first zero pivot, and the system is usable afterwards."""
import numpy as np
import pytest

from test_gpu_precision import _block_diagonal

pytestmark = pytest.mark.gpu

SIZES = [24, 64, 74, 100, 120, 150, 200, 300, 400]


@pytest.fixture(scope="module")
def ctx():
    from kore_amd import backend
    c = backend.Context(0)
    yield c
    c.close()


def _spoiled(A, rows, cols, value):
    """A with the stored entries of these rows and columns replaced."""
    C = A.copy()
    row = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    C.data = np.where(np.isin(row, rows) & np.isin(A.indices, cols), value, A.data)
    return C


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("precision", [0, 1])
def test_zero_columns(ctx, N, precision):
    """A zero column stays zero under elimination, so its pivot is the first zero one;
    the first block of a reduction's levels, blocks eliminated first and the last one."""
    from kore_amd import backend
    lay, A, D, at = _block_diagonal(N, 6, precision, N)
    S = backend.System(ctx, lay, A)
    for k, cols in ((0, [0]), (1, [7]), (2, [8]), (3, [N - 1]), (4, [min(31, N - 2), N - 1]), (5, [min(32, N - 1)]),
                    (1, [N // 2, N // 2 + 3])):
        print("case: zero columns", cols, "of block", k, "of", N, "rows, precision", precision, flush=True)
        S.update_a(_spoiled(A, at[k], at[k][cols], 0.0).data)
        with pytest.raises(backend.KoreError, match=r"zero pivot in degree block %d \(column %d\)" % (k, cols[0] + 1)):
            S.factor(0.0, precision)
        with pytest.raises(backend.KoreError):
            S.solve(np.ones(S.n))
    S.update_a(A.data)
    S.factor(0.0, precision)
    x = S.solve(np.ones(S.n), ir_tol=1e-14, ir_maxit=20)[0]
    assert np.linalg.norm(A @ x - 1) <= 1e-9 * np.linalg.norm(abs(A) @ np.abs(x))
    S.close()


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_entries(ctx, N, precision, value):
    """One entry that is no finite number: no pivot is taken from it, what it spreads to is
    refused as a zero pivot."""
    from kore_amd import backend
    lay, A, D, at = _block_diagonal(N, 6, precision, N)
    S = backend.System(ctx, lay, A)
    for k, i, j in ((0, 0, 0), (1, N // 2, 3), (2, 5, N - 1)):
        print("case:", value, "at", i, j, "of block", k, "of", N, "rows, precision", precision, flush=True)
        S.update_a(_spoiled(A, at[k][[i]], at[k][[j]], value).data)
        with pytest.raises(backend.KoreError, match="zero pivot"):
            S.factor(0.0, precision)
    S.update_a(A.data)
    S.factor(0.0, precision)
    S.close()
