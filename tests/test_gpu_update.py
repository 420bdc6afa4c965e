"""New values of A on a resident system: patterns small and large (one host
thread and several), with an entry stored twice, and refused column indices."""
import numpy as np
import pytest
import scipy.sparse as ss

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from kore_amd import backend
    c = backend.Context(0)
    yield c
    c.close()


def _matrices(N, lmax):
    from kore_amd import assembly, backend
    from kore_amd.params import Params
    par = Params(m=1, symm=1, Ek=1e-4, N=N, lmax=lmax)
    A, B, _ = assembly.assemble(par)
    return A.tocsr(), B.tocsr(), backend.layout_from_params(par)


def _solve(S):
    S.factor(0.4j, 0)
    b = np.random.default_rng(3).standard_normal(S.n) + 0j
    return S.solve(b, ir_maxit=0)[0]


@pytest.mark.parametrize("N,lmax", [(24, 40), (64, 120), (96, 200)])
@pytest.mark.parametrize("repeat", [False, True])
def test_update_equals_fresh(ctx, N, lmax, repeat):
    """An updated system solves exactly as one created from the new values
    (an entry stored twice counts as the sum of its two values)."""
    from kore_amd import backend
    A, B, lay = _matrices(N, lmax)
    data, ix, ip = A.data.copy(), A.indices.copy(), A.indptr.copy()
    if repeat:                                    # the last entry of every row once more, its value split in two
        last = ip[1:] - 1
        data = np.insert(data, ip[1:], 0.25 * data[last])
        data[np.arange(len(last)) + last] *= 0.75
        ix = np.insert(ix, ip[1:], ix[last])
        ip = ip + np.arange(len(ip))
    A1 = ss.csr_matrix((0.5 * data, ix, ip), shape=A.shape)
    A2 = ss.csr_matrix((data, ix, ip), shape=A.shape)
    print("case: update", N, lmax, "repeat", repeat, "entries", len(data), flush=True)
    S = backend.System(ctx, lay, A1, B)
    F = backend.System(ctx, lay, A2, B)
    S.update_a(data)
    assert S.nnz_a == len(data)
    assert np.array_equal(_solve(S), _solve(F))
    S.close()
    F.close()


@pytest.mark.parametrize("which", ["A", "B"])
@pytest.mark.parametrize("index", [-1, None])
def test_column_out_of_range(ctx, which, index):
    """A column index below zero or past the last column is refused (on the host)."""
    from kore_amd import backend
    A, B, lay = _matrices(24, 40)
    M = {"A": A.copy(), "B": B.copy()}
    M[which].indices = M[which].indices.copy()
    M[which].indices[len(M[which].indices) // 2] = A.shape[0] if index is None else index
    with pytest.raises(Exception, match="out of range"):
        backend.SystemPlan(lay, M["A"], M["B"])
