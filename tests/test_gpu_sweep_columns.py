"""Solve sweeps by column count and block size: one below, at and one above what a
group of k, a batch, a row tile or a size class of the sweep kernels holds."""
import numpy as np
import pytest
import scipy.sparse.linalg as sla

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from kore_amd import backend
    c = backend.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("N", [17, 31, 33, 127, 128, 129, 131, 161, 256, 257])
@pytest.mark.parametrize("precision", [0, 1])
def test_columns(ctx, N, precision):
    """Solves with 1 to 17 columns (17: two passes) on one factor against
    SuperLU, 1e-10 (the plain sweep in FP64, refined in complex64)."""
    from kore_amd import assembly, backend
    from kore_amd.params import Params
    par = Params(m=1, symm=1, Ek=1e-4, N=N, lmax=6)
    A, B, _ = assembly.assemble(par)
    S = backend.System(ctx, backend.layout_from_params(par), A, B)
    sigma = 0.4j
    rng = np.random.default_rng(N)
    b = rng.standard_normal((S.n, 17)) + 1j * rng.standard_normal((S.n, 17))
    xr = sla.splu((A - sigma * B).tocsc()).solve(b)
    S.factor(sigma, precision)
    for k in (1, 2, 3, 4, 5, 8, 9, 15, 16, 17):
        print("case: block size", N, "precision", precision, "columns", k, flush=True)
        x, _ = S.solve(b[:, :k], ir_tol=1e-14, ir_maxit=0 if precision == 0 else 20)
        err = np.linalg.norm(x - xr[:, :k], axis=0) / np.linalg.norm(xr[:, :k], axis=0)
        assert err.max() <= 1e-10
    S.close()


@pytest.mark.parametrize("N,lmax", [(63, 830), (64, 830), (65, 830), (77, 550)])
@pytest.mark.parametrize("precision", [0, 1])
def test_many_blocks(ctx, N, lmax, precision):
    """Sweeps with one and two columns over launches of few and of many
    workgroups, odd block sizes: residual of the refined solution, 1e-13 of
    |A - sigma B| |x| + |b| by rows (the refinement's own stopping size is
    1e-14 of the solution)."""
    from kore_amd import assembly, backend
    from kore_amd.params import Params
    par = Params(m=1, symm=1, Ek=1e-4, N=N, lmax=lmax)
    A, B, _ = assembly.assemble(par)
    S = backend.System(ctx, backend.layout_from_params(par), A, B)
    sigma = 0.4j
    M = (A - sigma * B).tocsr()
    rng = np.random.default_rng(N)
    b = rng.standard_normal((S.n, 2)) + 1j * rng.standard_normal((S.n, 2))
    S.factor(sigma, precision)
    for k in (1, 2):
        print("case: many blocks", N, lmax, "precision", precision, "columns", k, flush=True)
        x, _ = S.solve(b[:, :k], ir_tol=1e-14, ir_maxit=20)
        r = np.abs(b[:, :k] - M @ x) / (abs(M) @ np.abs(x) + np.abs(b[:, :k]))
        assert r.max() <= 1e-13
    S.close()
