"""Tile edges of the dense kernels: block sizes and products one below, at and
one above what a tile, a slab, a panel or a size class of the dispatch holds."""
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


def _system(ctx, **kw):
    from kore_amd import assembly, backend
    from kore_amd.params import Params
    par = Params(m=1, symm=1, Ek=1e-4, **kw)
    A, B, _ = assembly.assemble(par)
    return A, B, backend.System(ctx, backend.layout_from_params(par), A, B)


@pytest.mark.parametrize("ns,nd", [(1, 17), (4, 32), (15, 33), (16, 64), (17, 65), (33, 70)])
@pytest.mark.parametrize("size", ["small", "large"])
def test_product_tiles(ctx, size, ns, nd):
    """V[:, d] = beta V[:, d] + alpha V[:, s] Q against numpy: sums of at most
    33 products, so the error stays below 1e-13 of the sum of their magnitudes.
    960 rows take tiles of 32, 70 000 rows with nd >= 65 tiles of 64."""
    from kore_amd import backend
    A, B, S = _system(ctx, **(dict(N=24, lmax=40) if size == "small" else dict(N=100, lmax=700)))
    print("case: product", size, "rows", S.n, "ns", ns, "nd", nd, flush=True)
    rng = np.random.default_rng(ns * 100 + nd)
    V = rng.standard_normal((S.n, ns + nd)) + 1j * rng.standard_normal((S.n, ns + nd))
    Q = rng.standard_normal((ns, nd)) + 1j * rng.standard_normal((ns, nd))
    ws = backend.Workspace(S, ns + nd)
    ws.set(0, V)
    ws.gemm(ns, nd, 0, ns, Q, alpha=-0.5, beta=2.0)
    got = ws.get(ns, nd)
    ref = 2.0 * V[:, ns:] - 0.5 * (V[:, :ns] @ Q)
    mag = 2.0 * np.abs(V[:, ns:]) + 0.5 * (np.abs(V[:, :ns]) @ np.abs(Q))
    assert np.max(np.abs(got - ref) / mag) <= 1e-13
    ws.close()
    S.close()


@pytest.mark.parametrize("N", [17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 191, 193, 255, 256, 257,
                               383, 384, 385, 500, 511, 512])
@pytest.mark.parametrize("precision", [0, 1])
def test_block_size_edges(ctx, N, precision):
    """Factor and solve of six blocks of N rows against SuperLU, 1e-10 (the
    plain sweep in FP64, refined in complex64), as the other solve tests."""
    A, B, S = _system(ctx, N=N, lmax=6)
    sigma = 0.4j
    print("case: block size", N, "precision", precision, flush=True)
    rng = np.random.default_rng(N)
    b = rng.standard_normal((S.n, 2)) + 1j * rng.standard_normal((S.n, 2))
    S.factor(sigma, precision)
    x, _ = S.solve(b, ir_tol=1e-14, ir_maxit=0 if precision == 0 else 20)
    xr = sla.splu((A - sigma * B).tocsc()).solve(b)
    err = np.linalg.norm(x - xr, axis=0) / np.linalg.norm(xr, axis=0)
    print("  rel err", err, flush=True)
    assert err.max() <= 1e-10
    S.close()
