"""Kernels that only launches of many or of wide blocks reach, at sizes that are no
multiples of their tiles: 64-wide tiles of the products and of the inversions' updates, the
sweep kernels of large launches, of few wide blocks, and every size class's edge."""
import numpy as np
import pytest

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
    lay = backend.layout_from_params(par)
    return A, B, lay, backend.System(ctx, lay, A, B)


def _block_elimination(M, lay, b):
    """M^{-1} b by block LU down the degrees, refined twice."""
    from kore_amd import backend
    _, sizes, order = backend.layout_blocks(lay)
    off = np.concatenate([[0], np.cumsum(sizes)])
    M = M.tocsr()
    scale = 1.0 / abs(M).max(axis=1).toarray().ravel()
    P = M[order][:, order].tocsr()
    P.data *= np.repeat(scale[order], np.diff(P.indptr))
    block = lambda i, j: P[off[i]:off[i + 1], off[j]:off[j + 1]]  # noqa: E731
    nb = len(sizes)
    inv, low, up = [], [], []
    for k in range(nb):
        D = block(k, k).toarray()
        if k:
            low.append(block(k, k - 1))
            D = D - low[-1] @ (inv[-1] @ up[-1].toarray())
        inv.append(np.linalg.inv(D))
        if k + 1 < nb:
            up.append(block(k, k + 1))

    def once(r):
        r = (r * scale[:, None])[order]
        y = []
        for k in range(nb):
            v = r[off[k]:off[k + 1]]
            y.append(v - low[k - 1] @ (inv[k - 1] @ y[-1]) if k else v)
        x = [inv[-1] @ y[-1]]
        for k in range(nb - 2, -1, -1):
            x.append(inv[k] @ (y[k] - up[k] @ x[-1]))
        out = np.empty_like(r)
        out[order] = np.concatenate(x[::-1])
        return out

    x = once(b)
    for _ in range(2):
        x = x + once(b - M @ x)
    return x


def _check_solves(ctx, N, lmax, precision, columns):
    """Solves of a hydrodynamic system against block elimination on the host, 1e-10:
    one plain sweep in FP64, in complex64 at most six sweeps (each gains three
    digits and more)."""
    A, B, lay, S = _system(ctx, N=N, lmax=lmax)
    sigma = 0.4j
    rng = np.random.default_rng(N)
    b = rng.standard_normal((S.n, max(columns))) + 1j * rng.standard_normal((S.n, max(columns)))
    xr = _block_elimination(A - sigma * B, lay, b)
    S.factor(sigma, precision)
    for k in columns:
        print("case: large launches", N, lmax, "precision", precision, "columns", k, flush=True)
        x, info = S.solve(b[:, :k], ir_tol=1e-14, ir_maxit=0 if precision == 0 else 20)
        err = np.linalg.norm(x - xr[:, :k], axis=0) / np.linalg.norm(xr[:, :k], axis=0)
        print("  rel err", err, "sweeps", info.iterations, flush=True)
        assert err.max() <= 1e-10
        assert info.iterations == 1 if precision == 0 else info.iterations <= 6
    S.close()


@pytest.mark.parametrize("N", [115, 116, 117, 127, 129])
@pytest.mark.parametrize("precision", [0, 1])
def test_wide_sweeps(ctx, N, precision):
    """Launches of 115 blocks, of 400 workgroups and more: one below, at and one above
    the k that a full batch of loads needs (116) and the k of two batches."""
    _check_solves(ctx, N, 230, precision, (1, 2))


@pytest.mark.parametrize("N,lmax", [(300, 130), (437, 60)])
@pytest.mark.parametrize("precision", [0, 1])
def test_many_wide_blocks(ctx, N, lmax, precision):
    """65 blocks of 300 rows: products and rank-128 updates of 1536 tiles and more, so
    tiles of edge 64 in both types, with rows and columns left over; 437 rows: sweeps over
    several batches of an odd k."""
    _check_solves(ctx, N, lmax, precision, (1, 2, 5))


@pytest.mark.parametrize("N", [112, 113, 192, 289, 384, 511])
@pytest.mark.parametrize("precision", [0, 1])
def test_size_class_edges(ctx, N, precision):
    """Edges of the inversion's workgroup sizes; above 256 rows also sweeps of one and two
    columns on a few blocks, which hold all products of a launch in registers."""
    _check_solves(ctx, N, 6, precision, (1, 2))


@pytest.mark.parametrize("ns,nd", [(15, 97), (16, 127), (17, 128), (33, 129), (33, 161)])
def test_product_tiles_of_64(ctx, ns, nd):
    """V[:, d] = beta V[:, d] + alpha V[:, s] Q on 70 700 rows (no multiple of 16), in
    tiles of edge 64: more than 1536 of them, and at least 3.2 times as many of edge 32.
    Sums of at most 33 products: error below 1e-13 of the sum of their magnitudes."""
    from kore_amd import backend
    A, B, lay, S = _system(ctx, N=101, lmax=700)
    assert S.n % 16 and -(-S.n // 64) * -(-nd // 64) >= 1536
    assert -(-S.n // 32) * -(-nd // 32) >= 3.2 * -(-S.n // 64) * -(-nd // 64)
    print("case: product of", ns, "and", nd, "columns, rows", S.n, flush=True)
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
