"""Panels of the UDT kernel at the sizes where its rows per lane, its pivot merge and its panel
width change: the pivot order against a plain replay of the reference's swaps (UDT.jl:216-334,
the w largest residual norms per panel), exactly, and U D T = X with zero and equal columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 200, 255, 257, 320, 511, 513, 1023, 1025, 1100]


def replayed_pivots(norms):
    """Slots of columns whose residual norms never change, panel after panel."""
    n = len(norms)
    slots = list(range(n))
    p0 = 0
    while p0 < n:
        w = min(16 if n - p0 <= 1024 else 8, n - p0)
        order = sorted(range(p0, n), key=lambda s: (-norms[slots[s]], s))[:w]
        chosen = [slots[s] for s in order]
        for t, c in enumerate(chosen):
            s = slots.index(c)
            slots[p0 + t], slots[s] = slots[s], slots[p0 + t]
        p0 += w
    return slots


@pytest.mark.parametrize("n", EDGES)
def test_pivot_order_is_the_reference_swaps(hip, n):
    # a scaled permutation matrix: orthogonal columns, so every residual norm is the column's own,
    # and powers of two, so every step is exact; few distinct norms, so most choices are ties
    rng = np.random.default_rng(n)
    s = 2.0 ** rng.integers(-2, 3, n)
    X = np.zeros((n, n), order="F")
    X[rng.permutation(n), np.arange(n)] = s
    U, D, T, piv = hip.la_udt(X, True)
    assert piv.tolist() == replayed_pivots(s)
    assert np.array_equal(D, s[piv])
    assert np.array_equal(U @ np.diag(D) @ T, X)


@pytest.mark.parametrize("n", EDGES[1:])
@pytest.mark.parametrize("kind", ["dense", "zeros", "equal"])
def test_reconstruction_at_panel_edges(hip, n, kind):
    rng = np.random.default_rng(5 * n)
    X = rng.standard_normal((n, n)) * 10.0 ** rng.uniform(-6, 6, n)[None, :]
    if kind == "zeros":
        X[:, rng.choice(n, max(1, n // 3), replace=False)] = 0.0
    elif kind == "equal":
        X = rng.choice([-1.0, 1.0], (n, n))
    X = np.asfortranarray(X)
    U, D, T, piv = hip.la_udt(X, True)
    assert sorted(piv.tolist()) == list(range(n))
    # Householder QR: the columns' relative error and U's loss of orthogonality are of order n eps
    tol = 8 * n * np.finfo(float).eps
    assert np.abs(U.T @ U - np.eye(n)).max() < tol
    scale = np.linalg.norm(X, axis=0)
    err = np.linalg.norm(U @ (D[:, None] * T) - X, axis=0)
    assert (err <= tol * np.where(scale > 0, scale, 1.0)).all()
    R = T[:, piv]
    assert np.abs(np.tril(R, -1)).max() == 0.0
