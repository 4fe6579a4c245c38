"""rdivp is a substitution from 513 to 1024 rows, for any T: the residual stays of the size of the
roundings where a product with the diagonal blocks' inverses loses digits, and an infinite entry
leaves the columns before it alone (rdivp!, real.jl:198-226)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def system(n, size, rng, unit=True):
    """T with entries of the given size in its 16 x 16 diagonal blocks, weakly coupled."""
    T = np.triu(rng.standard_normal((n, n)), 1) / n
    for p in range(0, n, 16):
        b = T[p:p + 16, p:p + 16]
        b[...] = np.triu(size * rng.standard_normal(b.shape), 1)
    T += np.diag(rng.choice([-1.0, 1.0], n) * (1.0 if unit else rng.choice([0.3, 0.7, 1.5, 3.0], n)))
    dirty = np.asfortranarray(T + np.tril(rng.standard_normal((n, n)), -1))
    return T, dirty


@pytest.mark.parametrize("n", [513, 520, 640, 641, 1000, 1024])
@pytest.mark.parametrize("size,unit", [(1.0, True), (3.0, True), (10.0, True), (1.0, False)])
def test_backward_stable_with_large_blocks(hip, oracle, n, size, unit):
    rng = np.random.default_rng(n + int(size))
    T, dirty = system(n, size, rng, unit)
    A = np.asfortranarray(rng.standard_normal((n, n)))
    piv = rng.permutation(n).astype(np.int32)
    X = hip.la_rdivp(A, dirty, piv)
    # entries of size 10 take the solution itself out of range from some column on (n = 640: 553), by
    # the oracle's substitution: the columns up to there
    with np.errstate(all="ignore"):
        inside = (np.abs(oracle.rdivp(A, dirty, piv)) < 1e290).all(axis=0)
    k = n if inside.all() else int(np.argmin(inside))
    assert k == n or (size == 10.0 and k > 512)
    X, T, B = X[:, :k], T[:k, :k], A[:, piv[:k]]
    assert np.isfinite(X).all()
    # a column's sum has at most n terms and one quotient; as many roundings in the check
    bound = 2 * (n + 2) * np.finfo(float).eps * (np.abs(X) @ np.abs(T))
    assert np.all(np.abs(X @ T - B) <= bound)


@pytest.mark.parametrize("n", [520, 1024])
@pytest.mark.parametrize("where", [0, 5, 15, 16, 300, 511])
def test_infinite_entry_leaves_earlier_columns(hip, n, where):
    rng = np.random.default_rng(n + where)
    T, dirty = system(n, 0.5, rng)
    A = np.asfortranarray(rng.standard_normal((n, n)))
    piv = rng.permutation(n).astype(np.int32)
    X = hip.la_rdivp(A, dirty, piv)
    row = 37
    A2 = A.copy(order="F")
    A2[row, piv[where]] = np.inf
    Y = hip.la_rdivp(A2, dirty, piv)
    other = np.arange(n) != row
    assert np.array_equal(Y[other], X[other])
    assert np.array_equal(Y[row, :where], X[row, :where])
    assert np.isinf(Y[row, where])
