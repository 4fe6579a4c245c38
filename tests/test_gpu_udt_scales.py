"""UDT of columns whose squared norm is subnormal or next to the overflow limit: the reflectors
stay the reference's (tau = xi / nu, v = x / xi, UDT.jl:216-334), which only lose the digits that
the squares lose."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one size for each number of rows per lane of the panel kernel, and its 8-column form
@pytest.mark.parametrize("n", [17, 40, 100, 200, 400, 600, 1030])
@pytest.mark.parametrize("scale", [1e-157, 1e-155, 1e-140, 1e140, 1e154])
def test_extreme_column_scales(hip, n, scale):
    rng = np.random.default_rng(n)
    # diagonally dominant: x1 is nearly ||x||, so that nu xi = ||x||^2 + |x1| ||x|| is twice the
    # squared norm, which stays below 1.5e308 for the largest scale
    X = np.asfortranarray(scale * (np.eye(n) + 0.02 * rng.standard_normal((n, n))))
    U, D, T, piv = hip.la_udt(X, True)
    assert np.isfinite(U).all() and np.isfinite(D).all() and np.isfinite(T).all()
    assert sorted(piv.tolist()) == list(range(n))
    # Householder QR loses 8 n eps; every square below the normal range is off by up to 2^-1075, so a
    # reflector's squared norm by n 2^-1075 / scale^2 of itself, and n reflectors follow each other
    tol = 8 * n * np.finfo(float).eps + 8 * n * n * (2.0 ** -1074 / scale / scale) / 2
    assert np.abs(U.T @ U - np.eye(n)).max() < tol
    err = np.linalg.norm(U @ ((D / scale)[:, None] * T) - X / scale, axis=0)
    assert (err <= tol * np.linalg.norm(X / scale, axis=0)).all()
    assert np.abs(np.tril(T[:, piv], -1)).max() == 0.0
