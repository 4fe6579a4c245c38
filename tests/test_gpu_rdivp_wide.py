"""rdivp from 513 to 1024 rows: around its limits and at ragged sizes, by the residual
X triu(T) = A[:, piv].  Large entries and infinities: test_gpu_rdivp_stability.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [512, 513, 528, 575, 640, 641, 1000, 1023, 1024])
def test_residual(hip, n):
    rng = np.random.default_rng(n)
    A = np.asfortranarray(rng.standard_normal((n, n)))
    T = np.triu(rng.uniform(-1.0, 1.0, (n, n)), 1) / np.sqrt(n) + np.diag(rng.choice([-1.0, 1.0], n))
    dirty = np.asfortranarray(T + np.tril(rng.standard_normal((n, n)), -1))
    piv = rng.permutation(n).astype(np.int32)
    X = hip.la_rdivp(A, dirty, piv)
    # a column is a sum of n products and a product with a 16 x 16 inverse whose entries stay
    # below 2 (entries of T below 1/sqrt(512)): n + 16 * 2 roundings, and as many in the check
    bound = 2 * (n + 32) * np.finfo(float).eps * (np.abs(X) @ np.abs(T))
    assert np.all(np.abs(X @ T - A[:, piv]) <= bound)
