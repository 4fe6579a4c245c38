"""The product at the edges of the tiles, of the K chunks (128 and 32) and of the 16-wide pieces of
K: 32-wide tiles, and 64-wide ones at n = 1000 (one matrix takes them from n = 865 to 1024:
test_gpu_gemm_wide_tiles.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 17, 31, 33, 63, 65, 127, 129, 257, 1000, 1037])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_tile_edges(hip, n, ta, tb):
    rng = np.random.default_rng(n + 10 * ta + 20 * tb)
    A = np.asfortranarray(rng.standard_normal((n, n)))
    B = np.asfortranarray(rng.standard_normal((n, n)))
    opA, opB = (A.T if ta else A), (B.T if tb else B)
    C, ref = hip.la_gemm(A, B, ta, tb), opA @ opB
    # both sides sum n terms in FP64: n eps |A| |B| each, element by element
    bound = 2 * n * np.finfo(float).eps * (np.abs(opA) @ np.abs(opB))
    assert np.all(np.abs(C - ref) <= bound)
