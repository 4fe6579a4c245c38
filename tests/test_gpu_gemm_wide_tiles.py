"""The product on 64-wide tiles, which one matrix takes from n = 865 to 1024: remainders of K from 1
to 3, last K chunks of 1 to 3 steps in an even and an odd chunk, single-row edge tiles, FP64 and
FP32; and the sizes around it, which take 32-wide tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WIDE = [865, 866, 879, 895, 897, 929, 961, 963, 993, 1023, 1024]


def bounded(C, A, B, opA, opB, eps):
    # both sides sum n terms: n eps |A| |B| each, element by element
    n = len(A)
    return np.all(np.abs(C - opA @ opB) <= 2 * n * eps * (np.abs(opA) @ np.abs(opB)))


@pytest.mark.parametrize("n", [864, *WIDE, 1025])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_fp64(hip, n, ta, tb):
    rng = np.random.default_rng(n + 10 * ta + 20 * tb)
    A = np.asfortranarray(rng.standard_normal((n, n)))
    B = np.asfortranarray(rng.standard_normal((n, n)))
    C = hip.la_gemm(A, B, ta, tb)
    assert bounded(C, A, B, A.T if ta else A, B.T if tb else B, np.finfo(np.float64).eps)


@pytest.mark.parametrize("n", [1, 33, 865, 897, 963, 1023, 1025])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_fp32(hip, n, ta, tb):
    rng = np.random.default_rng(n + 10 * ta + 20 * tb)
    A = np.asfortranarray(rng.standard_normal((n, n)).astype(np.float32).astype(np.float64))
    B = np.asfortranarray(rng.standard_normal((n, n)).astype(np.float32).astype(np.float64))
    C = hip.la_gemm(A, B, ta, tb, precision="mixed")
    assert bounded(C, A, B, A.T if ta else A, B.T if tb else B, np.finfo(np.float32).eps)
