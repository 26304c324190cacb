"""Products over operands split into bf16 terms once (csrc/gemm_planes.hip), at sizes where each of its tiles is chosen:
edges that no tile divides, a last block of k that is part empty, rows that are no multiple of 16 bytes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


@pytest.mark.parametrize("precision,tol", [("bf16x6", 2.0 ** -20), ("bf16x3", 2.0 ** -15), ("bf16", 2.0 ** -7)])
@pytest.mark.parametrize("m,n,k", [(73, 2786, 631), (131, 2895, 2001), (1803, 131, 640), (1501, 2767, 72), (2355, 1286, 90), (2562, 1165, 67),
                                   (2722, 2401, 65), (4095, 3071, 129), (1500, 1500, 1500)])
def test_matmul_planes(ops, m, n, k, precision, tol):
    rng = np.random.default_rng(m + k)
    a, b = rng.normal(0, 1, (m, k)).astype(np.float32), rng.normal(0, 1, (k, n)).astype(np.float32)
    a[:, k - 1] *= 30.0  # the last k, next to the block's padding
    got = ops.matmul(a, b, precision=precision)
    rows = np.unique(np.r_[0:40, m - 40:m, rng.integers(0, m, 100)])
    want = a[rows].astype(np.float64) @ b.astype(np.float64)
    assert got.shape == (m, n)
    assert np.all(np.abs(got[rows] - want) <= tol * (np.abs(a[rows]) @ np.abs(b)))
    relu = ops.matmul(a, b, relu=True, precision=precision)
    assert np.array_equal(relu, np.maximum(got, 0.0))
