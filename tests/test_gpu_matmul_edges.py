"""Matrix products whose rows are no whole 16-byte pieces, at the ends of tiles, steps and shares: every element in its place, nothing read from
outside an operand (what lies around them is NaN), nothing stored outside the result."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# two fp32 sums of K products, one term (2^-9 an operand), two (2^-16 of a product dropped), three (fp32 grade)
TOL = {0: 2e-6, 1: 6e-3, 2: 2e-5, 3: 2e-6}


@pytest.fixture(scope="module")
def lib():
    from caten_amd import _lib
    return _lib.init(0)


@pytest.mark.parametrize("precision", [0, 1, 2, 3])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (3, 2, 5), (5, 3, 7), (2, 5, 3), (1, 4, 4), (1, 5, 6), (63, 61, 33), (64, 64, 63), (65, 67, 65), (17, 130, 127),
                                   (33, 66, 129), (70, 71, 191), (64, 128, 193), (31, 253, 321), (20, 232, 142), (129, 190, 62), (300, 6, 1027), (6, 299, 2050),
                                   (48, 189, 1655), (257, 258, 259), (513, 514, 101), (401, 403, 406), (1027, 1030, 66), (900, 1100, 1001)])
def test_matmul_edges(lib, m, n, k, precision):
    from caten_amd import _lib
    rng = np.random.default_rng(m * n + k)
    a, b = rng.normal(0, 1, (m, k)).astype(np.float32), rng.normal(0, 1, (k, n)).astype(np.float32)
    pads = (5, 3, 9)  # operands and result at addresses of any alignment
    host = [np.concatenate([np.full(p, np.nan, np.float32), x.ravel(), np.full(16, np.nan, np.float32)]) for p, x in zip(pads, (a, b, np.zeros((m, n), np.float32)))]
    dev = []
    for h in host:
        p = C.c_void_p()
        _lib.check(lib.cthip_alloc(C.byref(p), h.nbytes))
        _lib.check(lib.cthip_h2d(p, h.ctypes.data_as(C.c_void_p), h.nbytes))
        dev.append(p)
    pa, pb, pc = (C.c_void_p(d.value + 4 * p) for d, p in zip(dev, pads))
    want = a.astype(np.float64) @ b.astype(np.float64)
    size = np.abs(a).astype(np.float64) @ np.abs(b)  # a bound in what the products add up to, element by element
    for act in (0, 1):
        _lib.check(lib.cthip_matmul(pc, pa, pb, m, n, k, act, precision))
        got = np.empty_like(host[2])
        _lib.check(lib.cthip_d2h(got.ctypes.data_as(C.c_void_p), dev[2], got.nbytes))
        assert np.isnan(got[:9]).all() and np.isnan(got[9 + m * n:]).all()
        c = got[9:9 + m * n].reshape(m, n)
        assert np.all(np.abs(c - (np.maximum(want, 0) if act else want)) <= TOL[precision] * size)
    for d in dev:
        _lib.check(lib.cthip_free(d))
