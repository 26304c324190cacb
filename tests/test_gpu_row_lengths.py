"""Row operations at the row lengths where their launches change: rows of a block's registers (multiples of the block's
chunks, one more, one less, no multiple of four), rows shared by several blocks, and rows no block holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def close(a, b, rtol, atol):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    bad = ~(np.abs(a - b) <= atol + rtol * np.abs(b))  # (a NaN is a difference)
    assert not bad.any(), f"{bad.sum()} of {bad.size} differ; max abs err {np.abs(a - b).max():.3e}"


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


@pytest.mark.parametrize("rows,n", [(3, 3), (3, 4), (5, 5), (2, 255), (2, 257), (2, 1023), (7, 1025), (2, 2047), (2, 2049), (2, 4097),
                                    (3, 8190), (2, 8193), (2, 16386), (2, 32769), (49, 32769), (2, 53248), (2, 53251), (2, 65536), (1, 65541)])
def test_rows_of_any_length(ops, oracle, rows, n):
    rng = np.random.default_rng(n)
    x = rng.normal(0.3, 1, (rows, n)).astype(np.float32)
    g, b = rng.normal(1, 0.02, n).astype(np.float32), rng.normal(0, 0.02, n).astype(np.float32)
    close(ops.softmax(x), oracle.softmax(x), 1e-4, 1e-7)
    close(ops.layernorm(x, g, b), oracle.layernorm(x, g, b), 1e-4, 3e-5)
    close(ops.rmsnorm(x, g), oracle.rmsnorm(x, g), 1e-4, 1e-5)
    close(ops.layernorm_softmax(x, g, b), oracle.softmax(oracle.layernorm(x, g, b)), 1e-4, 1e-7)


# where norms of more than 1280 / 1536 floats go from a block to a wavefront per row (ten / five rows to each of 256 compute units), and softmax of aligned rows to one
@pytest.mark.parametrize("rows,n", [(1279, 1537), (1280, 1537), (1279, 1536), (2559, 1281), (2560, 1281), (2559, 2047), (2560, 2046), (7, 128), (7, 132), (7, 256), (6, 260)])
def test_either_side_of_a_row_count(ops, oracle, rows, n):
    test_rows_of_any_length(ops, oracle, rows, n)


@pytest.mark.parametrize("rows,n", [(3, 1025), (2, 8193), (1, 32769), (3, 50257), (49, 32769), (1, 65541), (2, 70001)])
@pytest.mark.parametrize("masked", [-np.inf, np.finfo(np.float32).min])
def test_softmax_of_masked_rows(ops, oracle, rows, n, masked):
    """A row of which a sampler keeps a few values: whole stretches of it, and whole pieces where a row is shared, are masked.
    Rows without a probability distribution stay what they are: NaN."""
    rng = np.random.default_rng(n)
    x = np.full((rows, n), masked, np.float32)
    for r in range(rows):
        x[r, rng.choice(n // 2, 40, replace=False) + (n // 2 if r % 2 else 0)] = rng.normal(0, 3, 40)
    with np.errstate(over="ignore"):
        want = oracle.softmax(x)
    assert np.isfinite(want).all()
    close(ops.softmax(x), want, 1e-4, 1e-7)
    for bad in (np.inf, np.nan):
        y = x.copy()
        y[0, n - 1] = bad
        got = ops.softmax(y)
        assert np.isnan(got[0]).all()
        close(got[1:], want[1:], 1e-4, 1e-7)
    y = x.copy()
    y[0] = -np.inf
    assert np.isnan(ops.softmax(y)[0]).all()


@pytest.mark.parametrize("rows,n", [(3, 1), (3, 3), (5, 5), (4, 1023), (4, 1025), (2, 4099), (2, 8191), (16, 8192), (17, 16385), (3, 50257)])
def test_argmax_of_any_length(ops, rows, n):
    rng = np.random.default_rng(n)
    x = rng.integers(0, max(2, n // 3), (rows, n)).astype(np.float32)  # many ties: the lowest index counts
    x[0, n - 1] = n  # the last element, which a row that is no multiple of four reads through an overlapping piece
    for _ in range(2):  # the counters behind a row's last part are back at zero
        assert np.array_equal(np.atleast_1d(ops.argmax(x)).ravel(), x.argmax(-1))


@pytest.mark.parametrize("rows,n", [(4, 3), (5, 1025), (6, 8191), (5, 8193), (4, 50257), (17, 16385)])
def test_argmax_of_rows_that_are_not_finite(ops, rows, n):
    """Masked stretches and infinities are ordinary values, a NaN is never chosen; the lowest index where nothing is larger."""
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (rows, n)).astype(np.float32)
    x[0, n // 2:] = -np.inf
    x[1] = -np.inf
    x[2, [1, n - 1]] = np.inf
    x[3, rng.random(n) < 0.7] = np.nan
    x[3, 0] = -np.inf
    if rows > 4:
        x[4] = np.nan
    want = np.where(np.isnan(x), -np.inf, x).argmax(-1)
    assert np.array_equal(ops.argmax(x).ravel(), want)


@pytest.mark.parametrize("rows,n", [(3, 1024), (3, 2051), (2, 8193), (2, 53251), (1, 70001)])
def test_layernorm_softmax_of_rows_that_are_not_finite(ops, rows, n):
    """A row with an infinity or a NaN has no mean: NaN throughout, and the rows beside it what they are alone."""
    rng = np.random.default_rng(n)
    x = rng.normal(0.3, 1, (rows, n)).astype(np.float32)
    alone = ops.layernorm_softmax(x)
    for bad in (np.inf, -np.inf, np.nan):
        y = x.copy()
        y[0, n - 1] = bad
        got = ops.layernorm_softmax(y)
        assert np.isnan(got[0]).all() and np.array_equal(got[1:], alone[1:])


@pytest.mark.parametrize("n", [4, 5, 40, 63, 64, 65, 87, 127, 128, 129, 200, 255, 256, 258, 513, 770, 1023, 1537, 2047])
@pytest.mark.parametrize("rows", [1, 7, 33, 40001])
def test_rows_of_a_part_of_a_wavefront(ops, oracle, rows, n):
    """Several rows per wavefront, one or two passes of them, at element offsets of any alignment; results may go where the input was,
    a row that is not finite leaves its neighbours alone, and nothing is stored behind the last row."""
    import ctypes as C
    from caten_amd import _lib
    lib = _lib.load()
    if rows * n > 6_000_000:
        rows = 6_000_000 // n
    rng = np.random.default_rng(n)
    x = rng.normal(0.3, 1, (rows, n)).astype(np.float32)
    g, b = rng.normal(1, 0.02, n).astype(np.float32), rng.normal(0, 0.02, n).astype(np.float32)
    bad = rows // 2
    x[bad, n // 2] = np.inf
    dev, gd, bd = C.c_void_p(), C.c_void_p(), C.c_void_p()
    for p, k in ((dev, rows * n + 16), (gd, n + 1), (bd, n + 1)):
        _lib.check(lib.cthip_alloc(C.byref(p), 4 * k))
    g1, b1 = np.concatenate([[0], g]).astype(np.float32), np.concatenate([[0], b]).astype(np.float32)
    _lib.check(lib.cthip_h2d(gd, g1.ctypes.data_as(C.c_void_p), 4 * (n + 1)))
    _lib.check(lib.cthip_h2d(bd, b1.ctypes.data_as(C.c_void_p), 4 * (n + 1)))
    ok = np.arange(rows) != bad
    for op, want, tol in (("softmax", oracle.softmax(x[ok]), (1e-4, 1e-7)), ("layernorm", oracle.layernorm(x[ok], g, b), (1e-4, 3e-5)),
                          ("rmsnorm", oracle.rmsnorm(x[ok], g), (1e-4, 1e-5)), ("layernorm_softmax", oracle.softmax(oracle.layernorm(x[ok], g, b)), (1e-4, 1e-7))):
        for off in (0, 1):
            buf = np.full(rows * n + 16, 7.5, np.float32)
            buf[off:off + rows * n] = x.ravel()
            _lib.check(lib.cthip_h2d(dev, buf.ctypes.data_as(C.c_void_p), buf.nbytes))
            p = C.c_void_p(dev.value + 4 * off)
            gp, bp = C.c_void_p(gd.value + 4), C.c_void_p(bd.value + 4)
            if op == "softmax":
                rc = lib.cthip_softmax(p, p, rows, n)
            elif op == "rmsnorm":
                rc = lib.cthip_rmsnorm(p, p, gp, 1e-5, rows, n)
            else:
                rc = getattr(lib, "cthip_" + op)(p, p, gp, bp, 1e-5, rows, n)
            _lib.check(rc)
            _lib.check(lib.cthip_d2h(buf.ctypes.data_as(C.c_void_p), dev, buf.nbytes))
            assert (buf[:off] == 7.5).all() and (buf[off + rows * n:] == 7.5).all()
            y = buf[off:off + rows * n].reshape(rows, n)
            close(y[ok], want, *tol)
            assert np.isnan(y[bad, n // 2])
    for p in (dev, gd, bd):
        _lib.check(lib.cthip_free(p))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 1023, 1024, 1027, 4099, 100_001])
def test_unary_of_any_length(ops, n):
    import ctypes as C
    from caten_amd import _lib
    lib = _lib.load()
    x = np.random.default_rng(n).normal(0, 2, n + 9).astype(np.float32)
    dev = C.c_void_p()
    _lib.check(lib.cthip_alloc(C.byref(dev), x.nbytes))
    for off in (0, 1):
        _lib.check(lib.cthip_h2d(dev, x.ctypes.data_as(C.c_void_p), x.nbytes))
        p = C.c_void_p(dev.value + 4 * off)
        _lib.check(lib.cthip_unary(3, p, p, n))
        y = np.empty_like(x)
        _lib.check(lib.cthip_d2h(y.ctypes.data_as(C.c_void_p), dev, x.nbytes))
        want = x.astype(np.float64)
        want[off:off + n] /= 1 + np.exp(-want[off:off + n])
        close(y, want, 1e-5, 1e-6)
    _lib.check(lib.cthip_free(dev))
