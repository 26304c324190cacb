"""Launches that take scratch from the allocator, recorded into a graph on the library's stream: a replay must not find its scratch
in other hands, so they take the path that needs none, and what stays with a matrix is not made by launches that have not
run.  Every replay, with other work of the library between them, gives what the eager call gives."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def packed(kind, a):
    from caten_amd.llm import Tensor
    return Tensor.from_f32(a, kind).raw


def cases(ops, _lib, lib, rng):
    def linear(kind, rows, cols, m, tol, pro=_lib.PRO_NONE):
        w = ops.WeightMatrix(kind, packed(kind, rng.normal(0, 0.05, (rows, cols)).astype(np.float32)), rows, cols)
        x = ops.DeviceArray.from_numpy(rng.normal(0.3, 1, (m, cols * (2 if pro == _lib.PRO_SWIGLU else 1))).astype(np.float32))
        y, g, b = ops.DeviceArray((m, rows)), *(ops.DeviceArray.from_numpy(rng.normal(1, 0.1, cols).astype(np.float32)) for _ in range(2))
        gamma = g.ptr if pro in (_lib.PRO_LAYERNORM, _lib.PRO_RMSNORM) else None
        beta = b.ptr if pro == _lib.PRO_LAYERNORM else None
        return y, tol, (w, x, g, b), lambda: _lib.check(lib.cthip_linear(y.ptr, w.handle, x.ptr, m, None, None, 0, pro, gamma, beta, 1e-5))

    def row(n):
        x = rng.normal(0, 1, (2, n)).astype(np.float32)
        x[:, n // 3:] = -np.inf
        x, y = ops.DeviceArray.from_numpy(x), ops.DeviceArray((2, n))
        return y, 1e-5, (x,), lambda: _lib.check(lib.cthip_softmax(y.ptr, x.ptr, 2, n))

    def best(n):
        x, y = ops.DeviceArray.from_numpy(rng.normal(0, 1, (2, n)).astype(np.float32)), ops.DeviceArray((2,), np.int64)
        return y, 0.0, (x,), lambda: _lib.check(lib.cthip_argmax(y.ptr, x.ptr, 2, n))

    def matmul(m, n, k):
        a, b = (ops.DeviceArray.from_numpy(rng.normal(0, 1, s).astype(np.float32)) for s in ((m, k), (k, n)))
        y = ops.DeviceArray((m, n))
        return y, 5e-5, (a, b), lambda: _lib.check(lib.cthip_matmul(y.ptr, a.ptr, b.ptr, m, n, k, 0, 2))

    # few rows; many rows of a matrix that would keep its terms, and of one that makes them at every call; long rows; a large product; products and Linears
    # that share their reduction, then Linears with a norm or SwiGLU in front: rows past and below the tiles', widths that no single-row kernel is laid out for
    return [linear("q8_0", 4100, 2048, 7, 1e-6), linear("q4_0", 12000, 2080, 5, 1e-6), linear("f16", 4100, 1008, 777, 5e-5), linear("q8_0", 11270, 2080, 391, 5e-5),
            linear("f32", 6402, 1600, 517, 5e-5), row(50257), row(70001), best(50257), matmul(1500, 1500, 1500),
            matmul(130, 190, 1024), linear("f16", 300, 4096, 20, 5e-5), linear("q8_0", 640, 5120, 70, 5e-5),
            linear("q8_0", 520, 1024, 40, 5e-5, _lib.PRO_RMSNORM), linear("f32", 333, 512, 100, 5e-5, _lib.PRO_LAYERNORM), linear("f16", 300, 1024, 9, 5e-5, _lib.PRO_SWIGLU),
            linear("q4_0", 2600, 4096, 12, 5e-5, _lib.PRO_SWIGLU), linear("f32", 200, 1001, 12, 5e-5, _lib.PRO_LAYERNORM), linear("f32", 200, 1001, 3, 1e-6, _lib.PRO_RMSNORM),
            linear("f16", 201, 999, 5, 1e-6, _lib.PRO_SWIGLU), linear("q8_0", 70, 40960, 3, 1e-6, _lib.PRO_LAYERNORM), linear("q4_0", 70, 40960, 9, 5e-5, _lib.PRO_RMSNORM)]


def test_captured_calls_take_no_scratch():
    from caten_amd import _lib, ops
    lib = _lib.init(0)
    stream = C.c_void_p(lib.cthip_stream())

    def allocator():
        v = [C.c_size_t() for _ in range(3)]
        _lib.check(lib.cthip_cache_stats(*[C.byref(s) for s in v]))
        return [s.value for s in v]

    rng = np.random.default_rng(0)
    for k, (y, tol, keep, call) in enumerate(cases(ops, _lib, lib, rng)):
        print("case", k, flush=True)
        _lib.check(lib.cthip_cache_trim())
        _lib.check(lib.cthip_sync())
        before = allocator()
        graph, run = C.c_void_p(), C.c_void_p()
        assert lib.hipStreamBeginCapture(stream, 1) == 0
        call()
        assert lib.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert allocator() == before
        assert lib.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        call()  # eager, on its own path
        want = y.numpy().astype(np.float64)
        other = [ops.DeviceArray.from_numpy(np.full(1 << 18, 7.0, np.float32)) for _ in range(8)]  # in what the call gave back
        for _ in range(3):
            _lib.check(lib.cthip_memset(y.ptr, 0xff, y.nbytes))
            assert lib.hipGraphLaunch(run, stream) == 0
            got = y.numpy().astype(np.float64)
            assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), k
            call()
            assert np.linalg.norm(y.numpy() - want) <= tol * np.linalg.norm(want), k
        assert all((o.numpy() == 7.0).all() for o in other)
        lib.hipGraphExecDestroy(run)
        lib.hipGraphDestroy(graph)
        for d in other:
            d.free()
        for d in keep:
            d.free()
