"""Products over operands split into bf16 terms once (csrc/gemm_planes.hip), at sizes where each of its tiles is chosen:
edges that no tile divides, a last block of k that is part empty, rows that are no multiple of 16 bytes; the Linears and
prompts that take it."""
import ctypes as C

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
                                   (2722, 2401, 65), (4095, 3071, 129), (1500, 1500, 1500),
                                   (3001, 4099, 1605)])
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


@pytest.mark.parametrize("kind,rows,cols,m", [("q8_0", 11270, 2080, 391), ("q8_0", 5001, 2048, 1543), ("q4_0", 11270, 2080, 800), ("q4_0", 4096, 11008, 777),
                                              ("f16", 4100, 1008, 777), ("f16", 1601, 6400, 1030), ("f32", 6402, 1600, 517)])
@pytest.mark.parametrize("prologue", [None, "rmsnorm"])
def test_linear_planes(ops, kind, rows, cols, m, prologue):
    from caten_amd.llm import Tensor
    rng = np.random.default_rng(rows + m)
    w = ops.WeightMatrix(kind, Tensor.from_f32(rng.normal(0, 0.05, (rows, cols)).astype(np.float32), kind).raw, rows, cols)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32)
    x[:, 3] *= 100.0
    g = rng.normal(1, 0.05, cols).astype(np.float32)
    bias, res = rng.normal(0, 1, rows).astype(np.float32), rng.normal(0, 1, (m, rows)).astype(np.float32)
    at, rs = np.unique(np.r_[0:40, rows - 40:rows, rng.integers(0, rows, 100)]), np.unique(np.r_[0:9, m - 9:m, rng.integers(0, m, 40)])
    x64 = x[rs].astype(np.float64)
    if prologue:
        x64 = x64 / np.sqrt((x64 * x64).mean(-1, keepdims=True) + 1e-5) * g
    want = np.maximum(x64 @ w.dequantize()[at].astype(np.float64).T + bias[at], 0.0) + res[rs][:, at]
    for _ in range(2):  # with the matrix's terms made, and as they are kept
        got = ops.linear(x, w, bias, res, act="relu", prologue=prologue, **(dict(norm_g=g) if prologue else {}))[np.ix_(rs, at)]
        assert np.linalg.norm(got - want) < 1e-5 * np.linalg.norm(want)
    w.free()


@pytest.mark.parametrize("arch,kind,rows", [("llama", "q8_0", 1501), ("llama", "q4_0", 1100), ("llama", "f16", 900), ("gpt2", "f16", 777), ("gpt2", "q8_0", 1900)])
def test_long_prompt_equals_short_pieces(ops, arch, kind, rows):
    from caten_amd import llm, synth
    if arch == "llama":
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=1024, n_heads=16, n_kv_heads=4, ffn=5632, n_layers=3, vocab=500, max_seq=2048)
        model = llm.make_llama(cfg, llm.llama_state_dict(synth.llama_weights(cfg, seed=3), kind))
    else:
        cfg = dict(synth.GPT2_CONFIGS["gpt2"], dim=1024, n_heads=16, n_layers=3, vocab=500, max_seq=2048)
        model = llm.make_gpt2(cfg, llm.gpt2_state_dict(synth.gpt2_weights(cfg, seed=3), kind))
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows + 1, seed=3)]
    got = [model.forward(ids[:rows], rows, 0, return_logits=True), model.forward(ids[rows:], 1, rows, return_logits=True)]
    for n in range(0, rows, 63):
        want = [model.forward(ids[n:min(n + 63, rows)], min(63, rows - n), n, return_logits=True)]
    want.append(model.forward(ids[rows:], 1, rows, return_logits=True))
    for (t0, l0), (t1, l1) in zip(got, want):
        assert t0 == t1
        assert np.linalg.norm(l0 - l1) < 1e-4 * np.linalg.norm(l1)
    model.close()


@pytest.mark.parametrize("heads,kv_heads,first,rows", [(32, 4, 0, 1333), (32, 8, 37, 1500), (16, 16, 0, 2000), (16, 4, 3, 1999)])
def test_long_prompt_attention_equals_short_pieces(ops, heads, kv_heads, first, rows):
    """csrc/attn_planes.hip: grouped and single heads of 64 and 128, cached rows that are no multiple of a key tile in front."""
    from caten_amd import llm, synth
    cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=2048, n_heads=heads, n_kv_heads=kv_heads, ffn=512, n_layers=2, vocab=500, max_seq=2048)
    model = llm.make_llama(cfg, llm.llama_state_dict(synth.llama_weights(cfg, seed=4), "q8_0"))
    ids = [float(t) for t in synth.prompt(cfg["vocab"], first + rows + 1, seed=4)]
    n = first + rows
    if first:
        model.forward(ids[:first], first, 0)
    got = [model.forward(ids[first:n], rows, first, return_logits=True), model.forward(ids[n:], 1, n, return_logits=True)]
    for at in range(0, n, 63):
        want = [model.forward(ids[at:min(at + 63, n)], min(63, n - at), at, return_logits=True)]
    want.append(model.forward(ids[n:], 1, n, return_logits=True))
    for (t0, l0), (t1, l1) in zip(got, want):
        assert t0 == t1
        assert np.linalg.norm(l0 - l1) < 1e-4 * np.linalg.norm(l1)
    model.close()


def allocated(lib):
    """bytes in use, bytes taken from the driver"""
    from caten_amd import _lib
    live, cached, drv = C.c_size_t(), C.c_size_t(), C.c_size_t()
    _lib.check(lib.cthip_cache_stats(C.byref(live), C.byref(cached), C.byref(drv)))
    return live.value, live.value + cached.value


def matrix(ops, kind, rows, cols, seed):
    from caten_amd.llm import Tensor
    rng = np.random.default_rng(seed)
    return ops.WeightMatrix(kind, Tensor.from_f32(rng.normal(0, 0.05, (rows, cols)).astype(np.float32), kind).raw, rows, cols)


def test_weight_terms_are_bounded_and_given_back(ops):
    """Option "weight_planes" bounds what matrices keep; cthip_cache_trim, a lower limit, an allocation that finds no memory and the
    end of a matrix give it back, and the next call makes the terms again with the same result."""
    from caten_amd import HipError, _lib
    lib = _lib.init(0)
    a, b = matrix(ops, "q8_0", 5001, 2048, 1), matrix(ops, "q8_0", 11270, 2080, 2)
    a_bytes, b_bytes = 5001 * 64 * 64, 11270 * 65 * 64  # 20.5 + 46.9 MB
    x, y = (np.random.default_rng(3).normal(0, 1, (3000, n)).astype(np.float32) for n in (2048, 2080))  # rows that pay for the terms at every call
    try:
        _lib.check(lib.cthip_set_option(b"weight_planes", 0))
        none = allocated(lib)[0]
        ra, rb = ops.linear(x, a), ops.linear(y, b)
        assert allocated(lib)[0] == none
        _lib.check(lib.cthip_set_option(b"weight_planes", 64))  # room for one of them
        same = lambda: np.array_equal(ops.linear(x, a), ra) and np.array_equal(ops.linear(y, b), rb)
        assert same()
        kept = allocated(lib)[0] - none
        assert a_bytes <= kept < b_bytes
        assert same() and allocated(lib)[0] - none == kept
        _lib.check(lib.cthip_cache_trim())
        assert allocated(lib)[0] == none
        assert same() and allocated(lib)[0] - none == kept
        p = C.c_void_p()
        with pytest.raises(HipError, match="hipMalloc"):
            _lib.check(lib.cthip_alloc(C.byref(p), 1 << 50))
        assert allocated(lib)[0] == none
        assert same() and allocated(lib)[0] - none == kept  # (and the failed call's error is not found by a later launch)
        _lib.check(lib.cthip_set_option(b"weight_planes", 32768))
        assert same() and a_bytes + b_bytes <= allocated(lib)[0] - none
        _lib.check(lib.cthip_set_option(b"weight_planes", 8))
        assert allocated(lib)[0] == none
        assert same() and allocated(lib)[0] == none
        _lib.check(lib.cthip_set_option(b"weight_planes", 32768))
        assert same()
        both = allocated(lib)[0]
        a.free()
        assert allocated(lib)[0] <= both - a_bytes - 5001 * 2048
        with pytest.raises(HipError, match="weight_planes"):
            _lib.check(lib.cthip_set_option(b"weight_planes", -1))
    finally:
        _lib.check(lib.cthip_set_option(b"weight_planes", 32768))
    b.free()


@pytest.mark.parametrize("kind,rows", [("q4_0", 200), ("q8_0", 200), ("f16", 260)])
def test_prompt_without_room_for_weight_terms(ops, kind, rows):
    """Past the limit a Linear takes terms only where making them at every call pays, and none are made to be thrown away: at
    these rows the gate|up matrix is faster with kept terms and slower with its own."""
    from caten_amd import _lib, llm, synth
    lib = _lib.init(0)
    cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=2048, n_heads=32, n_kv_heads=4, ffn=5632, n_layers=2, vocab=500, max_seq=1024)
    model = llm.make_llama(cfg, llm.llama_state_dict(synth.llama_weights(cfg, seed=5), kind))
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows, seed=5)]
    model.forward(ids[:8], 8, 0)
    try:
        _lib.check(lib.cthip_set_option(b"weight_planes", 0))
        _lib.check(lib.cthip_cache_trim())
        before = allocated(lib)[1]
        t0, l0 = model.forward(ids, rows, 0, return_logits=True)
        taken = allocated(lib)[1] - before
        terms = 11264 * 2048 * (4 if kind == "f16" else 2)  # of the gate|up matrix
        assert taken < terms, (taken, terms)
    finally:
        _lib.check(lib.cthip_set_option(b"weight_planes", 32768))
    live = allocated(lib)[0]
    t1, l1 = model.forward(ids, rows, 0, return_logits=True)
    assert allocated(lib)[0] - live >= terms
    assert t0 == t1
    assert np.linalg.norm(l0 - l1) < 1e-4 * np.linalg.norm(l1)
    model.close()
