"""Linears over 2 .. 32 rows in one pass over the weights (csrc/linear_rows.hip) at the shapes where it takes over: column
groups and units of k that the matrix does not fill, rows of an odd number of blocks (scales fetched one by one), widths
that are no multiple of a block, every prologue and terms per input, the largest and smallest row counts of its tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


def packed(kind, a):
    from caten_amd.llm import Tensor
    return Tensor.from_f32(a, kind).raw


def norm(x, g, b, kind):
    if kind == "layernorm":
        x = x - x.mean(-1, keepdims=True)
    x = x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5) * g
    return x + b if kind == "layernorm" else x


@pytest.mark.parametrize("kind,rows,cols,m", [
    ("q8_0", 2611, 2080, 7), ("q8_0", 12000, 2048, 3), ("q8_0", 9001, 2560, 8), ("q8_0", 9001, 2560, 16),
    ("q4_0", 2611, 2080, 7), ("q4_0", 2600, 11008, 2), ("q4_0", 9001, 2560, 9), ("q4_0", 700, 11008, 6),
    ("f16", 2603, 2056, 7), ("f16", 4099, 5000, 5), ("f16", 9001, 2560, 16), ("f16", 15001, 4104, 17), ("f16", 15001, 4104, 32), ("f16", 11000, 5632, 24),
    ("f32", 2603, 2052, 7), ("f32", 1501, 4100, 4)])
@pytest.mark.parametrize("prologue", [None, "layernorm", "rmsnorm", "swiglu"])
def test_linear_rows(ops, kind, rows, cols, m, prologue):
    rng = np.random.default_rng(rows + m)
    w = ops.WeightMatrix(kind, packed(kind, rng.normal(0, 0.05, (rows, cols)).astype(np.float32)), rows, cols)
    x = rng.normal(0, 1, (m, cols * (2 if prologue == "swiglu" else 1))).astype(np.float32)
    x[:, 3] *= 300.0  # one input far above the others of its row
    g, b = rng.normal(1, 0.05, cols).astype(np.float32), rng.normal(0, 0.05, cols).astype(np.float32)
    bias, res = rng.normal(0, 1, rows).astype(np.float32), rng.normal(0, 1, (m, rows)).astype(np.float32)
    at = np.unique(np.r_[0:40, rows - 40:rows, rng.integers(0, rows, 100)])  # output columns that are checked
    x64 = x.astype(np.float64)
    if prologue == "swiglu":
        x64 = x64[:, :cols] / (1 + np.exp(-x64[:, :cols])) * x64[:, cols:]
    elif prologue:
        x64 = norm(x64, g, b, prologue)
    want = np.maximum(x64 @ w.dequantize()[at].astype(np.float64).T + bias[at], 0.0) + res[:, at]
    kw = dict(norm_g=g, norm_b=b if prologue == "layernorm" else None) if prologue in ("layernorm", "rmsnorm") else {}
    for _ in range(2):  # the shares' counters are back at zero
        got = ops.linear(x, w, bias, res, act="relu", prologue=prologue, **kw)[:, at]
        rel = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert rel < (1e-6 if m < 8 else 1e-5), rel
    w.free()


def tree_bound(cols):
    """Additions behind one output value: terms of a block or two on the matrix cores, blocks, shares of k.  What any order of them in
    fp32 may be off by, in units of the sum of the products' magnitudes."""
    return (3 * 64 + cols / 32 + 32) * 2.0 ** -24


@pytest.mark.parametrize("kind,rows,cols,m", [("q8_0", 2611, 2080, 7), ("q8_0", 9001, 2560, 12), ("q4_0", 2611, 2080, 7), ("q4_0", 9001, 2560, 16), ("f16", 2603, 2056, 7),
                                              ("f16", 9001, 2560, 11), ("f16", 15001, 4104, 23), ("f32", 2603, 2052, 5)])
@pytest.mark.parametrize("outlier", [1e8, 2.0 ** 100])
def test_inputs_of_any_magnitude(ops, kind, rows, cols, m, outlier):
    """An input far above the others costs them no bits, column by column: where its weight is zero the result is what the
    others give.  Nor does one row of inputs cost another."""
    rng = np.random.default_rng(rows + m)
    a = rng.normal(0, 0.05, (rows, cols)).astype(np.float32)
    a[:, 5], a[:, cols - 7] = 0.0, 0.0
    w = ops.WeightMatrix(kind, packed(kind, a), rows, cols)
    x = (rng.normal(0, 1, (m, cols)) * 10.0 ** rng.uniform(-9, 0, (m, cols))).astype(np.float32)
    x[:, 5], x[:, cols - 7] = outlier, -outlier
    x[1] *= np.float32(2.0 ** -60)
    x[1, 5], x[1, cols - 7] = 1.0, 2.0 ** -70
    x[2] = rng.normal(0, 1, cols) * 2.0 ** -126  # subnormal numbers among them: a term of 16-bit hardware takes them for zero
    w64 = w.dequantize().astype(np.float64)
    assert not w64[:, 5].any() and not w64[:, cols - 7].any()
    got = ops.linear(x, w)
    x64 = x.astype(np.float64)
    assert np.all(np.abs(got - x64 @ w64.T) <= tree_bound(cols) * (np.abs(x64) @ np.abs(w64).T))
    w.free()


@pytest.mark.parametrize("kind,rows,cols,m", [("q8_0", 2611, 2080, 7), ("q8_0", 9001, 2560, 12), ("q4_0", 2611, 2080, 7), ("f16", 2603, 2056, 7),
                                              ("f16", 15001, 4104, 23), ("f32", 2603, 2052, 5)])
def test_inputs_that_are_not_finite_or_nearly_so(ops, kind, rows, cols, m):
    """Infinities and NaN as in fp32 arithmetic (infinity of a weight's sign; NaN against a weight of zero or another
    infinity), rows beside them untouched; the largest floats times weights below one half."""
    rng = np.random.default_rng(rows + m)
    a = rng.normal(0, 0.05, (rows, cols)).astype(np.float32)
    a[::3, 40] = 0.0
    w = ops.WeightMatrix(kind, packed(kind, a), rows, cols)
    w64 = w.dequantize().astype(np.float64)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32)
    top = np.finfo(np.float32).max if kind in ("f16", "f32") else np.float32(2.0 ** 119)  # (integers up to 127 come before their scale)
    x[0, 40] = np.inf
    x[1, 40], x[1, 41] = -np.inf, np.inf
    x[2, 7] = np.nan
    x[3] = 0.0
    x[3, 11] = top
    got = ops.linear(x, w)
    with np.errstate(invalid="ignore"):
        want = np.stack([(x[r].astype(np.float64) * w64).sum(1) for r in range(m)])
    ok = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    bound = tree_bound(cols) * (np.abs(np.where(np.isfinite(x), x, 0).astype(np.float64)) @ np.abs(w64).T)
    assert np.all(np.abs(got[ok] - want[ok]) <= bound[ok])
    w.free()


@pytest.mark.parametrize("rows,cols,m", [(2603, 2052, 5), (1100, 11000, 7)])
def test_small_rows_against_large_weights(ops, rows, cols, m):
    """fp32 weights about 1e35 and rows down to subnormal numbers: the results are ordinary floats."""
    rng = np.random.default_rng(rows)
    a = rng.normal(0, 1e35, (rows, cols)).astype(np.float32)
    w = ops.WeightMatrix("f32", a, rows, cols)
    x = rng.normal(0, 1, (m, cols)) * np.array([1.0, 2.0 ** -33, 1e-12, 1e-30, 1e-39, 1e-20, 1e-10])[:m, None]
    x = x.astype(np.float32)
    got, want = ops.linear(x, w), x.astype(np.float64) @ a.astype(np.float64).T
    assert np.abs(want).max() < 2.0 ** 127  # (rows of ones: 1e35 sqrt(cols) = 1e37, and a few times that)
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - want) <= tree_bound(cols) * (np.abs(x.astype(np.float64)) @ np.abs(a.astype(np.float64)).T))
    w.free()


@pytest.mark.parametrize("prologue", [None, "swiglu"])
@pytest.mark.parametrize("rows,cols", [(4096, 2052), (1100, 11000)])
def test_rows_small_in_part_or_whole(ops, rows, cols, prologue):
    """Several blocks share an input row without a norm, 2048 columns each: ordinary rows, rows that only one block can tell from small ones, small ones, one of zeros.  With SwiGLU
    at gates of 16, silu(g) = g (1 - 1e-7): its own error, a few 2^-24 of a value, adds to the sums'."""
    rng = np.random.default_rng(rows)
    a = rng.normal(0, 1e30, (rows, cols)).astype(np.float32)
    w = ops.WeightMatrix("f32", a, rows, cols)
    v = rng.normal(0, 1, (7, cols))
    v[1, :2048] *= 1e-20
    v[2, 2048:] *= 1e-20
    v[3] *= 1e-15
    v[4] *= 1e-30
    v[4, -1] = 2.0 ** -20
    v[5] *= 2.0 ** -40
    v[5, :2048] = 0.0
    v[6] = 0.0
    x = v.astype(np.float32)
    if prologue:
        gate = np.full_like(x, 16.0)
        x64 = 16.0 / (1 + np.exp(-16.0)) * (x / 16.0).astype(np.float64)
        x = np.concatenate([gate, x / np.float32(16.0)], 1)
    else:
        x64 = x.astype(np.float64)
    got, want = ops.linear(x, w, prologue=prologue), x64 @ a.astype(np.float64).T
    bound = (tree_bound(cols) + (8 * 2.0 ** -24 if prologue else 0)) * (np.abs(x64) @ np.abs(a.astype(np.float64)).T)
    assert np.all(np.abs(got - want) <= bound)
    w.free()


@pytest.mark.parametrize("kind,rows,cols,m,precision", [
    ("f16", 2100, 28672, 27, 2), ("f16", 2100, 28672, 32, 2), ("f16", 2100, 28672, 18, 3), ("f16", 2100, 28672, 32, 3), ("f16", 2050, 29568, 25, 2),
    ("f16", 2500, 24576, 31, 2), ("q4_0", 4098 * 128, 2240, 16, 2), ("f16", 2100, 28672, 17, 2), ("f16", 2100, 28672, 16, 2), ("q8_0", 1700, 28672, 16, 3)])
def test_wide_rows_and_many_columns(ops, oracle, kind, rows, cols, m, precision):
    """Matrices whose rows no share of a workgroup's memory holds, whether for their width or because more column groups than
    tickets allow one share only: another launch takes them.  The last three are of this kernel's."""
    from caten_amd import _lib
    lib = _lib.init(0)
    rng = np.random.default_rng(rows + m)
    base = min(rows, 4098)
    raw = packed(kind, rng.normal(0, 0.05, (base, cols)).astype(np.float32))
    w = ops.WeightMatrix(kind, np.tile(np.ascontiguousarray(raw).view(np.uint8).ravel(), rows // base), rows, cols)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32)
    at = np.unique(np.r_[0:40, base - 40:base, rng.integers(0, base, 100)])
    dense = ops.WeightMatrix(kind, raw, base, cols)
    want = x.astype(np.float64) @ dense.dequantize()[at].astype(np.float64).T
    dense.free()
    try:
        _lib.check(lib.cthip_set_option(b"gemm_precision", precision))
        got = ops.linear(x, w)
    finally:
        _lib.check(lib.cthip_set_option(b"gemm_precision", 2))
    for first in {0, rows - base}:
        assert np.linalg.norm(got[:, first + at] - want) < 1e-5 * np.linalg.norm(want)
    w.free()


# dim, ffn, heads: but for the first three, matrices of each are large enough for the launch at the rows beside it
SHORT = [("llama", "q8_0", 512, 1024, 8, 2), ("llama", "q8_0", 512, 1024, 8, 3), ("llama", "q8_0", 512, 1024, 8, 7), ("llama", "q8_0", 2048, 5632, 32, 3), ("llama", "q4_0", 2048, 5632, 32, 7), ("llama", "f32", 2048, 2048, 16, 4),
         ("gpt2", "f16", 1152, 4608, 18, 6), ("gpt2", "f16", 1024, 4096, 16, 7), ("gpt2", "q8_0", 2816, 1024, 22, 12), ("llama", "q4_0", 2048, 5632, 32, 16),
         ("llama", "f16", 2048, 14848, 32, 17), ("llama", "f16", 2048, 14848, 32, 32)]


@pytest.mark.parametrize("arch,kind,dim,ffn,heads,rows", SHORT)
def test_short_prompt_equals_its_rows_one_by_one(ops, arch, kind, dim, ffn, heads, rows):
    """A prompt of a few rows (thirds of the fused projection stored and split, or routed to the cache rows) against the decode step."""
    from caten_amd import _lib, llm, synth
    if arch == "llama":
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=dim, ffn=ffn, n_heads=heads, n_kv_heads=heads // 4, n_layers=2 if ffn < 9000 else 1, vocab=1000, max_seq=700)
        model = llm.make_llama(cfg, llm.llama_state_dict(synth.llama_weights(cfg, seed=3), kind))
    else:
        cfg = dict(synth.GPT2_CONFIGS["gpt2-tiny"], dim=dim, ffn=ffn, n_heads=heads, vocab=1000, max_seq=700)
        model = llm.make_gpt2(cfg, llm.gpt2_state_dict(synth.gpt2_weights(cfg, seed=3), kind))
    ids = [float(t) for t in synth.prompt(cfg["vocab"], 640 + rows, seed=3)]
    lib = _lib.load()
    model.forward(ids[:640], 640, 0)
    got = [model.forward(ids[n:n + rows], rows, n, return_logits=True) for n in (5, 640)]  # a short and a long context
    try:
        _lib.check(lib.cthip_set_option(b"prefill_gemm", 0))
        model.forward(ids[5:5 + rows], rows, 5)
        model.forward(ids[5:640], 635, 5)
        want = [model.forward(ids[n:n + rows], rows, n, return_logits=True) for n in (5, 640)]
    finally:
        _lib.check(lib.cthip_set_option(b"prefill_gemm", 1))
    for (t0, l0), (t1, l1) in zip(got, want):
        assert t0 == t1
        assert np.linalg.norm(l0 - l1) < 1e-4 * np.linalg.norm(l1)
    model.close()


@pytest.mark.parametrize("arch,rows", [("gpt2", 8), ("gpt2", 12), ("llama", 12)])
def test_sessions_hold_the_same_rows_whatever_their_cache(oracle, arch, rows):
    """A prompt of a few rows takes the same launches over both kinds of cache (thirds routed to the cache rows, or stored and
    split): layer 0's Q8_0 rows are the quantised fp32 rows of the other session bit for bit."""
    from caten_amd import _lib, llm, synth
    lib = _lib.init(0)
    if arch == "gpt2":  # 8448 x 2816
        cfg = dict(synth.GPT2_CONFIGS["gpt2-tiny"], dim=2816, n_heads=22, ffn=256, n_layers=1, vocab=300)
        make, sd = llm.make_gpt2, llm.gpt2_state_dict(synth.gpt2_weights(cfg, seed=6), "q8_0")
    else:  # 8448 x 2816 likewise
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=2816, n_heads=22, n_kv_heads=22, ffn=256, n_layers=1, vocab=300)
        make, sd = llm.make_llama, llm.llama_state_dict(synth.llama_weights(cfg, seed=6), "q8_0")
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows, seed=6)]
    held = []
    try:
        for mode in (0, 1):
            _lib.check(lib.cthip_set_option(b"kv_cache", mode))
            model = make(cfg, sd)
            model.forward(ids, rows, 0)
            if mode == 0:
                held += [oracle.quantize("q8_0", model.peek(f"{c}_cache.0")[:rows * 2816]) for c in "kv"]
                held = [np.asarray(h).view(np.uint8).reshape(-1, 34) for h in held]
            else:
                for c, h in zip("kv", held):
                    assert np.array_equal(model.peek(f"{c}_cache_q8.0").view(np.uint8)[:rows * 2816].reshape(-1, 32), h[:, 2:])
                    assert np.array_equal(model.peek(f"{c}_cache_d.0").view(np.uint8)[:rows * 176].reshape(-1, 2), h[:, :2])
            model.close()
    finally:
        _lib.check(lib.cthip_set_option(b"kv_cache", 0))
