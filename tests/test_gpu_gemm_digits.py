"""Linears over many rows on 4-bit weights, whose operands lie as 6-bit digits (csrc/gemm_digits.hip): every tile, with one share of K and several, at edges that
no tile divides and odd numbers of blocks; rows of any magnitude and rows that are not finite; prompts, whose norms, attention and GELU / SwiGLU write digits; values that are small beside others of their block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


def weights(ops, rows, cols, rng):
    from caten_amd.llm import Tensor
    return ops.WeightMatrix("q4_0", Tensor.from_f32(rng.normal(0, 0.05, (rows, cols)).astype(np.float32), "q4_0").raw, rows, cols)


def bound(x, w):
    """2^-19 of the largest value of a block of 32 goes with every value of it (csrc/digits.h), and fp32 sums of at most K terms, here in runs of 32, round K / 32 + 32 times."""
    xb, wb = np.abs(x).reshape(len(x), -1, 32), np.abs(w).reshape(len(w), -1, 32)
    return 2.0 ** -19 * xb.max(-1) @ wb.sum(-1).T + (x.shape[1] / 32 + 32) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)


# tile 64 x 64 with 1, 3, 5 shares; 64 x 128 with few workgroups (1, 2, 4, 7 shares) and many (the line behind them too); 128 x 128 with 1 and 3 shares (the last line)
@pytest.mark.parametrize("rows,cols,m", [(3001, 64, 2049), (9001, 64, 701), (1026, 4128, 513), (514, 8224, 577),
                                         (6401, 96, 577), (2051, 288, 1025), (4100, 4128, 129), (6401, 4128, 65), (4100, 8224, 97), (6401, 64, 1537),
                                         (12001, 288, 1537), (3001, 544, 2049), (2051, 8224, 701), (2051, 8224, 577),
                                         (9001, 1056, 641), (12001, 544, 1537), (9001, 8224, 193)])
def test_linear_digits(ops, rows, cols, m):
    rng = np.random.default_rng(rows + m)
    w = weights(ops, rows, cols, rng)
    x = rng.normal(0, 1, (m, cols)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (m, 1))).astype(np.float32)
    x[:, ::37] *= 50.0
    at, rs = np.unique(np.r_[0:40, rows - 40:rows, rng.integers(0, rows, 60)]), np.unique(np.r_[0:9, m - 9:m, rng.integers(0, m, 40)])
    x64, w64 = x[rs].astype(np.float64), w.dequantize()[at].astype(np.float64)
    want, most = x64 @ w64.T, bound(x64, w64)
    for _ in range(2):  # with the matrix's digits made, and as they are kept
        got = ops.linear(x, w)[np.ix_(rs, at)]
        assert np.all(np.abs(got - want) <= most)
    bias, res = rng.normal(0, 1, rows).astype(np.float32), rng.normal(0, 1, (m, rows)).astype(np.float32)
    ends = 4 * 2.0 ** -24 * (np.abs(want) + np.abs(bias[at]) + np.abs(res[rs][:, at]))
    got = ops.linear(x, w, bias, res)[np.ix_(rs, at)]
    assert np.all(np.abs(got - (want + bias[at] + res[rs][:, at])) <= most + ends)
    got = ops.linear(x, w, bias, act="relu")[np.ix_(rs, at)]
    assert np.all(np.abs(got - np.maximum(want + bias[at], 0.0)) <= most + ends)
    w.free()


def test_rows_of_any_magnitude_and_rows_that_are_not_finite(ops):
    rng = np.random.default_rng(5)
    w = weights(ops, 4100, 4128, rng)
    w64 = w.dequantize().astype(np.float64)
    x = rng.normal(0, 1, (129, 4128)).astype(np.float32)
    scale = np.array([1e-25, 1e-20, 1e-10, 1.0, 1e10, 1e30, 1e33] * 19)[:129]  # (1e-25: every digit of a block is a normal power of two)
    x = (x * scale[:, None]).astype(np.float32)
    x[7] = 0.0
    x[8, 100:] = 0.0
    x[40, 5], x[41, 4127], x[42, 64] = np.inf, -np.inf, np.nan
    got = ops.linear(x, w)
    odd = np.arange(129)[~np.isfinite(x).all(1)]
    assert list(odd) == [40, 41, 42]
    assert np.isnan(got[odd]).all()
    fine = np.setdiff1d(np.arange(129), odd)
    x64 = x[fine].astype(np.float64)
    assert np.all(np.abs(got[fine] - x64 @ w64.T) <= bound(x64, w64))
    assert not got[7].any()
    w.free()


@pytest.mark.parametrize("arch,kinds,rows", [("gpt2", ("q4_0", "q4_0"), 65), ("gpt2", ("q4_0", "q4_0"), 223), ("gpt2", ("q4_0", "q4_0"), 897), ("gpt2", ("q4_0", "q8_0"), 700),
                                             ("gpt2", ("q8_0", "q4_0"), 700), ("llama", ("q4_0", "q4_0"), 96), ("llama", ("q4_0", "q4_0"), 333), ("llama", ("q4_0", "q8_0"), 1300)])
def test_prompt_equals_short_pieces(ops, arch, kinds, rows):
    """kinds: of the Linears behind a norm, and of the attention projection and the second MLP Linear; pieces of 63 rows take other kernels."""
    from caten_amd import llm, synth
    if arch == "llama":
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=1024, n_heads=16, n_kv_heads=4, ffn=2816, n_layers=3, vocab=500, max_seq=2048)
        w = synth.llama_weights(cfg, seed=3)
        make, dicts = llm.make_llama, [llm.llama_state_dict(w, k) for k in kinds]
    else:
        cfg = dict(synth.GPT2_CONFIGS["gpt2"], dim=1024, n_heads=16, n_layers=3, vocab=500, max_seq=2048)
        w = synth.gpt2_weights(cfg, seed=3)
        make, dicts = llm.make_gpt2, [llm.gpt2_state_dict(w, k) for k in kinds]
    behind = ("attn.c_proj.weight", "mlp.c_proj.weight", "attention.wo.weight", "feed_forward.w2.weight")
    model = make(cfg, {k: dicts[1][k] if k.endswith(behind) else dicts[0][k] for k in dicts[0]})
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows + 1, seed=3)]
    got = [model.forward(ids[:rows], rows, 0, return_logits=True), model.forward(ids[rows:], 1, rows, return_logits=True)]
    for n in range(0, rows, 63):
        want = [model.forward(ids[n:min(n + 63, rows)], min(63, rows - n), n, return_logits=True)]
    want.append(model.forward(ids[rows:], 1, rows, return_logits=True))
    for (t0, l0), (t1, l1) in zip(got, want):
        assert t0 == t1
        assert np.linalg.norm(l0 - l1) < 1e-4 * np.linalg.norm(l1)
    model.close()


def terms_bound(x, w):
    """What two bf16 terms of every value leave: 2^-18 of each, and fp32 sums as in bound(); values whose terms end below 2^-126, where the matrix cores have zero."""
    return (2.0 ** -18 + (x.shape[1] / 32 + 32) * 2.0 ** -24) * (np.abs(x) @ np.abs(w).T) + 2.0 ** -124 * np.abs(w).sum(-1)


# columns of a block of 32 that are larger, by how much, in which rows; 2^18 (digits of a small value all zero) and what a model's own largest channels are
@pytest.mark.parametrize("cols_large,factor,rows_large", [(1, 1e3, "all"), (4, 700.0, "all"), (16, 1e3, "all"), (24, 2.0 ** 18, "all"), (31, 2.0 ** 16, "all"), (1, 1e3, "one"), (1, 2.0 ** 26, "few"), (0, 1.0, "wide")])
@pytest.mark.parametrize("rows,cols,m", [(3001, 288, 577), (2051, 4128, 129), (4100, 1056, 65), (9001, 544, 1537)])
def test_results_that_the_large_values_do_not_reach(ops, rows, cols, m, cols_large, factor, rows_large):
    """Weights of zero at the large columns: the results are sums of small values alone, and as near as two terms of every value make them.  "wide": values of exp(6 x)."""
    from caten_amd.llm import Tensor
    print(f"case: {rows} x {cols}, {m} rows, {cols_large} columns of 32, {factor}, {rows_large}", flush=True)
    rng = np.random.default_rng(rows + cols_large)
    a = rng.normal(0, 0.05, (rows, cols)).astype(np.float32)
    large = np.zeros(cols, bool)
    for b in range(cols // 32):
        large[32 * b + rng.permutation(32)[:cols_large]] = True
    a[:, large] = 0.0
    w = ops.WeightMatrix("q4_0", Tensor.from_f32(a, "q4_0").raw, rows, cols)
    x = rng.uniform(0.5, 1.0, (m, cols)) * rng.choice([-1.0, 1.0], (m, cols))
    at_rows = np.ones(m, bool) if rows_large == "all" else np.arange(m) % 32 == 5 if rows_large == "one" else np.arange(m) % 7 == 3
    x[np.ix_(at_rows, large)] *= factor
    if rows_large == "wide":
        x = np.exp(6.0 * rng.normal(0, 1, (m, cols))) * np.sign(x)
        x[:, ::2] = 0.0
    x = x.astype(np.float32)
    at, rs = np.unique(np.r_[0:20, rows - 20:rows, rng.integers(0, rows, 40)]), np.unique(np.r_[0:9, m - 9:m, rng.integers(0, m, 60), np.flatnonzero(at_rows)[:9]])
    x64, w64 = x[rs].astype(np.float64), w.dequantize()[at].astype(np.float64)
    assert not w64[:, large].any()
    got = ops.linear(x, w)[np.ix_(rs, at)]
    most = terms_bound(x64, w64) if rows_large != "wide" else bound(x64, w64)
    assert np.all(np.abs(got - x64 @ w64.T) <= most)
    if rows_large == "wide":  # blocks that have no terms lose less than twice what those that have them keep
        assert np.linalg.norm((got - x64 @ w64.T) / (np.abs(x64) @ np.abs(w64).T)) <= 2.0 * 2.0 ** -18 * np.sqrt(got.size)
    w.free()


def test_rows_beside_rows_that_are_not_finite(ops):
    """One row of every 32 is infinities or NaNs, one is past 2^127: the others' small values are as near as without them."""
    from caten_amd.llm import Tensor
    rng = np.random.default_rng(9)
    rows, cols, m = 4100, 1056, 129
    a = rng.normal(0, 0.05, (rows, cols)).astype(np.float32)
    a[:, 7::8] = 0.0
    w = ops.WeightMatrix("q4_0", Tensor.from_f32(a, "q4_0").raw, rows, cols)
    x = (rng.uniform(0.5, 1.0, (m, cols)) * rng.choice([-1.0, 1.0], (m, cols))).astype(np.float32)
    x[:, 7::8] *= 1000.0  # (one in a block would be found by its row alone)
    x[3::32], x[3::64, 9:] = np.nan, np.inf
    x[11::32] *= np.float32(2.0 ** 117)
    assert np.abs(x[11]).max() >= 2.0 ** 126
    fine = np.setdiff1d(np.arange(m), np.arange(3, m, 32))
    x64, w64 = x[fine].astype(np.float64), w.dequantize().astype(np.float64)
    got = ops.linear(x, w)
    assert np.isnan(got[3::32]).all()
    assert np.all(np.abs(got[fine] - x64 @ w64.T) <= terms_bound(x64, w64))
    w.free()


def test_rows_of_the_smallest_magnitudes(ops):
    """Below 2^-110 a digit's power of two would end past the smallest: what is left goes as terms."""
    rng = np.random.default_rng(8)
    w = weights(ops, 4100, 1056, rng)
    w64 = w.dequantize().astype(np.float64)
    x = rng.normal(0, 1, (129, 1056)) * np.array([1e-32, 1e-33, 1e-34, 1e-35, 1e-36, 1e-37, 1.0])[np.arange(129) % 7][:, None]
    x = x.astype(np.float32)
    x64 = x.astype(np.float64)
    got = ops.linear(x, w)
    assert np.all(np.abs(got - x64 @ w64.T) <= np.maximum(bound(x64, w64), terms_bound(x64, w64)))
    w.free()


@pytest.mark.parametrize("arch,rows", [("gpt2", 97), ("gpt2", 700), ("llama", 96), ("llama", 1300)])
def test_prompt_with_large_channels(arch, rows):
    """A model whose norms, attention and MLP each have a few channels a thousand times as large that the Linears behind do not read (weights of zero there): what norms, attention and the
    GELU / SwiGLU launches write carries the others as well as pieces of 63 rows do, whose inputs are two terms or fp32."""
    print(f"case: {arch}, {rows} rows", flush=True)
    from caten_amd import llm, synth
    cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=1024, n_heads=16, n_kv_heads=4, ffn=2816) if arch == "llama" else dict(synth.GPT2_CONFIGS["gpt2"], dim=1024, n_heads=16)
    cfg.update(n_layers=3, vocab=500, max_seq=2048)
    w = (synth.llama_weights if arch == "llama" else synth.gpt2_weights)(cfg, seed=3)
    rng = np.random.default_rng(1)
    D, F, H, HK = cfg["dim"], cfg["ffn"], cfg["n_heads"], cfg.get("n_kv_heads", cfg["n_heads"])
    Dh = D // H
    pick = lambda n: np.arange(0, n, 32) + rng.integers(0, 32, n // 32)  # noqa: E731  (one of every 32)
    ch, ff, vh = pick(D), pick(F), pick(HK * Dh)
    oh = np.concatenate([h * Dh + vh[vh // Dh == h // (H // HK)] % Dh for h in range(H)])  # where the attention's result has them
    keys = dict(n1="attn_norm", n2="ffn_norm", qkv=("wq", "wk", "wv"), v="wv", o="wo", fc=("w_gate", "w_up"), up="w_up", down="w_down") if arch == "llama" else \
        dict(n1="ln1_g", n2="ln2_g", qkv=("attn_w",), v="attn_w", o="proj_w", fc=("fc_w",), up="fc_w", down="fc2_w")
    for l in range(3):
        for norm, behind in ((keys["n1"], keys["qkv"]), (keys["n2"], keys["fc"])):
            w[norm][l][ch] *= 1000.0
            for k in behind:
                w[k][l][:, ch] = 0.0
        w[keys["v"]][l][(0 if arch == "llama" else 2 * D) + vh] *= 1000.0
        w[keys["o"]][l][:, oh] = 0.0
        w[keys["up"]][l][ff] *= 1000.0
        w[keys["down"]][l][:, ff] = 0.0
    sd = (llm.llama_state_dict if arch == "llama" else llm.gpt2_state_dict)(w, "q4_0")
    make = llm.make_llama if arch == "llama" else llm.make_gpt2
    model = make(cfg, sd)
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows + 1, seed=3)]
    got = [model.forward(ids[:rows], rows, 0, return_logits=True), model.forward(ids[rows:], 1, rows, return_logits=True)]
    for n in range(0, rows, 63):
        want = [model.forward(ids[n:min(n + 63, rows)], min(63, rows - n), n, return_logits=True)]
    want.append(model.forward(ids[rows:], 1, rows, return_logits=True))
    # the last row's single-row Linears, which take nibbles times inputs less eight times the inputs' sum, are off by up to 1e-4 of these logits on either side
    for (t0, l0), (t1, l1) in zip(got, want):
        assert np.linalg.norm(l0 - l1) < 2e-4 * np.linalg.norm(l1)
    model.close()


@pytest.mark.parametrize("arch,rows", [("gpt2", 97), ("gpt2", 700), ("llama", 96), ("llama", 1300)])
def test_prompt_behind_a_norm_with_most_channels_large(arch, rows):
    """Norms in front of the attention that leave 24 of 32 channels 256 times as large, which q, k and v do not read: rows by themselves say which blocks have the rest as terms.  Against the
    pieces of 63 rows of test_prompt_with_large_channels: two terms are off by 2.5e-6 a Linear, twelve on either side by 1.2e-5, and as much again
    for scores of some size."""
    print(f"case: {arch}, {rows} rows", flush=True)
    from caten_amd import llm, synth
    cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=1024, n_heads=16, n_kv_heads=4, ffn=2816) if arch == "llama" else dict(synth.GPT2_CONFIGS["gpt2"], dim=1024, n_heads=16)
    cfg.update(n_layers=3, vocab=500, max_seq=2048)
    w = (synth.llama_weights if arch == "llama" else synth.gpt2_weights)(cfg, seed=3)
    rng = np.random.default_rng(1)
    large = np.concatenate([32 * b + rng.permutation(32)[:24] for b in range(cfg["dim"] // 32)])
    norm, behind = ("attn_norm", ("wq", "wk", "wv")) if arch == "llama" else ("ln1_g", ("attn_w",))
    for l in range(3):
        w[norm][l][large] *= 256.0
        for k in behind:
            w[k][l] *= 2.0  # (a quarter of the columns is left)
            w[k][l][:, large] = 0.0
    model = (llm.make_llama if arch == "llama" else llm.make_gpt2)(cfg, (llm.llama_state_dict if arch == "llama" else llm.gpt2_state_dict)(w, "q4_0"))
    ids = [float(t) for t in synth.prompt(cfg["vocab"], rows, seed=3)]
    got = model.forward(ids, rows, 0, return_logits=True)[1]
    for n in range(0, rows, 63):
        want = model.forward(ids[n:n + 63], min(63, rows - n), n, return_logits=True)[1]
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("off by", off, flush=True)
    assert off < 2.5e-5
    model.close()


def test_both_forms_of_a_matrix_are_kept(ops):
    """A 4-bit matrix is integers in bf16 to Linears at one term and digits at two: each form is made once and stays; with room for one of them alone, the one in use takes the other's."""
    import ctypes as C
    from caten_amd import _lib
    lib = _lib.init(0)
    rows, cols = 5001, 2048
    form = {1: rows * cols // 32 * 64, 2: (rows + 31) // 32 * (cols // 32) * 1024}  # 20.5 and 10.3 MB
    w = weights(ops, rows, cols, np.random.default_rng(1))
    x = np.random.default_rng(2).normal(0, 1, (3000, cols)).astype(np.float32)  # (rows that pay for the form at every call)

    def live():
        a, b, c = C.c_size_t(), C.c_size_t(), C.c_size_t()
        _lib.check(lib.cthip_cache_stats(C.byref(a), C.byref(b), C.byref(c)))
        return a.value

    def run(precision):
        _lib.check(lib.cthip_set_option(b"gemm_precision", precision))
        return ops.linear(x, w)

    try:
        _lib.check(lib.cthip_set_option(b"weight_planes", 0))
        none, want = live(), {p: run(p) for p in (1, 2)}
        assert live() == none
        for limit, both in ((256, True), (24, False)):
            _lib.check(lib.cthip_cache_trim())
            _lib.check(lib.cthip_set_option(b"weight_planes", limit))
            held = {1: 0, 2: 0}
            for p in (2, 1, 2, 1, 1, 2):
                assert np.array_equal(run(p), want[p])
                held = {q: form[q] if q == p or (both and held[q]) else 0 for q in held}
                assert sum(held.values()) <= live() - none <= sum(held.values()) * 1.25, (limit, p)  # (blocks come in size classes)
    finally:
        _lib.check(lib.cthip_set_option(b"gemm_precision", 2))
        _lib.check(lib.cthip_set_option(b"weight_planes", 32768))
    w.free()


@pytest.mark.parametrize("rows,cols,m", [(1026, 4128, 513), (6401, 96, 577)])
def test_rows_at_any_alignment(ops, rows, cols, m):
    """Input rows that do not lie on 16 bytes take the same launches as rows that do: the same results."""
    from caten_amd import _lib
    lib = _lib.init(0)
    rng = np.random.default_rng(4)
    w, x = weights(ops, rows, cols, rng), rng.normal(0, 1, (m, cols)).astype(np.float32)
    dx, dy = ops.DeviceArray((m * cols + 4,)), ops.DeviceArray((m, rows))
    want = ops.linear(x, w)
    for off in (4, 8, 12):
        _lib.check(lib.cthip_h2d(dx.ptr + off, x.ctypes.data, x.nbytes))
        _lib.check(lib.cthip_linear(dy.ptr, w.handle, dx.ptr + off, m, None, None, 0, 0, None, None, 0.0))
        assert np.array_equal(dy.numpy(), want), off
    w.free()
