"""The single-row Linear by integer matrix instructions (csrc/gemv_int.hip): rows that are no multiple of 16, units of 128 bytes that
end inside a row, one wavefront's share of several units, one to many groups a workgroup; every prologue and epilogue it
carries; inputs of any magnitude; (gate, up) row pairs and the fused argmax through sessions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


def matrix(ops, kind, rows, cols, seed):
    from caten_amd.llm import Tensor
    rng = np.random.default_rng(seed)
    w = ops.WeightMatrix(kind, Tensor.from_f32(rng.normal(0, 0.05, (rows, cols)).astype(np.float32), kind).raw, rows, cols)
    return w, w.dequantize().astype(np.float64), rng


# Error of a sum of n products against 64 bits: the inputs' digits keep 2^-30 of their chunk's largest value, the scales and sums round in
# fp32, 2^-24 a step over at most 16 wavefronts x 6 units x 2 chunks of a lane: bounded by 2^-17 of the sum of magnitudes, seen at 1e-7 of the result.
# A step whose result is subnormal rounds by 2^-150 instead, at most 2^-142 over those 192 steps.
def close(got, want, scale):
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - want) <= 2.0 ** -17 * scale + 2.0 ** -142)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("kind,rows,cols", [("q4_0", 2563, 1024), ("q4_0", 2575, 1088), ("q4_0", 4096, 4096), ("q4_0", 2560, 11008), ("q4_0", 8207, 4160), ("q4_0", 8207, 4352), ("q4_0", 20011, 1600),
                                            ("q4_0", 50257, 1280), ("q4_0", 2561, 1216), ("q4_0", 12288, 2048)])
def test_linear(ops, kind, rows, cols):
    w, wd, rng = matrix(ops, kind, rows, cols, rows + cols)
    x = rng.normal(0.1, 1, cols).astype(np.float32)
    x[5], x[64:96] = 60.0, 0.0  # a large input among small ones, a chunk of zeros
    x[cols - 1] = 7.0           # next to the padding
    b, r, g = rng.normal(0, 1, rows).astype(np.float32), rng.normal(0, 1, rows).astype(np.float32), rng.normal(1, 0.1, cols).astype(np.float32)
    beta = rng.normal(0, 0.1, cols).astype(np.float32)
    x64 = x.astype(np.float64)
    aw = np.abs(wd)
    close(ops.linear(x, w), wd @ x64, aw @ np.abs(x64))
    close(ops.linear(x, w, b, r, act="relu"), np.maximum(wd @ x64 + b, 0) + r, aw @ np.abs(x64) + np.abs(b) + np.abs(r))
    n = x64 / np.sqrt((x64 * x64).mean() + 1e-5) * g
    close(ops.linear(x, w, None, r, prologue="rmsnorm", norm_g=g), wd @ n + r, aw @ np.abs(n) + np.abs(r))
    if cols <= 4096:
        w.fold_layernorm(g, beta, b)
        n = (x64 - x64.mean()) / np.sqrt(x64.var() + 1e-5) * g
        got = w.linear_folded(x)
        want = wd @ (n + beta) + b
        assert np.linalg.norm(got - want) <= 3e-6 * np.linalg.norm(want)  # (the mean's part is taken off behind the product)
    w.free()


# A folded LayerNorm with no bias of its own takes the mean off the vector: integers about a mean whose sums are exact in fp32 in any order, so that the error
# is that of the product however many deviations the mean is (taken off behind the product: that many times as much, 1e-4 at the last).
@pytest.mark.parametrize("kind,rows,cols", [("q4_0", 6500, 1280), ("q4_0", 20011, 1600), ("q4_0", 2600, 4096), ("q4_0", 2575, 1088)])
def test_a_mean_of_many_deviations(ops, kind, rows, cols):
    w, wd, rng = matrix(ops, kind, rows, cols, rows + cols)
    g, beta = rng.normal(1, 0.1, cols).astype(np.float32), rng.normal(0, 0.1, cols).astype(np.float32)
    w.fold_layernorm(g, beta)
    d = rng.integers(-3, 4, cols // 2)
    d = rng.permutation(np.concatenate([d, -d])).astype(np.float64)
    want = wd @ (d / np.sqrt((d * d).mean() + 1e-5) * g + beta)
    for mean in (0, -64, 2047):  # 2047 x 4096 < 2^23
        got = w.linear_folded((mean + d).astype(np.float32))
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want), mean
    w.free()


@pytest.mark.parametrize("kind,rows,cols", [("q4_0", 2600, 1024)])
@pytest.mark.parametrize("scale", [1e-38, 1e-37, 1e-35, 1e-33, 1e-30, 1e-12, 1e12, 1e30, 1e36])
def test_inputs_of_any_magnitude(ops, kind, rows, cols, scale):
    w, wd, rng = matrix(ops, kind, rows, cols, 3)
    x = (rng.normal(0, 1, cols) * scale).astype(np.float32)
    x[:32] *= np.float32(1e-6)  # a chunk of its own magnitude (of subnormal numbers at the small end)
    close(ops.linear(x, w), wd @ x.astype(np.float64), np.abs(wd) @ np.abs(x.astype(np.float64)))
    w.free()


@pytest.mark.parametrize("kind,rows,cols", [("q4_0", 2600, 1024)])
def test_inputs_that_are_not_finite(ops, kind, rows, cols):
    w, wd, rng = matrix(ops, kind, rows, cols, 4)
    x = rng.normal(0, 1, cols).astype(np.float32)
    x[40] = np.inf
    got, with_weight = ops.linear(x, w), wd[:, 40] != 0
    assert np.array_equal(got[with_weight], np.sign(wd[with_weight, 40]) * np.inf) and np.all(np.isnan(got[~with_weight]))
    x[40] = np.nan
    assert np.all(np.isnan(ops.linear(x, w)))
    # several in one block of 32: never a finite number or an infinity where products of both signs (or of a zero weight) meet
    for a, b in ((np.inf, np.inf), (np.inf, -np.inf), (-np.inf, -np.inf)):
        x[40], x[61] = a, b
        with np.errstate(invalid="ignore"):
            want = wd[:, 40] * a + wd[:, 61] * b
        got = ops.linear(x, w)
        assert np.all(np.isnan(got[np.isnan(want)])) and not np.any(np.isfinite(got))
    # ... and in two blocks: as of floats
    x[61], x[64 + 61] = 1.0, -np.inf
    with np.errstate(invalid="ignore"):
        want = wd[:, 40] * x[40] + wd[:, 64 + 61] * x[64 + 61]
    assert np.array_equal(ops.linear(x, w), want.astype(np.float32), equal_nan=True)
    w.free()


@pytest.mark.parametrize("arch,kind", [("llama", "q4_0"), ("gpt2", "q4_0")])
def test_sessions_match_the_vector_kernels(ops, arch, kind):
    from caten_amd import _lib, llm, synth
    lib = _lib.load()
    if arch == "llama":  # (dim 1024: no three-launch layer, 8192 gate|up rows in pairs)
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=1024, n_heads=8, n_kv_heads=8, ffn=4096, n_layers=2, vocab=4099, max_seq=128)
        sd = llm.llama_state_dict(synth.llama_weights(cfg, seed=5), kind)
    else:                # (dim 1280: a launch per Linear, LayerNorm folded)
        cfg = dict(synth.GPT2_CONFIGS["gpt2"], dim=1280, n_heads=20, n_layers=2, vocab=6500, max_seq=128)
        sd = llm.gpt2_state_dict(synth.gpt2_weights(cfg, seed=5), kind)
    prompt, runs = synth.prompt(cfg["vocab"], 9, seed=5), []
    try:
        for wide in (1, 0):
            _lib.check(lib.cthip_set_option(b"gemv_wide", wide))
            model = (llm.make_llama if arch == "llama" else llm.make_gpt2)(cfg, sd)
            tokens, logits = llm.gpt2_generate(model, prompt, 10, on_device=False, keep_logits=True)
            model.close()
            model = (llm.make_llama if arch == "llama" else llm.make_gpt2)(cfg, sd)
            assert llm.gpt2_generate(model, prompt, 10, on_device=True) == tokens
            model.close()
            runs.append((tokens, logits))
    finally:
        _lib.check(lib.cthip_set_option(b"gemv_wide", 1))
    assert runs[0][0] == runs[1][0]
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)


# The three-launch layer's MLP: a workgroup to 32 hidden units, one of them, an odd number, whole rounds and a last one.  Against a launch per Linear: hidden units and
# down projection are sums of 2048 and ffn products, off by at most (n + 2) 2^-24 of their terms' magnitudes on either side, which are a few times the sums here; two layers and the head.
@pytest.mark.parametrize("ffn", [32, 96, 1120])
def test_layers_of_slabs_match_a_launch_per_linear(ffn):
    print(f"case: three-launch layer, {ffn} hidden units", flush=True)
    from caten_amd import _lib, llm, synth
    lib = _lib.load()
    cfg = dict(synth.LLAMA_CONFIGS["llama-1.1b"], ffn=ffn, n_layers=2, vocab=1003, max_seq=64)
    sd = llm.llama_state_dict(synth.llama_weights(cfg, seed=17), "q4_0")
    prompt, runs = synth.prompt(cfg["vocab"], 7, seed=17), []
    try:
        for fused in (1, 0):
            _lib.check(lib.cthip_set_option(b"decode_fused", fused))
            model = llm.make_llama(cfg, sd)
            runs.append(llm.gpt2_generate(model, prompt, 8, on_device=False, keep_logits=True))
            model.close()
    finally:
        _lib.check(lib.cthip_set_option(b"decode_fused", 1))
    assert runs[0][0] == runs[1][0]
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)


def test_slabs_whose_large_values_meet_weights_of_zero(ops):
    """A layer of slabs whose MLP has channels a thousand times as large that gate, up and down do not read: its digits, 30 bits below a chunk's largest value, against the
    same model in fp32.  The launch per Linear takes nibbles times inputs less eight times the inputs' sum, which has 24 bits below the largest."""
    print("case: three-launch layer, large channels", flush=True)
    from caten_amd import _lib, llm, synth
    lib = _lib.load()
    cfg = dict(synth.LLAMA_CONFIGS["llama-1.1b"], ffn=1120, n_layers=2, vocab=1003, max_seq=64)
    w, rng = synth.llama_weights(cfg, seed=17), np.random.default_rng(2)
    ch, ff = (np.arange(0, n, 32) + rng.integers(0, 32, n // 32) for n in (cfg["dim"], cfg["ffn"]))
    for l in range(2):
        w["ffn_norm"][l][ch] *= 1000.0
        w["w_up"][l][ff] *= 1000.0
        w["w_gate"][l][:, ch] = w["w_up"][l][:, ch] = 0.0
        w["w_down"][l][:, ff] = 0.0
    sd = llm.llama_state_dict(w, "q4_0")
    exact = {k: llm.Tensor.from_f32(ops.WeightMatrix(t.kind, t.raw, t.rows, t.cols).dequantize()) if t.kind == "q4_0" else t for k, t in sd.items()}
    prompt, last = synth.prompt(cfg["vocab"], 2, seed=17), []
    try:
        for fused, d in ((1, sd), (0, sd), (0, exact)):
            _lib.check(lib.cthip_set_option(b"decode_fused", fused))
            model = llm.make_llama(cfg, d)
            model.forward(prompt[:1], 1, 0)
            last.append(model.forward(prompt[1:], 1, 1, return_logits=True)[1].astype(np.float64))
            model.close()
    finally:
        _lib.check(lib.cthip_set_option(b"decode_fused", 1))
    digits, vector = (np.linalg.norm(x - last[2]) / np.linalg.norm(last[2]) for x in last[:2])
    print("digits", digits, "vector kernels", vector, flush=True)
    assert digits <= vector and digits <= 1e-5
