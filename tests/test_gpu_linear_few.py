"""Linears over 8 .. 64 rows as operands of two bf16 terms (csrc/linear_few.hip): every count of row blocks and of columns per workgroup, rows and
columns that fill none of them, shares of K from one block to two batches; through cthip_linear and through short prompts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from caten_amd import _lib, ops as o
    _lib.init(0)
    return o


@pytest.mark.parametrize("kind", ["q8_0", "q4_0", "f16"])
@pytest.mark.parametrize("rows,cols", [(260, 256), (768, 768), (2308, 1024), (4100, 1280), (516, 1600), (2564, 2048), (8196, 544), (11268, 2016)])
def test_linear_few(ops, kind, rows, cols):
    from caten_amd.llm import Tensor
    rng = np.random.default_rng(rows + cols)
    w = ops.WeightMatrix(kind, Tensor.from_f32(rng.normal(0, 0.05, (rows, cols)).astype(np.float32), kind).raw, rows, cols)
    wd = w.dequantize().astype(np.float64)
    g, beta = rng.normal(1, 0.1, cols).astype(np.float32), rng.normal(0, 0.1, cols).astype(np.float32)
    b = rng.normal(0, 1, rows).astype(np.float32)
    for m in (8, 16, 17, 32, 33, 48, 49, 63, 64):
        x, r = rng.normal(0.1, 1, (m, cols)).astype(np.float32), rng.normal(0, 1, (m, rows)).astype(np.float32)
        x[m - 1, cols - 1] = 20.0
        x64 = x.astype(np.float64)
        ln = (x64 - x64.mean(-1, keepdims=True)) / np.sqrt(x64.var(-1, keepdims=True) + 1e-5) * g + beta
        rms = x64 / np.sqrt((x64 * x64).mean(-1, keepdims=True) + 1e-5) * g
        # two terms an operand: 2^-16 of a product is dropped, 2.5e-6 (quantised) or 3.7e-6 (fp16) of the result is what that leaves of sums of many
        for got, want in ((ops.linear(x, w, b, r, act="relu", prologue="layernorm", norm_g=g, norm_b=beta), np.maximum(ln @ wd.T + b, 0) + r),
                          (ops.linear(x, w, None, r, prologue="rmsnorm", norm_g=g), rms @ wd.T + r), (ops.linear(x, w, b), x64 @ wd.T + b)):
            assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want), (m, np.linalg.norm(got - want) / np.linalg.norm(want))
            assert np.max(np.abs(got - want)) <= 1e-4 * np.max(np.abs(want))
    w.free()


@pytest.mark.parametrize("kv", [0, 2])
@pytest.mark.parametrize("arch,kind", [("gpt2", "f16"), ("gpt2", "q4_0"), ("llama", "q8_0"), ("llama", "f16")])
def test_short_prompts(ops, arch, kind, kv):
    """A prompt in one batch leaves what pieces of seven rows (single-row kernels, fp32 products) leave, at every count of row blocks."""
    from caten_amd import _lib, llm, synth
    lib = _lib.load()
    if arch == "llama":
        cfg = dict(synth.LLAMA_CONFIGS["llama-tiny"], dim=512, n_heads=8, n_kv_heads=2, ffn=1408, n_layers=3, vocab=500, max_seq=160)
        sd = llm.llama_state_dict(synth.llama_weights(cfg, seed=6), kind)
    else:
        cfg = dict(synth.GPT2_CONFIGS["gpt2"], dim=640, n_heads=10, n_layers=3, vocab=500, max_seq=160)
        sd = llm.gpt2_state_dict(synth.gpt2_weights(cfg, seed=6), kind)
    ids = [float(t) for t in synth.prompt(cfg["vocab"], 130, seed=6)]
    try:
        _lib.check(lib.cthip_set_option(b"kv_cache", kv))
        model = (llm.make_llama if arch == "llama" else llm.make_gpt2)(cfg, sd)
    finally:
        _lib.check(lib.cthip_set_option(b"kv_cache", 0))
    for rows in (8, 15, 31, 47, 64):
        t0, l0 = model.forward(ids[:rows], rows, 0, return_logits=True)
        t1, l1 = model.forward(ids[rows:rows + 1], 1, rows, return_logits=True)
        for n in range(0, rows, 7):
            want = model.forward(ids[n:min(n + 7, rows)], min(7, rows - n), n, return_logits=True)
        for (t, l), (u, k) in (((t0, l0), want), ((t1, l1), model.forward(ids[rows:rows + 1], 1, rows, return_logits=True))):
            assert t == u
            assert np.linalg.norm(l - k) < 1e-4 * np.linalg.norm(k)
    model.close()
