"""What a user of this framework has it do, as cases that can be timed: decoding and prompts through a decoder session,
the two Linears of an MLP on packed weights, matrix products, row operations, and a whole model as a compiled graph.

Each case is one family at one size.  `listed()` holds the cases that are looked at by name, `draw()` gives further ones
of the same ranges, `prepare()` makes what a program has in hand before the call, `run()` is the call, `work()` what it
cannot do without and `tolerance()` how far two correct implementations may be apart.

Shapes are those of caten_amd.synth and of the repository's benchmarks; weights are drawn ~N(0, 0.02) and stored as a GGUF
file stores them.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from caten_amd import _lib, graphs, llm, ops, synth

# the models that sessions are opened for: GPT-2 sizes and Llama-shaped ones (the 7B shape of the size benchmark)
MODELS = {name: dict(synth.GPT2_CONFIGS[name], arch="gpt2") for name in ("gpt2", "gpt2-medium", "gpt2-large", "gpt2-xl", "gpt2-mini")}
MODELS["llama-1.1b"] = dict(synth.LLAMA_CONFIGS["llama-1.1b"], arch="llama")
MODELS["llama-7b"] = dict(n_layers=32, n_heads=32, n_kv_heads=32, dim=4096, ffn=11008, vocab=32000, max_seq=2048, eps=1e-5,
                          rope_base=10000.0, arch="llama")
BYTES = {"f32": 4.0, "f16": 2.0, "q8_0": 34.0 / 32.0, "q4_0": 18.0 / 32.0}  # of one stored weight
PRECISIONS = {"fp32": 0, "bf16": 1, "bf16x3": 2, "bf16x6": 3}  # operand formats of cthip_matmul
UNARY = {"gelu": _lib.ACT_GELU, "silu": _lib.ACT_SILU}
EPS = 1e-5


def listed():
    return [
        # ---- a session's greedy loop, one token after the other: the host asks for the next `steps` tokens ----
        # the headline: GPT-2 small from a Q8_0 file, early in a conversation; bound by launches and latencies
        dict(name="decode gpt2 q8_0", family="decode", model="gpt2", kind="q8_0", kv=0, pos=20, steps=24),
        # a small chat model from a Q4_0 file far into its context
        dict(name="decode llama-1.1b q4_0 long", family="decode", model="llama-1.1b", kind="q4_0", kv=0, pos=1501, steps=16),
        # a 7B model with its cache kept as Q8_0 rows: what a step reads is what counts
        dict(name="decode llama-7b q4_0 kvq", family="decode", model="llama-7b", kind="q4_0", kv=1, pos=203, steps=8),
        # ---- a prompt (or the next piece of one) as one batch ----
        # half a context of GPT-2 small
        dict(name="prompt gpt2 q8_0 512", family="prompt", model="gpt2", kind="q8_0", kv=0, pos=0, rows=512),
        # a document in front of a question: nearly the whole context
        dict(name="prompt llama-1.1b q4_0 1900", family="prompt", model="llama-1.1b", kind="q4_0", kv=0, pos=0, rows=1900),
        # the user's next turn: a few dozen tokens behind a cached conversation
        dict(name="prompt gpt2-medium f16 turn", family="prompt", model="gpt2-medium", kind="f16", kv=0, pos=301, rows=37),
        # ---- the MLP of a layer on packed weights: a handful of sequences decoded together ----
        dict(name="mlp 4096x11008 q8_0 m5", family="mlp", arch="llama", dim=4096, ffn=11008, kind="q8_0", rows=5),
        # ---- relu(matmul), the repository's first benchmark item, and a product that fills the card, ragged ----
        dict(name="matmul 1024 bf16x6 relu", family="matmul", m=1024, n=1024, k=1024, precision="bf16x6", relu=True),
        dict(name="matmul 3000x4100x5000 bf16x3", family="matmul", m=3000, n=4100, k=5000, precision="bf16x3", relu=False),
        # ---- row operations: the (64,1024,768) benchmark tensor, and the last step of sampling one token ----
        dict(name="rows ln_softmax 65536x768", family="rows", op="ln_softmax", rows=65536, n=768),
        dict(name="rows sample 1x50257", family="rows", op="sample", rows=1, n=50257),
        # ---- GPT-2 small as a compiled graph, node by node: a short prompt and the tokens after it ----
        dict(name="graph gpt2", family="graph", model="gpt2", rows=16, steps=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _linears(c):
    """(weights per layer, weights of the head)"""
    d, f = c["dim"], c["ffn"]
    kd = d // c["n_heads"] * c.get("n_kv_heads", c["n_heads"])
    per = d * (d + 2 * kd) + d * d + (2 if c["arch"] == "gpt2" else 3) * d * f
    return per, c["vocab"] * d


def draw(rng):
    family = rng.choice(["decode", "prompt", "prompt", "mlp", "matmul", "rows", "graph"])
    if family == "decode":
        model = rng.choice(["gpt2", "gpt2-medium", "gpt2-large", "gpt2-xl", "llama-1.1b", "llama-7b"])
        kind = "q4_0" if model == "llama-7b" else rng.choice(["q8_0", "q4_0", "f16", "f32"] if model != "llama-1.1b" else ["q8_0", "q4_0", "f16"])
        pos = _log(rng, 1, MODELS[model]["max_seq"] - 100)
        return dict(family=family, model=model, kind=kind, kv=rng.choice([0, 0, 1, 2]), pos=pos, steps=rng.randint(6, 12))
    if family == "prompt":
        model = rng.choice(["gpt2", "gpt2-medium", "gpt2-large", "llama-1.1b", "llama-7b"])
        kind = "q4_0" if model == "llama-7b" else rng.choice(["q8_0", "q4_0", "f16"])
        c = MODELS[model]
        top = min(c["max_seq"] - 100, int(1900 * 0.97e9 / (_linears(c)[0] * c["n_layers"])))
        rows = _log(rng, 2, top)
        pos = rng.choice([0, _log(rng, 1, c["max_seq"] - rows - 50)])
        return dict(family=family, model=model, kind=kind, kv=rng.choice([0, 0, 1, 2]), pos=pos, rows=rows)
    if family == "mlp":
        arch, kind = rng.choice(["gpt2", "llama"]), rng.choice(["q8_0", "q4_0", "f16", "f32"])
        dim = 32 * _log(rng, 8, 160)
        ffn = 32 * max(1, int(dim * rng.uniform(2.5, 4.0)) // 32)
        return dict(family=family, arch=arch, dim=dim, ffn=ffn, kind=kind, rows=_log(rng, 1, 2048))
    if family == "matmul":
        m, n, k = (_log(rng, 16, 5000) for _ in range(3))
        return dict(family=family, m=m, n=n, k=k, precision=rng.choice(list(PRECISIONS)), relu=rng.random() < 0.5)
    if family == "rows":
        op = rng.choice(["ln_softmax", "sample", "ln_gelu", "rms_silu"])
        n = _log(rng, 40, 8000) if op != "sample" else _log(rng, 1000, 50257)
        return dict(family=family, op=op, rows=_log(rng, 1, min(65536, 50_000_000 // n)), n=n)
    return dict(family=family, model=rng.choice(["gpt2", "gpt2-mini"]), rows=_log(rng, 1, 64), steps=rng.randint(4, 12))


# ---------------------------------------------------------------------------------------------------------------------
# inputs


def _normal(g, *shape, mean=0.0, std=0.02):
    return torch.randn(*shape, generator=g, device="cuda").mul_(std).add_(mean)


def _host(t):
    """A device tensor's bytes in host memory, as a loader hands them over."""
    out = torch.empty(t.numel() * t.element_size(), dtype=torch.uint8, pin_memory=True)
    out.copy_(t.contiguous().view(-1).view(torch.uint8))
    return out.numpy()


def _gguf(g, kind, rows, cols):
    """A (rows, cols) matrix ~N(0, 0.02) as the bytes of a GGUF tensor, on the device."""
    x = _normal(g, rows, cols)
    if kind == "f32":
        return x
    if kind == "f16":
        return x.half()
    b = x.view(-1, 32)
    if kind == "q8_0":
        d = (b.abs().amax(1, keepdim=True) / 127.0).half()
        q = (b / d.float().clamp_min(1e-12)).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        top = b.gather(1, b.abs().argmax(1, keepdim=True))
        d = (top / -8.0).half()
        u = (b / torch.where(d == 0, torch.ones_like(d), d).float() + 8.5).floor_().clamp_(0, 15).to(torch.uint8)
        q = u[:, :16] | (u[:, 16:] << 4)
    return torch.cat([d.view(torch.uint8), q], 1)


def _state_dict(c, kind, g):
    """The tensors of a model file.  Up to four layers are drawn, larger models repeat them."""
    d, f, v, nl = c["dim"], c["ffn"], c["vocab"], c["n_layers"]
    sd = {}

    def mat(key, rows, cols, k=kind):
        sd[key] = llm.Tensor(k, _host(_gguf(g, k, rows, cols)), rows, cols)

    def vec(key, n, mean=0.0):
        sd[key] = llm.Tensor("f32", _host(_normal(g, n, mean=mean)), 1, n)

    if c["arch"] == "gpt2":
        mat("wte.weight", v, d, "f16")
        mat("wpe.weight", c["max_seq"], d, "f16")
        vec("ln_f.affine", d, 1.0)
        vec("ln_f.bias", d)
        mat("lm_head.weight", v, d)
    else:
        mat("tok_embeddings.weight", v, d, "f16")
        vec("norm.weight", d, 1.0)
        mat("output.weight", v, d)
    kd = d // c["n_heads"] * c.get("n_kv_heads", c["n_heads"])
    prefix, drawn = ("h" if c["arch"] == "gpt2" else "layers"), min(nl, 4)
    for l in range(drawn):
        p = f"{prefix}.{l}."
        if c["arch"] == "gpt2":
            for ln in ("ln_1", "ln_2"):
                vec(p + ln + ".affine", d, 1.0)
                vec(p + ln + ".bias", d)
            for key, rows, cols in (("attn.c_attn", 3 * d, d), ("attn.c_proj", d, d), ("mlp.c_fc", f, d), ("mlp.c_proj", d, f)):
                mat(p + key + ".weight", rows, cols)
                vec(p + key + ".bias", rows)
        else:
            vec(p + "attention_norm.weight", d, 1.0)
            vec(p + "ffn_norm.weight", d, 1.0)
            for key, rows, cols in (("attention.wq", d, d), ("attention.wk", kd, d), ("attention.wv", kd, d), ("attention.wo", d, d),
                                    ("feed_forward.w1", f, d), ("feed_forward.w2", d, f), ("feed_forward.w3", f, d)):
                mat(p + key + ".weight", rows, cols)
    for key in [k for k in sd if k.startswith(prefix + ".")]:
        _, l, rest = key.split(".", 2)
        for other in range(int(l) + drawn, nl, drawn):
            sd[f"{prefix}.{other}.{rest}"] = sd[key]
    return sd


class _View:
    """Device memory of the library as an array that torch can wrap."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 3, "strides": None}


def _cache_rows(session, kv, first, count):
    """The rows that a pass leaves in the last layer's cache, in place: fp32 rows, or the quants of Q8_0 rows.  (Pages
    have no address of their own to look at; what they hold shows in the logits.)"""
    rows = []
    for which in "kv" if kv < 2 else "":
        p, n = C.c_void_p(), C.c_int64()
        name = f"{which}_cache{'_q8' if kv else ''}.{session.cfg['n_layers'] - 1}"
        _lib.check(session.lib.cthip_decoder_peek(session.handle, name.encode(), C.byref(p), C.byref(n)))
        shape = (session.cfg["max_seq"], n.value * (4 if kv else 1) // session.cfg["max_seq"])
        rows.append(torch.as_tensor(_View(p.value, shape, "|i1" if kv else "<f4"), device="cuda")[first:first + count])
    return rows


def _session(case, seed):
    c, g = MODELS[case["model"]], torch.Generator("cuda").manual_seed(seed)
    lib = _lib.init()
    sd = _state_dict(c, case["kind"], g)
    _lib.check(lib.cthip_set_option(b"kv_cache", case["kv"]))
    try:
        session = (llm.make_gpt2 if c["arch"] == "gpt2" else llm.make_llama)(c, sd)
        pos = case["pos"]
        ids = [float(t) for t in synth.prompt(c["vocab"], pos + case.get("rows", 1), seed=seed)]
        session.forward(ids[:max(pos, 1)], max(pos, 1), 0)  # the conversation so far
    finally:
        _lib.check(lib.cthip_set_option(b"kv_cache", 0))
    return session, ids[pos:]


def prepare(case, seed):
    lib = _lib.init()
    family = case["family"]
    if family in ("decode", "prompt"):
        session, ids = _session(case, seed)
        return dict(family=family, session=session, ids=ids, pos=case["pos"], steps=case.get("steps", 0),
                    cache=_cache_rows(session, case["kv"], case["pos"], case.get("rows") or case["steps"]))
    if family == "graph":
        c, g = MODELS[case["model"]], torch.Generator("cuda").manual_seed(seed)
        d, f, v, nl = c["dim"], c["ffn"], c["vocab"], c["n_layers"]

        def n(*shape, mean=0.0):
            return _normal(g, *shape, mean=mean).cpu().numpy()

        w = dict(wte=n(v, d), wpe=n(c["max_seq"], d), lnf_g=n(d, mean=1.0), lnf_b=n(d), lm_head=n(v, d))
        for key, shape, mean in (("ln1_g", (d,), 1.0), ("ln1_b", (d,), 0.0), ("attn_w", (3 * d, d), 0.0), ("attn_b", (3 * d,), 0.0),
                                 ("proj_w", (d, d), 0.0), ("proj_b", (d,), 0.0), ("ln2_g", (d,), 1.0), ("ln2_b", (d,), 0.0),
                                 ("fc_w", (f, d), 0.0), ("fc_b", (f,), 0.0), ("fc2_w", (d, f), 0.0), ("fc2_b", (d,), 0.0)):
            w[key] = [n(*shape, mean=mean) for _ in range(nl)]
        graph = graphs.GPT2Graph(c, w)
        return dict(family=family, graph=graph, prompt=synth.prompt(v, case["rows"], seed=seed), steps=case["steps"])
    g = torch.Generator("cuda").manual_seed(seed)
    if family == "mlp":
        d, f, m, llama = case["dim"], case["ffn"], case["rows"], case["arch"] == "llama"
        up = ops.WeightMatrix(case["kind"], _host(_gguf(g, case["kind"], (2 if llama else 1) * f, d)), (2 if llama else 1) * f, d)
        down = ops.WeightMatrix(case["kind"], _host(_gguf(g, case["kind"], d, f)), d, f)
        return dict(family=family, lib=lib, llama=llama, rows=m, up=up, down=down, x=_normal(g, m, d, std=1.0),
                    gamma=_normal(g, d, mean=1.0), beta=_normal(g, d), up_b=_normal(g, f), down_b=_normal(g, d),
                    h=torch.empty(m, up.rows, device="cuda"), y=torch.empty(m, d, device="cuda"))
    if family == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        a, b = (torch.rand(*sh, generator=g, device="cuda").mul_(2).sub_(1) for sh in ((m, k), (k, n)))
        return dict(family=family, lib=lib, a=a, b=b, c=torch.empty(m, n, device="cuda"), m=m, n=n, k=k,
                    act=_lib.ACT_RELU if case["relu"] else _lib.ACT_NONE, precision=PRECISIONS[case["precision"]])
    rows, n = case["rows"], case["n"]
    return dict(family=family, lib=lib, op=case["op"], rows=rows, n=n, x=_normal(g, rows, n, std=1.0), y=torch.empty(rows, n, device="cuda"),
                z=torch.empty(rows, n, device="cuda") if case["op"] in ("ln_gelu", "rms_silu") else torch.empty(rows, dtype=torch.int64, device="cuda"),
                gamma=_normal(g, n, mean=1.0), beta=_normal(g, n))


# ---------------------------------------------------------------------------------------------------------------------
# one pass


def run(s):
    family, check = s["family"], _lib.check
    if family == "decode":
        # the token in hand goes in, its successors come out
        token, logits = s["session"].forward(s["ids"][:1], 1, s["pos"], return_logits=True)
        return [logits, [token] + s["session"].generate_on_device(s["steps"] - 1), s["cache"]]
    if family == "prompt":
        token, logits = s["session"].forward(s["ids"], len(s["ids"]), s["pos"], return_logits=True)
        return [logits, token, s["cache"]]
    if family == "graph":
        return s["graph"].generate(s["prompt"], s["steps"])
    lib = s["lib"]
    if family == "mlp":
        x, h, y, m = s["x"].data_ptr(), s["h"].data_ptr(), s["y"].data_ptr(), s["rows"]
        gamma, beta = s["gamma"].data_ptr(), s["beta"].data_ptr()
        if s["llama"]:
            check(lib.cthip_linear(h, s["up"].handle, x, m, None, None, _lib.ACT_NONE, _lib.PRO_RMSNORM, gamma, None, EPS))
            check(lib.cthip_linear(y, s["down"].handle, h, m, None, x, _lib.ACT_NONE, _lib.PRO_SWIGLU, None, None, EPS))
        else:
            check(lib.cthip_linear(h, s["up"].handle, x, m, s["up_b"].data_ptr(), None, _lib.ACT_GELU, _lib.PRO_LAYERNORM, gamma, beta, EPS))
            check(lib.cthip_linear(y, s["down"].handle, h, m, s["down_b"].data_ptr(), x, _lib.ACT_NONE, _lib.PRO_NONE, None, None, EPS))
        return [s["h"], s["y"]]
    if family == "matmul":
        check(lib.cthip_matmul(s["c"].data_ptr(), s["a"].data_ptr(), s["b"].data_ptr(), s["m"], s["n"], s["k"], s["act"], s["precision"]))
        return s["c"]
    op, x, y, z, rows, n = s["op"], s["x"].data_ptr(), s["y"].data_ptr(), s["z"].data_ptr(), s["rows"], s["n"]
    if op == "ln_softmax":
        check(lib.cthip_layernorm_softmax(y, x, s["gamma"].data_ptr(), s["beta"].data_ptr(), EPS, rows, n))
        return s["y"]
    if op == "sample":
        check(lib.cthip_softmax(y, x, rows, n))
        check(lib.cthip_argmax(z, x, rows, n))
    elif op == "ln_gelu":
        check(lib.cthip_layernorm(y, x, s["gamma"].data_ptr(), s["beta"].data_ptr(), EPS, rows, n))
        check(lib.cthip_unary(UNARY["gelu"], z, y, rows * n))
    else:
        check(lib.cthip_rmsnorm(y, x, s["gamma"].data_ptr(), EPS, rows, n))
        check(lib.cthip_unary(UNARY["silu"], z, y, rows * n))
    return [s["y"], s["z"]]


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    family = case["family"]
    if family in ("decode", "prompt", "graph"):
        c = MODELS[case["model"]]
        d, nl = c["dim"], c["n_layers"]
        kd = d // c["n_heads"] * c.get("n_kv_heads", c["n_heads"])
        per, head = _linears(c)
        weight = BYTES[case.get("kind", "f32")]
        row = 2 * nl * kd * (BYTES["q8_0"] if case.get("kv") == 1 else 4.0)  # cache bytes of one position, all layers
        # (rows that go in together, position of the first, position behind the last): a weight is read once for each
        parts = [(case["rows"], case.get("pos", 0))] if family != "decode" else []
        first = case["pos"] if family == "decode" else case["rows"]
        if family != "prompt":
            parts += [(1, first + i) for i in range(case["steps"] - (1 if family == "graph" else 0))]
        nbytes = flops = 0.0
        for s, pos in parts:
            nbytes += weight * (nl * per + head) + row * (pos + s) + 4.0 * d * s
            keys = s * pos + s * (s + 1) / 2
            flops += 2.0 * (s * nl * per + head) + 4.0 * nl * d * keys
        return {"bytes": nbytes, "flops": flops}
    if family == "mlp":
        d, f, m = case["dim"], case["ffn"], case["rows"]
        wide = 2 * f if case["arch"] == "llama" else f
        return {"bytes": BYTES[case["kind"]] * (d * wide + f * d) + 4.0 * m * (2 * d + wide), "flops": 2.0 * m * (d * wide + f * d)}
    if family == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    rows, n = case["rows"], case["n"]
    if case["op"] == "ln_softmax":
        return {"bytes": 8.0 * rows * n, "flops": 12.0 * rows * n}
    if case["op"] == "sample":
        return {"bytes": 8.0 * rows * n + 8.0 * rows, "flops": 5.0 * rows * n}
    return {"bytes": 12.0 * rows * n, "flops": 20.0 * rows * n}


def tolerance(case):
    family = case["family"]
    if family == "graph":  # greedy tokens: alike but where two logits tie, and a tie changes the tokens after it
        return {"differ": 0.5}
    if family in ("decode", "prompt"):
        # two bf16 terms per operand (2^-16 of a product dropped) through all layers of a prompt, fp32 behind it; over
        # Q8_0 cache rows a value that rounds the other way moves by a step of its block (and its quant by one)
        return {"rel": 1e-2 if case["kv"] == 1 else 1e-4, "max": 0.05 if case["kv"] == 1 else 5e-4, "differ": 0.5}
    if family == "mlp":  # fp32 for a few rows, two bf16 terms per operand for more
        return {"rel": 5e-5, "max": 1e-3}
    if family == "matmul":
        return {"fp32": {"rel": 1e-5}, "bf16x6": {"rel": 1e-5}, "bf16x3": {"rel": 5e-5}, "bf16": {"rel": 1e-2}}[case["precision"]]
    return {"rel": 1e-5, "differ": 0.0}
