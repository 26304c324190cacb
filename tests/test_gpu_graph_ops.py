"""Operations of a graph forward that share launches (csrc/graph_ops.hip) leave every buffer as one launch each does: the walk
in the library (which shares) against the walk on the host (which does not), prompts of one, two and more rows, contexts
on both sides of the 64 keys a workgroup asks for at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,lengths", [("gpt2-tiny", (1, 1, 1)), ("gpt2-tiny", (2, 1, 3, 1)), ("gpt2-mini", (17, 1, 2)), ("gpt2-mini", (62, 1, 1, 1, 2)),
                                          ("gpt2-mini", (100, 1))])
def test_shared_launches_leave_the_same_buffers(name, lengths):
    from caten_amd import graphs, synth
    from caten_amd.buffer import transfer_into_array
    cfg = synth.GPT2_CONFIGS[name]
    w = synth.gpt2_weights(cfg, seed=1)
    ids = synth.prompt(cfg["vocab"], sum(lengths), seed=1)
    models = [graphs.GPT2Graph(cfg, w, native=native) for native in (True, False)]
    names = ["h0", "mask", "lnf", "logits", "out"] + [f"l{l}_{b}" for l in range(cfg["n_layers"])
                                                     for b in ("ln1", "qkv", "kc", "vc", "sc", "pr", "ao", "am", "h1", "ln2", "fc", "h2")]
    try:
        n = 0
        for s in lengths:
            for m in models:
                m.forward(ids[n:n + s], n)
            for b in names:
                got, want = (np.asarray(transfer_into_array(m.vm.getvar(b)), np.float64) for m in models)
                seen = np.isfinite(want)  # (a masked score is -inf in both)
                assert got.shape == want.shape and np.array_equal(seen, np.isfinite(got)), (b, n)
                err, ref = np.linalg.norm(got[seen] - want[seen]), np.linalg.norm(want[seen])
                assert err <= 2e-5 * ref + 1e-12, (b, n, err, ref)
            n += s
    finally:
        for m in models:
            m.close()


def test_a_failing_node_leaves_what_ran_before_it(oracle):
    """The walk stops at a node whose argument was never set; the operations in front of it, queued to share launches, have run."""
    import ctypes as C
    from caten_amd import _lib, blueprints, ops
    from caten_amd.renderer import item_sexp
    lib = _lib.init(0)
    x = np.random.default_rng(0).normal(0, 1, (5, 77)).astype(np.float32)
    dx, dy, dz = ops.DeviceArray.from_numpy(x), ops.DeviceArray((5, 77)), ops.DeviceArray((5, 77))
    program, vm = C.c_void_p(), C.c_void_p()
    _lib.check(lib.cthip_program_create(C.byref(program), item_sexp(blueprints.softmax_rows()).encode()))
    _lib.check(lib.cthip_vm_create(C.byref(vm), 5))
    dtypes, none, one = (C.c_int * 4)(0, 5, 5, 0), (C.c_double * 4)(), (C.c_int * 1)(0)
    for out, src in ((2, 0), (3, 2), (3, 4)):  # softmax of x, of that, and of a buffer nobody sets
        reads = (C.c_longlong * 4)(out, 5, 77, src)
        _lib.check(lib.cthip_vm_add_kernel(vm, program, 4, (C.c_int * 4)(2, 0, 0, 2), reads, none, dtypes, 1, one, (C.c_int * 1)(out)))
    for slot, d in ((0, dx), (2, dy), (3, dz)):
        _lib.check(lib.cthip_vm_set_buffer(vm, slot, d.ptr))
    assert lib.cthip_vm_run(vm) == _lib.E_STATE and b"vm: node 2" in lib.cthip_last_error()
    want = oracle.softmax(x)
    assert np.allclose(dy.numpy(), want, rtol=1e-5, atol=1e-6)
    assert np.allclose(dz.numpy(), oracle.softmax(want), rtol=1e-5, atol=1e-6)
    _lib.check(lib.cthip_vm_destroy(vm))
    _lib.check(lib.cthip_program_destroy(program))


@pytest.mark.parametrize("batches,h,s,t,dh", [((3,), 2, 5, 9, 64), ((3, 2), 5, 4, 70, 64), ((1, 7), 3, 2, 33, 128), ((5, 1), 2, 3, 65, 32)])
def test_attention_over_batches_and_heads(batches, h, s, t, dh):
    """Copies of the last batch's new key and value rows, scores, softmax, values and the copy that puts the heads side by side, as one launch over every batch axis: each buffer
    against 64 bits.  Sums of at most `t` or `dh` products of fp32 numbers; exp2's argument, scores below 16 in magnitude, is off by their own error."""
    import ctypes as C
    from caten_amd import _lib, blueprints as bp, ops
    from caten_amd.renderer import item_sexp
    lib = _lib.init(0)
    nb, rng, row = int(np.prod(batches)), np.random.default_rng(h * t), h * dh
    print(f"case: batches {batches}, {h} heads, {s} rows, {t} keys of {dh}", flush=True)
    add, mul, A = bp._add, bp._mul, bp._A

    def index(*terms):  # (stride, axis) pairs and constants
        e = 0
        for x in terms:
            x = mul(*x) if isinstance(x, tuple) else x
            e = x if e == 0 else add(e, x)
        return e

    def nest(name, ext, red, out, body):
        g = [f"_gid{q}" for q in range(len(ext))]
        head = [bp._for(x, e) for x, e in zip(g, ext)]
        mid = [bp._decl("acc", 0.0), bp._for("_gid9", red), bp._red("acc", add("acc", body(g, "_gid9"))), bp._end("_gid9")] if red else []
        return {"name": name, "blueprint": [bp._glob("val_o", "output", 1)] + [bp._glob(f"val_{x}", "input", 1) for x in ("a", "b")[:2 if red else 1]] + head + mid +
                [bp._store("val_o", out(g), mul("acc", 0.125) if name == "it_scores" else "acc" if red else body(g, None))] + [bp._end(x) for x in reversed(g)]}

    nax = len(batches)
    strides = [int(np.prod(batches[q + 1:])) for q in range(nax)]
    bt = lambda g, k: [(k * strides[q], g[q]) for q in range(nax)]  # noqa: E731
    copy = nest("it_copy", (row,), None, lambda g: g[0], lambda g, _: A("val_a", g[0]))
    scores = nest("it_scores", (*batches, h, s, t), dh, lambda g: index(*bt(g, h * s * t), (s * t, g[nax]), (t, g[nax + 1]), g[nax + 2]),
                  lambda g, k: mul(A("val_a", index(*bt(g, s * row), (dh, g[nax]), (row, g[nax + 1]), k)), A("val_b", index(*bt(g, t * row), (dh, g[nax]), (row, g[nax + 2]), k))))
    values = nest("it_values", (*batches, h, s, dh), t, lambda g: index(*bt(g, s * row), (s * dh, g[nax]), (dh, g[nax + 1]), g[nax + 2]),
                  lambda g, k: mul(A("val_a", index(*bt(g, h * s * t), (s * t, g[nax]), (t, g[nax + 1]), k)), A("val_b", index(*bt(g, t * row), (dh, g[nax]), (row, k), g[nax + 2]))))
    softmax = bp.softmax_rows(rows=nb * h * s, n=t)
    q, k, v, nk, nv = (rng.normal(0, 1, shape).astype(np.float32) for shape in ((nb, s, h, dh), (nb, t, h, dh), (nb, t, h, dh), (row,), (row,)))
    d = {n: ops.DeviceArray.from_numpy(x) for n, x in dict(q=q, k=k, v=v, nk=nk, nv=nv).items()}
    d.update(sc=ops.DeviceArray((nb, h, s, t)), pr=ops.DeviceArray((nb, h, s, t)), o=ops.DeviceArray((nb, h, s, dh)))
    slots = list(d) + ["k_new", "v_new"]
    vm, programs = C.c_void_p(), []
    _lib.check(lib.cthip_vm_create(C.byref(vm), len(slots)))
    try:
        for item, args in ((copy, ("k_new", "nk")), (copy, ("v_new", "nv")), (scores, ("sc", "q", "k")), (softmax, ("pr", "sc")), (values, ("o", "pr", "v"))):
            program, n = C.c_void_p(), len(args)
            _lib.check(lib.cthip_program_create(C.byref(program), item_sexp(item).encode()))
            programs.append(program)
            at = [slots.index(x) for x in args]
            _lib.check(lib.cthip_vm_add_kernel(vm, program, n, (C.c_int * n)(*[2] * n), (C.c_longlong * n)(*at), (C.c_double * n)(), (C.c_int * n)(), 1, (C.c_int * 1)(0), (C.c_int * 1)(at[0])))
        new = (nb * t - 1) * row * 4  # the last row of the last batch
        for slot, x in enumerate(slots):
            _lib.check(lib.cthip_vm_set_buffer(vm, slot, d[x].ptr if x in d else d[x[0]].ptr + new))
        for _ in range(2):
            _lib.check(lib.cthip_vm_run(vm))
        got = {x: d[x].numpy().astype(np.float64) for x in ("k", "v", "sc", "pr", "o")}
    finally:
        _lib.check(lib.cthip_vm_destroy(vm))
        for program in programs:
            _lib.check(lib.cthip_program_destroy(program))
    k.reshape(-1)[-row:], v.reshape(-1)[-row:] = nk, nv
    assert np.array_equal(got["k"], k) and np.array_equal(got["v"], v)
    q, k, v = (x.astype(np.float64).transpose(0, 2, 1, 3) for x in (q, k, v))
    want, eps = q @ k.transpose(0, 1, 3, 2) * 0.125, 2.0 ** -24
    assert np.all(np.abs(got["sc"] - want) <= dh * eps * (np.abs(q) @ np.abs(k).transpose(0, 1, 3, 2)))
    assert np.abs(want).max() < 16
    e = np.exp(got["sc"] - got["sc"].max(-1, keepdims=True))
    pr = e / e.sum(-1, keepdims=True)
    assert np.all(np.abs(got["pr"] - pr) <= (t + 64) * eps * pr)  # (16 log2(e) 2^-24 in the argument, twice, and the sum's)
    assert np.all(np.abs(got["o"] - got["pr"] @ v) <= t * eps * (got["pr"] @ np.abs(v)))
