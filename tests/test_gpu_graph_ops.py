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
