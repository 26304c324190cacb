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
                err, ref = np.linalg.norm((got - want)[seen]), np.linalg.norm(want[seen])
                assert err <= 2e-5 * ref + 1e-12, (b, n, err, ref)
            n += s
    finally:
        for m in models:
            m.close()
