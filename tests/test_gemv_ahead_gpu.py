"""Small plain launches that request their weights ahead of the staging of their vector (kernels_gemv.hip gemv_ahead_kernel, gemv_ahead_f_kernel, option
"gemv_ahead") against the plain kernel: another order of the same loads, so every logit and cache row has to be the same bits."""
import numpy as np
import pytest

from tools import synth

pytestmark = pytest.mark.gpu


# V2-Lite's own shapes; rows of one and of four column steps, shares that do not divide by the workgroups, blocks of scales that end inside a row and a
# column step; wo's rows another number of steps than x's
SHAPES = [("q2_k", {}), ("q3_k", {}), ("f8e5m2", {}), ("fp16", {}), ("f8e5m2", dict(dim=1024, n_heads=17, v_head_dim=64)), ("f8e5m2", dict(dim=4096, n_heads=16, block_size=(48, 80))),
          ("fp16", dict(dim=1024, n_heads=16)), ("fp16", dict(dim=512, n_heads=16, v_head_dim=64)), ("q3_k", dict(n_heads=18))]


@pytest.mark.parametrize("quant,over", SHAPES, ids=[q + "".join(f"-{k[:5]}{v}".replace(" ", "") for k, v in o.items()) for q, o in SHAPES])
def test_weights_ahead_same_bits(ctx, quant, over):
    import dsk
    o = dict(dict(n_layers=2, max_seq_len=64, hidden_dim=512, vocab_size=512), **over)
    block = o.pop("block_size", None)
    c = synth.preset("v2lite", quant, False, **o)
    if block:
        c.block_size = block
    A, B = (dsk.Model(ctx, c, None, synth_seed=29, options={"gemv_ahead": on}) for on in (0, 3))
    assert A.info("gemv_ahead_plans") == 0
    # (a wo of rows that are no whole steps, or of more than one step in K-quants, or of Q3_K stays with the plain kernel)
    n = c.n_heads * c.v_head_dim
    step = {"f8e5m2": 1024, "fp16": 512}.get(quant)
    wo = n % step == 0 and n // step in (1, 2, 4) if step else n == 2048 and quant == "q2_k"
    assert B.info("gemv_ahead_plans") == c.n_layers * (2 if wo else 1)
    for graph in (True, False):
        for m in (A, B):
            m.set_graph(graph)
        for pos, t in enumerate((3, 500, 17, 4)):
            la, lb = A.forward(t, pos), B.forward(t, pos)
            assert np.all(np.isfinite(la)) and np.array_equal(la, lb), (graph, pos)
    for layer in range(c.n_layers):
        for name, width in (("k_cache", c.n_heads * (c.qk_nope_head_dim + c.qk_rope_head_dim)), ("v_cache", c.n_heads * c.v_head_dim)):
            assert np.array_equal(A.get_cache_rows(layer, name, 0, 4, width), B.get_cache_rows(layer, name, 0, 4, width))
    A.close()
    B.close()


# classifiers as a stream of row groups: shares that are no whole rounds nor row groups, rows of 16, 32 and 64 lanes (K-quants) and of 1, 2 and 4 steps (floats),
# scales' blocks of no power of two
STREAMS = [("q2_k", 2048, 102400), ("q2_k", 1024, 40001), ("q2_k", 4096, 9001), ("f8e5m2", 2048, 102400), ("f8e5m2", 1024, 8193), ("f8e5m2", 2048, 10007),
           ("fp16", 2048, 10007), ("fp16", 512, 33333), ("fp16", 1024, 8200)]


@pytest.mark.parametrize("quant,dim,vocab", STREAMS)
def test_classifier_stream_same_bits(ctx, quant, dim, vocab):
    import dsk
    c = synth.preset("v2lite", quant, False, n_layers=2, max_seq_len=64, hidden_dim=512, vocab_size=vocab, dim=dim, n_heads=8)
    if vocab == 10007 and quant == "f8e5m2":
        c.block_size = (48, 80)
    A, B = (dsk.Model(ctx, c, None, synth_seed=31, options={"gemv_ahead": on}) for on in (0, 3))
    assert [m.info("gemv_stream_plans") for m in (A, B)] == [0, 2]
    for pos, t in enumerate((3, 500, 17)):
        la, lb = A.forward(t, pos), B.forward(t, pos)
        assert np.all(np.isfinite(la)) and np.array_equal(la, lb), pos
    x = np.random.default_rng(1).standard_normal(c.dim).astype(np.float32)
    assert np.array_equal(A.run_head(x), B.run_head(x))
    A.close()
    B.close()
