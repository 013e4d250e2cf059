"""The experts' launches of latency-bound models (kernels_experts.hip, option "expert_launches") against the generic launches, with both halves of float models
against the one launch: the same arithmetic per row in the same order, so logits, routing, slot outputs and the residual stream have to be the same bits."""
import numpy as np
import pytest

from tools import synth

pytestmark = pytest.mark.gpu


def same(ctx, c, T=None, seed=None, tokens=(5, 9, 700, 3, 44), options=None, up=False):
    import dsk
    # floats: the other side is the one launch (the generic launches stage x with as many waves as their rows ask for, and with four the sum of squares
    # can differ in its last bit)
    floats = c.quant in ("f8e5m2", "fp16") and up
    o = dict({"fuse_moe": int(floats), "q2k_tiles": 0}, **(options or {}))
    A, B = (dsk.Model(ctx, c, T, synth_seed=seed, options=dict(o, expert_launches=on)) for on in (1, 0))
    blocks = c.n_layers - c.first_k_dense_replace
    assert [m.info("expert_down_layers") for m in (A, B)] == [blocks, 0]
    assert [m.info("expert_up_layers") for m in (A, B)] == [blocks if up else 0, 0]
    assert [m.info("fused_moe_layers") for m in (A, B)] == [0, blocks if floats else 0]
    for graph in (True, False):
        for m in (A, B):
            m.set_graph(graph)
        for pos, tok in enumerate(tokens):
            la, lb = A.forward(tok, pos), B.forward(tok, pos)
            assert np.all(np.isfinite(lb)) and np.array_equal(la, lb), (graph, pos)
            for a, b in zip(A.routing(), B.routing()):
                assert np.array_equal(a, b), (graph, pos)
            assert np.array_equal(A.slot_outputs(), B.slot_outputs()), (graph, pos)
    x = np.random.default_rng(1).standard_normal(c.dim).astype(np.float32)
    layer = c.first_k_dense_replace
    assert np.array_equal(A.run_block(layer, x, 2), B.run_block(layer, x, 2))
    n = (c.n_active_routed + (c.n_shared_experts > 0)) * max(1, c.n_shared_experts) * c.moe_intermediate_size if c.quant in ("q2_k", "q3_k") else 0
    for name, count, dt in (("q8.hb.qs", n, np.int8), ("q8.hb.d", n // 256, np.float32)) if n else ():  # what the slots staged
        assert np.array_equal(A.stage(name, count, dt).view(np.uint8), B.stage(name, count, dt).view(np.uint8)), name
    A.close()
    B.close()


# rows of x per workgroup 1 (a part of the workgroups' rows missing) and 2; hidden vectors of 1 - 3 blocks; K = 1; without a shared expert
SMALL = [dict(), dict(dim=768, moe_intermediate_size=512), dict(n_shared_experts=0, moe_intermediate_size=768), dict(n_active_routed=1, n_shared_experts=1),
         dict(n_active_routed=8, dim=256)]


QUANTS = ["q2_k", "q3_k", "f8e5m2", "fp16"]


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("over", SMALL, ids=[",".join(f"{k[:8]}{v}" for k, v in o.items()) or "tiny" for o in SMALL])
def test_small_shapes_same_bits(ctx, quant, over):
    c = synth.preset("tiny_v2lite", quant, False, **over)
    same(ctx, c, synth.synth_model(c, seed=7))


@pytest.mark.parametrize("quant", QUANTS)
def test_v2lite_shapes_same_bits(ctx, quant):
    c = synth.preset("v2lite", quant, False, n_layers=3, max_seq_len=64)
    same(ctx, c, seed=5, tokens=(5, 90000, 3), up=True)


# the gate by one wave: an odd number of experts, all 64, as many as are chosen; sigmoid with a bias and normed weights; 32 and 64 lanes a row, two router
# pieces a slice; rows that no workgroup count divides; no shared expert
GATE = [dict(n_routed_experts=33, n_active_routed=5), dict(n_routed_experts=64, n_active_routed=8, n_shared_experts=0, moe_intermediate_size=768),
        dict(n_routed_experts=3, n_active_routed=3), dict(dim=4096, n_routed_experts=16, scoring_func="sigmoid", has_moegate_bias=True, norm_topk_prob=True,
                                                          routed_scaling_factor=2.5)]


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("over", GATE, ids=["33 of 5", "64 of 8", "3 of 3", "sigmoid 4096"])
def test_gate_inside_the_first_half_same_bits(ctx, quant, over):
    over = dict(over)
    if quant in ("f8e5m2", "fp16") and over.get("dim") == 4096:
        over["dim"] = 2048  # (floats: rows of up to 32 values a lane)
    if over.pop("has_moegate_bias", False):
        over["arch"] = "DeepseekV3ForCausalLM"
    c = synth.preset("v2lite", quant, False, **dict(dict(n_layers=2, hidden_dim=512, vocab_size=512, moe_intermediate_size=256, max_seq_len=64), **over))
    same(ctx, c, seed=9, tokens=(5, 400, 3), up=True)


# more steps of a workgroup than its twelve waves have on their way at once (two each): 30 and 36 of two rows, 55 of one row
MANY = [dict(n_routed_experts=12, n_active_routed=10, moe_intermediate_size=1280), dict(n_routed_experts=12, n_active_routed=10),
        dict(dim=4096, n_routed_experts=9, n_active_routed=9, moe_intermediate_size=1280)]


@pytest.mark.parametrize("quant", ["q2_k", "q3_k"])
@pytest.mark.parametrize("over", MANY, ids=["30 steps", "36 steps", "55 steps"])
def test_more_steps_than_waves_request_same_bits(ctx, quant, over):
    c = synth.preset("v2lite", quant, False, **dict(dict(n_layers=2, hidden_dim=512, vocab_size=512, max_seq_len=64), **over))
    same(ctx, c, seed=21, tokens=(5, 400, 3), up=True)


def test_float_rows_of_fewer_steps_same_bits(ctx):
    """F8E5M2 and F16 over two MoE blocks whose hidden rows end inside a group of lanes and whose block scales change within a row"""
    for quant, over in (("f8e5m2", dict(moe_intermediate_size=176, n_shared_experts=2)), ("fp16", dict(moe_intermediate_size=104, n_shared_experts=1))):
        c = synth.preset("v2lite", quant, False, n_layers=3, hidden_dim=512, vocab_size=512, max_seq_len=64, n_routed_experts=9, n_active_routed=4, **over)
        same(ctx, c, seed=13, tokens=(5, 400, 3), up=True)


@pytest.mark.parametrize("quant", ["q2_k", "q3_k"])
def test_largest_values_of_both_signs_in_a_block(ctx, quant):
    """hidden values in pairs v, -v: a block's largest magnitude occurs with both signs, and the first one's sign decides the codes"""
    c = synth.preset("tiny_v2lite", quant, False)
    T = synth.synth_model(c, seed=11)
    at = (81, 83) if quant == "q2_k" else (109,)  # the high bytes of the block's float16 factors
    per = 84 if quant == "q2_k" else 110
    for name, t in T.items():
        if ".mlp.w1." in name or "shared_mlp.w1." in name:
            t.data[..., 1::2, :] = t.data[..., 0::2, :]
        if ".mlp.w3." in name or "shared_mlp.w3." in name:
            d = t.data[..., 0::2, :].copy().reshape(-1, per)
            for b in at:
                d[:, b] ^= 0x80
            t.data[..., 1::2, :] = d.reshape(t.data[..., 0::2, :].shape)
    same(ctx, c, T)
