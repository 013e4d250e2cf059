"""Heads of models without a query latent, and V3's (kernels_head.hip, option "head_short"), against head_attn_kernel: the same values and sums in the same order, so
logits, cache rows and the attention output have to be the same bits."""
import numpy as np
import pytest

from tools import synth

pytestmark = pytest.mark.gpu


def cache_rows(c, n, seed):
    rng = np.random.default_rng(seed)
    H, hd = c.n_heads, c.qk_nope_head_dim + c.qk_rope_head_dim
    f16 = lambda *s: (0.5 * rng.standard_normal(s)).astype(np.float32).astype(np.float16).view(np.uint16)
    return {"k_cache": f16(n, H * hd), "v_cache": f16(n, H * c.v_head_dim)}


def same(ctx, c, positions, T=None, seed=3, short=True, in_wo=None, **options):
    import dsk
    A, B = (dsk.Model(ctx, c, T, synth_seed=None if T is not None else seed, options=dict(options, head_short=on)) for on in (1, 0))
    assert [m.info("head_short_layers") for m in (A, B)] == [c.n_layers if short else 0, 0]
    if in_wo is None:  # (without a query latent: all of these have up to 16 blocks of output)
        in_wo = int(c.quant in ("q2_k", "q3_k") and not c.q_lora_rank)
    assert [m.info("att_q8_in_wo") for m in (A, B)] == [in_wo, options.get("att_q8_in_wo", 0) if c.quant in ("q2_k", "q3_k") else 0]
    n = min(c.max_seq_len, c.rs_original_max_position_embeddings)
    for l in range(c.n_layers):
        for name, rows in cache_rows(c, n, 10 + l).items():
            A.set_cache_rows(l, name, 0, rows)
            B.set_cache_rows(l, name, 0, rows)
    width = {"k_cache": c.n_heads * (c.qk_nope_head_dim + c.qk_rope_head_dim), "v_cache": c.n_heads * c.v_head_dim}
    for i, pos in enumerate(positions):
        tok = (7 * pos + 3) % c.vocab_size
        la, lb = A.forward(tok, pos), B.forward(tok, pos)
        assert np.all(np.isfinite(lb)) and np.array_equal(la, lb), pos
        for l in range(c.n_layers):
            for name, w in width.items():
                assert np.array_equal(A.get_cache_rows(l, name, 0, n, w), B.get_cache_rows(l, name, 0, n, w)), (pos, l, name)
    x = np.random.default_rng(1).standard_normal(c.dim).astype(np.float32)
    pos = positions[0]
    assert np.array_equal(A.run_block(0, x, pos), B.run_block(0, x, pos))
    assert np.array_equal(A.stage("att_out", c.n_heads * c.v_head_dim), B.stage("att_out", c.n_heads * c.v_head_dim))
    if c.quant in ("q2_k", "q3_k"):
        for point, count in (("kv_a", c.kv_lora_rank), ("att", c.n_heads * c.v_head_dim)) + ((("q_a", c.q_lora_rank),) if c.q_lora_rank else ()):
            for a, b in zip(A.stage_q8(point, count), B.stage_q8(point, count)):
                assert np.array_equal(a, b), point
    A.close()
    B.close()


QUANTS = ["q2_k", "q3_k", "f8e5m2", "fp16"]


@pytest.mark.parametrize("quant", QUANTS)
def test_v2lite_heads_over_the_edges_of_positions(ctx, quant):
    """one position; the wave's 16, the softmax's 64, the early values' 64 / 128 / 256, the keys' 256, beyond; the split form from 1024 on"""
    c = synth.preset("v2lite", quant, False, n_layers=2, hidden_dim=512, vocab_size=512, n_routed_experts=0, max_seq_len=1100)
    same(ctx, c, [0, 1, 15, 16, 62, 63, 64, 127, 128, 200, 255, 256, 300, 511, 700, 1022, 1023, 1024])


@pytest.mark.parametrize("quant", QUANTS)
@pytest.mark.parametrize("over", [dict(), dict(n_heads=3, v_head_dim=128, qk_nope_head_dim=64, qk_rope_head_dim=64, kv_lora_rank=512, n_shared_experts=0),
                                  dict(n_heads=2, v_head_dim=128, qk_nope_head_dim=32, qk_rope_head_dim=16, kv_lora_rank=256)],
                         ids=["tiny", "3 heads", "small heads"])
def test_small_heads(ctx, quant, over):
    if quant in ("q2_k", "q3_k") and over.get("n_heads") == 3:
        over = dict(over, n_heads=4)
    c = synth.preset("tiny_v2lite", quant, False, **over)
    same(ctx, c, [0, 3, 40, 63], T=synth.synth_model(c, seed=5))


@pytest.mark.parametrize("quant", QUANTS)
def test_ring_and_sinks(ctx, quant):
    """past the ring: the current position is in the middle of the rows, and the sink keys turn by one position each token"""
    c = synth.preset("v2lite", quant, False, n_layers=2, hidden_dim=512, vocab_size=512, n_routed_experts=0, max_seq_len=96, rs_original_max_position_embeddings=80)
    same(ctx, c, [79, 80, 81, 130, 200])


@pytest.mark.parametrize("arch", ["DeepseekV3ForCausalLM", "DeepseekV2ForCausalLM"])  # (rope's pairs in place, or apart)
def test_heads_behind_a_query_latent(ctx, arch):
    c = synth.preset("v3", "q2_k", False, arch=arch, dim=512, hidden_dim=512, vocab_size=512, n_layers=2, n_routed_experts=0, n_shared_experts=0, max_seq_len=1100)
    same(ctx, c, [0, 1, 15, 16, 62, 63, 64, 127, 128, 200, 255, 256, 300, 511, 700, 1022, 1023, 1024])


def test_heads_behind_a_query_latent_past_the_ring(ctx):
    c = synth.preset("v3", "q2_k", False, dim=512, hidden_dim=512, vocab_size=512, n_layers=2, n_routed_experts=0, n_shared_experts=0, max_seq_len=96,
                     rs_original_max_position_embeddings=80)
    same(ctx, c, [79, 80, 81, 130, 200])


@pytest.mark.parametrize("quant", ["fp16", "q2_k", "q3_k"])
@pytest.mark.parametrize("over", [dict(qk_nope_head_dim=192, qk_rope_head_dim=64), dict(q_lora_rank=256)], ids=["heads of 256", "query latent"])
def test_heads_of_other_forms_keep_the_general_kernel(ctx, quant, over):
    c = synth.preset("tiny_v2lite", quant, False, **over)
    same(ctx, c, [0, 3, 40], T=synth.synth_model(c, seed=5), short=False)


@pytest.mark.parametrize("quant", ["q2_k", "q3_k"])
def test_who_quantises_the_output(ctx, quant):
    """the caller's word holds: never in wo, which heads that leave 32 bits then do not come in front of; always; by size, which 17 blocks are too large for"""
    c = synth.preset("tiny_v2lite", quant, False)
    T = synth.synth_model(c, seed=5)
    same(ctx, c, [0, 3, 40], T=T, short=False, in_wo=0, att_q8_in_wo=0)
    same(ctx, c, [0, 3, 40], T=T, in_wo=1, att_q8_in_wo=1)
    c = synth.preset("tiny_v2lite", quant, False, n_heads=34, v_head_dim=128)
    same(ctx, c, [0, 3, 40], T=synth.synth_model(c, seed=5), short=False, in_wo=0)
