"""The batched prompt path's products at row lengths of an odd number of blocks and at both sides of its groups of 16 and 32 tokens: the per-token
loop's bits (option q2k_tiles = 2), like tests/test_hydrate_gpu.py."""
import numpy as np
import pytest

from tests.test_hydrate_gpu import _assert_identical, _caches, _loop, compare_hydrate
from tools import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import dsk
    c = dsk.Ctx(0)
    yield c
    c.close()


# blocks per row: model width 3 or 11, dense hidden vectors 11 or 13 (items of 4 blocks, a last one of 3 or 1), experts' 3, wo 1; experts
# 4 of 6: most tasks have more than 16 rows, their last pass from 1 to 32
@pytest.mark.parametrize("dim,hidden", [(768, 2816), (2816, 3328)])
@pytest.mark.parametrize("P", [12, 31, 32, 33, 49, 65])
def test_odd_rows_of_blocks(ctx, dim, hidden, P):
    c = synth.preset("tiny_v3", "q2_k", False, dim=dim, hidden_dim=hidden, moe_intermediate_size=768, n_routed_experts=6, n_group=2, topk_group=3,
                     vocab_size=512, max_seq_len=96)
    T = synth.synth_model(c, seed=83)
    tokens = np.random.default_rng(P).integers(0, c.vocab_size, P)
    _assert_identical(compare_hydrate(ctx, c, T, tokens=tokens, pos0=1), P, 1)


# attention of 16 tokens at a time (from 8 tokens on, DeepSeek-V3's head sizes): full and ragged tiles of tokens, contexts that end at both sides of
# 32 (a step of the values), 64 (a sum of the softmax) and of a tile of keys, a chunk that begins inside a context
@pytest.mark.parametrize("P,pos0", [(7, 0), (8, 0), (9, 24), (17, 14), (31, 33), (40, 90)])
def test_attention_of_token_tiles(ctx, P, pos0):
    c = synth.preset("v3", "q2_k", False, n_layers=1, first_k_dense_replace=1, max_seq_len=192, vocab_size=1024)
    tokens = np.random.default_rng(P).integers(0, c.vocab_size, P)
    _assert_identical(compare_hydrate(ctx, c, None, seed=23, tokens=tokens, pos0=pos0), P, pos0)


# latent attention of 16 heads at a time (from 8 tokens on): contexts at both sides of 16 (a tile of keys, a step of the values), 64 (a sum of the
# softmax) and 128, up to the last one before the long-context kernels take over
@pytest.mark.parametrize("P,pos0", [(7, 0), (8, 0), (20, 1), (14, 55), (12, 123), (30, 294)])
def test_latent_attention_of_head_tiles(ctx, P, pos0):
    c = synth.preset("v3", "q2_k", True, n_layers=1, first_k_dense_replace=1, max_seq_len=384, vocab_size=1024)
    tokens = np.random.default_rng(P).integers(0, c.vocab_size, P)
    _assert_identical(compare_hydrate(ctx, c, None, seed=29, tokens=tokens, pos0=pos0), P, pos0)


# a key and value that overflow the cache's f16 (infinite) inside a tile of tokens: the tokens before it know nothing of them
def test_attention_before_an_infinite_value(ctx):
    import dsk
    c = synth.preset("tiny_v3", "q2_k", False, n_layers=1, first_k_dense_replace=1, v_head_dim=128, qk_nope_head_dim=128, qk_rope_head_dim=64, max_seq_len=96)
    T = synth.synth_model(c, seed=5)
    tokens = [int(t) for t in np.random.default_rng(3).integers(0, c.vocab_size, 30)]
    norm = T["model.layers.0.attn.kv_a_norm.weight"]

    def run(batched):
        m = dsk.Model(ctx, c, T, options={"q2k_tiles": 2})
        try:
            assert m.hydrate_why_not() == ""
            m.set_trace(True)
            if batched:
                m.hydrate(tokens, 0, dsk.MODE_OUTPUT_LOGITS)
                x = [m.hydrate_trace_x(0, i) for i in range(len(tokens))]
            else:
                x = [a[0] for a in _loop(m, tokens, 0, trace=True)[1]]
            return x, [np.asarray(r).view(np.float16).astype(np.float32) for r in _caches(m, c, len(tokens))[0]]
        finally:
            m.close()

    largest = np.max([np.abs(r).max(axis=1) for r in run(False)[1]], axis=0)
    first = 1 + int(np.argmax(largest[1:]))
    norm.data = (norm.data * np.float32(1.05 * 65504 / largest[first])).astype(np.float32)
    (want, rows), (got, same) = run(False), run(True)
    bad = ~np.isfinite(rows[0]).all(axis=1) | ~np.isfinite(rows[1]).all(axis=1)
    assert bad.any() and not bad[0]
    first = int(np.argmax(bad))
    for i in range(first):
        assert np.isfinite(want[i]).all() and np.array_equal(want[i], got[i]), i
        assert np.array_equal(rows[0][i], same[0][i]) and np.array_equal(rows[1][i], same[1][i]), i


# An infinite value inside every token's context: attention gives what the kernel for few tokens gives (chunks of up to 7), a tile of a single token whose
# context is whole steps of 32 included (the 17th: 32, 96 or 128 positions)
@pytest.mark.parametrize("pos0", [15, 79, 111])
def test_attention_over_an_infinite_value(ctx, pos0):
    import dsk
    c = synth.preset("tiny_v3", "q2_k", False, n_layers=1, first_k_dense_replace=1, v_head_dim=128, qk_nope_head_dim=128, qk_rope_head_dim=64, max_seq_len=160)
    T = synth.synth_model(c, seed=5)
    tokens = [int(t) for t in np.random.default_rng(3).integers(0, c.vocab_size, pos0 + 17)]
    width = c.n_heads * 128

    def run(sizes):
        m = dsk.Model(ctx, c, T, options={"q2k_tiles": 2, "hydrate_tap_layer": 0})
        try:
            assert m.hydrate_why_not() == ""
            m.hydrate(tokens[:pos0], 0)
            rows = m.get_cache_rows(0, "v_cache", 0, pos0, width)
            for i in (0, pos0 - 1):  # (columns of two waves)
                rows[i, 5 + i % 2 * 64::128] = 0x7C00
            m.set_cache_rows(0, "v_cache", 0, rows)
            out, at = [], pos0
            for n in sizes:
                m.hydrate(tokens[at:at + n], at)
                out.append(m.hydrate_buffer("att_out", 0, n, width))
                at += n
            return np.concatenate(out)
        finally:
            m.close()

    want, got = run([7, 7, 3]), run([17])
    assert np.isposinf(want).any(axis=1).all() and not np.isnan(want).any()
    assert np.array_equal(want, got, equal_nan=True)
