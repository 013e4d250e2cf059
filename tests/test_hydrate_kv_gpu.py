"""Key and value rows of a batched prompt, 16 heads of a token to a workgroup (kernels_hydrate.hip hyd_kv_write4_kernel): both layouts of the rotated part, heads that are
no whole workgroups, more values than a workgroup requests at once.  The bar is the loop's bits."""
import numpy as np
import pytest

from tools import synth

from .test_hydrate_gpu import _assert_identical, compare_hydrate

pytestmark = pytest.mark.gpu

V2 = dict(arch="DeepseekV2ForCausalLM", scoring_func="softmax", norm_topk_prob=False)


@pytest.mark.parametrize("over", [dict(n_heads=20), dict(n_heads=20, **V2), dict(n_heads=4, qk_rope_head_dim=16, **V2),
                                  dict(n_heads=18, qk_nope_head_dim=192, v_head_dim=128, qk_rope_head_dim=64, **V2)],
                         ids=["20 heads", "20 heads, halves", "rope 16, halves", "18 heads of 320, halves"])
def test_key_and_value_rows(ctx, over):
    c = synth.preset("tiny_v3", "q2_k", False, **dict(dict(n_layers=2, max_seq_len=64), **over))
    tokens = np.random.default_rng(3).integers(0, c.vocab_size, 21)
    _assert_identical(compare_hydrate(ctx, c, None, seed=5, tokens=tokens), 21, 0)
