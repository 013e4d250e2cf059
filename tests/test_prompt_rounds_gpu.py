"""Plain matrices of a batched prompt where their workgroups come in more than one round: 32 tokens a workgroup from one round of 16 on,
and what is left for the last round in workgroups of 16 (hyd_gemm_launch).  The bar is that of the other prompt tests: the loop's bits."""
import numpy as np
import pytest

from tools import synth

from .test_hydrate_gpu import _assert_identical, compare_hydrate

pytestmark = pytest.mark.gpu


# DeepSeek-V3's width is 56 groups of 8 strips (wo, W2): 280 workgroups of 16 tokens or 168 of 32 at 65 (one token in the last) and 77,
# 280 at 129 (24 left for a second round, all of a last chunk of one token: no second halves), 336 at 161 and 177 (80 left, one and 17 tokens in the last
# chunk), 560 at 300 (48 left, 12 tokens in the last chunk)
@pytest.mark.timeout(600)
@pytest.mark.parametrize("P", [65, 77, 129, 161, 177, 300])
def test_rounds_of_plain_products(ctx, P):
    c = synth.preset("v3", "q2_k", False, n_layers=1, first_k_dense_replace=1, max_seq_len=P + 8)
    tokens = np.random.default_rng(P).integers(0, c.vocab_size, P)
    _assert_identical(compare_hydrate(ctx, c, None, seed=5, tokens=tokens), P, 0)
