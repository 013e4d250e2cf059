"""Softmax attention of prompts (attn_tile.h) at the edges of its tiles: 64 queries, 64 keys, whole heads to an XCD (8 and 16 heads) and not."""
import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


# chunks that end inside a tile of keys, at its end and behind it (a tile that all of a wave's queries see is not masked), a second portion that reads kept keys
# and its own in one tile, sequences side by side; windows likewise.  Key sizes of one to eight k tiles, value sizes of up to 16 (the instances of attn_sizes)
@pytest.mark.parametrize("c", [
    U.config([U.parallel(left=U.attn(8, 2, 40, 24, 64))], width=72, eps=0.05), U.config([U.parallel(left=U.attn(16, 16, 128, 128, 100))], width=72, eps=0.05),
    U.config([U.parallel(left=U.attn(8, 4, 72, 100, 4096))], width=72, eps=0.05), U.config([U.parallel(left=U.attn(12, 4, 200, 130, 129))], width=72, eps=0.05),
    U.sandwich([U.no_ff(U.latent(8, 24, 12, 20, 36, 28, 64))]), U.sandwich([U.no_ff(U.latent(16, 128, 64, 128, 36, 60, 100))]),
    U.sandwich([U.no_ff(U.latent(9, 150, 34, 200, 36, 28, 700))])],
    ids=["chunk-64", "chunk-100", "chunk-4096", "chunk-129", "window-64", "window-100", "window-700"])
# Tolerances as in the tests of single mechanisms.  In bfloat16 theirs is of the worst of some tens of rows, here of 522: chunk-129 comes to 0.0601 there, all others
# stay below 0.06.  That is bfloat16, not the tiles: with masks everywhere and operands read where they are used it was the same 0.060079.
@pytest.mark.parametrize("dtype,tol", [("float32", 3e-5), ("bfloat16", 1.3 * U.B16)])
def test_attention_at_the_edges_of_its_tiles(case, c, dtype, tol):
    K = case(c, dtype=dtype)
    cuts = [(63, 66), (64, 2), (65, 200), (130, 63), (200, 129)]
    toks = [K.tokens(a + b, seed=a) for a, b in cuts]
    want = [K.want(t) for t in toks]
    seqs = [K.lm.seq_open() for _ in toks]
    got = K.lm.step([(s, t[:a], range(a)) for s, t, (a, _) in zip(seqs, toks, cuts)])
    assert U.err(got, np.concatenate([w[:a] for w, (a, _) in zip(want, cuts)])) < tol
    got = K.lm.step([(s, t[a:], range(b)) for s, t, (a, b) in zip(seqs, toks, cuts)])
    assert U.err(got, np.concatenate([w[a:] for w, (a, _) in zip(want, cuts)])) < tol
