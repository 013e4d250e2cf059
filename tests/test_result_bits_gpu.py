"""Results that keep their bits.

A router decides close calls by the last bits of what it reads, and a call that goes the other way is no rounding any more: behind a prompt of some hundred
tokens and 27 layers with routers a step's logits have come out 0.13 apart, relative, after a norm's sum had been rounded in another place.  So where a sum is rounded, and
the order of sums that routers read, are part of these models' results: tests/golden/result_bits.npz holds logits of three layers at full width, and of a sandwich
design without feed-forward products.  Whoever changes them for a reason shows first, with the same experts chosen, that nothing but rounding moved, and
writes the file anew (DSK_WRITE_BITS=1)."""
import os

import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu
FILE = os.path.join(os.path.dirname(__file__), "golden", "result_bits.npz")


def routed():
    moe = U.moe(64, 6, 1408, 7.0, 2816, 7.0)
    delta = U.delta(16, 16, 128, 128)
    return U.config([U.channel_delta(delta, moe), U.channel_delta(delta, moe), U.parallel(U.attn(16, 4, 128, 128, 4096, 0.0883883, 64, 500000.0), U.mlstm(16, 64, 128, 15.0), moe)],
                    width=2048, vocab=208)


def sandwich():
    return U.sandwich([U.no_ff(U.wkv(7, 72)), U.no_ff(U.head_delta(3, 3, 128, 64)), U.no_ff(U.latent(3, 64, 16, 64, 36, 28, 50))], width=2048, vocab=208)


def odd():
    return U.mixed(250, vocab=208)  # (routers, pairs of mixers, a width that four does not divide)


# last tokens of prompts of one, three and more row tiles, of several at once, and of two steps behind them
LENGTHS = {"routed": ((40,), (301,), (1300, 77), (2048,)), "sandwich": ((45,), (17, 3, 130)), "odd": ((45,), (17, 3, 130))}


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("design", ["routed", "sandwich", "odd"])
def test_logits_keep_their_bits(ctx, design, dtype):
    import dsk
    c = {"routed": routed, "sandwich": sandwich, "odd": odd}[design]()
    lm, rng, got = dsk.LM(ctx, dtype=dtype, config=c, seed=3), np.random.default_rng(11), {}
    for lengths in LENGTHS[design]:
        seqs = [lm.seq_open() for _ in lengths]
        out = [lm.step([(s, rng.integers(0, 208, n), [n - 1]) for s, n in zip(seqs, lengths)])]
        out += [lm.step([(s, rng.integers(0, 208, 1), [0]) for s in seqs]) for _ in range(2)]
        got["_".join([design, dtype, *map(str, lengths)])] = np.array(out)
        for s in seqs:
            lm.seq_close(s)
    lm.close()
    if os.environ.get("DSK_WRITE_BITS"):
        np.savez_compressed(FILE, **{**(dict(np.load(FILE)) if os.path.exists(FILE) else {}), **got})
    want = np.load(FILE)
    for k, v in got.items():
        assert np.isfinite(v).all() and np.array_equal(v, want[k]), (k, np.abs(v - want[k]).max())
