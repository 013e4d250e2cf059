"""The recurrences of prompts over chunks of 16 tokens (kernels_chunk_scan.hip) at the edges of their loop: sequences of one to nine chunks, whole
and ragged, together in one step (a workgroup per sequence, head and 16 columns), with all key channels of a wave's tiles there (64 and
128) and not; a second portion starts from the kept state."""
import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu
LENGTHS = [1, 2, 15, 16, 17, 32, 33, 48, 64, 79, 80, 81, 96, 113, 144]


@pytest.mark.parametrize("layer", [
    U.channel_delta(U.delta(2, 1, 128, 40, 3)), U.channel_delta(U.delta(2, 2, 64, 17, 2)), U.channel_delta(U.delta(1, 1, 100, 16, 2)),
    U.parallel(right=U.mlstm(2, 64, 32, 9.0)), U.parallel(right=U.mlstm(1, 128, 31, 9.0)), U.parallel(right=U.mlstm(2, 48, 16, 9.0))],
    ids=["delta-128", "delta-64", "delta-100", "mlstm-64", "mlstm-128", "mlstm-48"])
def test_chunks_of_ragged_sequences(case, layer):
    check(case(U.config([layer], width=72, eps=0.05)))


@pytest.mark.parametrize("dim", [64, 128, 36])
def test_chunks_of_time_mixing(case, dim):
    check(case(U.sandwich([U.no_ff(U.wkv(2, dim))], width=72)))


# key sizes past 128 (four tiles a wave, all of them there and not), several heads and column tiles, sequences of all lengths side by side
@pytest.mark.parametrize("layer", [U.channel_delta(U.delta(2, 1, 130, 40, 3)), U.channel_delta(U.delta(3, 3, 256, 33, 2)),
                                   U.parallel(right=U.mlstm(3, 130, 33, 9.0)), U.parallel(right=U.mlstm(2, 256, 16, 9.0))],
                         ids=["delta-130", "delta-256", "mlstm-130", "mlstm-256"])
def test_chunks_of_large_keys(case, layer):
    check(case(U.config([layer], width=72, eps=0.05)))


def test_gates_of_long_sequences(case):
    """the running maximum goes from wave to wave every 64 tokens, from round to round every 1024"""
    check(case(U.config([U.parallel(right=U.mlstm(1, 16, 16, 9.0))], width=72, eps=0.05)), [63, 64, 65, 128, 1023, 1024, 1025, 1090])


def check(K, LENGTHS=LENGTHS):
    toks = [K.tokens(n + 5, seed=n) for n in LENGTHS]
    want = [K.want(t) for t in toks]
    seqs = [K.lm.seq_open() for _ in toks]
    got = K.lm.step([(s, t[:n], range(n)) for s, t, n in zip(seqs, toks, LENGTHS)])
    assert U.err(got, np.concatenate([w[:n] for w, n in zip(want, LENGTHS)])) < 3e-5  # (as the tests of single mechanisms)
    got = K.lm.step([(s, t[n:], range(5)) for s, t, n in zip(seqs, toks, LENGTHS)])
    assert U.err(got, np.concatenate([w[n:] for w, n in zip(want, LENGTHS)])) < 3e-5
