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


# What goes in and comes out: heads of up to 64, 128 and 256 elements, whole and not, one to four of them to a wave at once and a last group of heads that is
# short; two to five taps (five: any number), portions shorter than the taps in front of another.  (The last one 300 wide has a row that nearly cancels in
# front of a norm: 3.1e-5 of error here, 1.6e-5 token by token; 72 wide 6e-7.)
@pytest.mark.parametrize("c", [
    U.config([U.channel_delta(U.delta(1, 1, 16, 65, 4))], width=72, eps=0.05), U.config([U.channel_delta(U.delta(5, 5, 65, 128, 4))], width=72, eps=0.05),
    U.config([U.channel_delta(U.delta(3, 1, 129, 64, 4))], width=72, eps=0.05), U.config([U.channel_delta(U.delta(6, 3, 20, 129, 5))], width=72, eps=0.05),
    U.config([U.parallel(right=U.mlstm(5, 16, 64, 9.0))], width=72, eps=0.05), U.config([U.parallel(right=U.mlstm(9, 16, 129, 9.0))], width=72, eps=0.05),
    U.sandwich([U.no_ff(U.head_delta(17, 1, 20, 64, 4))], width=70, taps=2), U.sandwich([U.no_ff(U.head_delta(3, 3, 64, 256, 3))], width=257, taps=3),
    U.sandwich([U.no_ff(U.wkv(18, 16))], width=72, taps=5), U.sandwich([U.no_ff(U.wkv(5, 65))], width=72), U.sandwich([U.no_ff(U.wkv(3, 130))], width=72)],
    ids=["delta-65", "delta-128", "delta-64", "delta-129", "mlstm-64", "mlstm-129", "head-64", "head-256", "wkv-16", "wkv-65", "wkv-130"])
def test_chunks_of_heads_of_all_sizes(case, c):
    check(case(c))


# 16-bit values are loads of two bytes out of buffers that start at any two bytes (odd numbers of columns) and end with the sequence: against the
# recurrence token by token on the same 16-bit inputs.  Both sum in 32 bits, so that a value may be rounded to the other of two neighbours behind
# the mixer and once more behind the last norm, 2^-8 of it each; a wrong row or column is far more.
@pytest.mark.parametrize("c", [U.config([U.parallel(right=U.mlstm(3, 64, 31, 9.0))], width=72, eps=0.05), U.config([U.parallel(right=U.mlstm(2, 130, 17, 9.0))], width=72, eps=0.05),
                               U.sandwich([U.no_ff(U.wkv(3, 21))], width=72), U.sandwich([U.no_ff(U.wkv(2, 64))], width=72)],
                         ids=["mlstm-64", "mlstm-130", "wkv-21", "wkv-64"])
def test_chunks_in_16_bits(case, c):
    K, L = case(c, dtype="bfloat16"), case(c, dtype="bfloat16", options="chunk_scan=0")
    toks = [K.tokens(n + 5, seed=n) for n in LENGTHS]
    a, b = [K.lm.seq_open() for _ in toks], [L.lm.seq_open() for _ in toks]
    for cut in ([(t[:n], range(n)) for t, n in zip(toks, LENGTHS)], [(t[n:], range(5)) for t, n in zip(toks, LENGTHS)]):
        got, want = K.lm.step([(s, *e) for s, e in zip(a, cut)]), L.lm.step([(s, *e) for s, e in zip(b, cut)])
        assert U.err(got, want) < 2 ** -7


@pytest.mark.parametrize("n", [1023, 1024, 1025, 1090, 2047, 2048, 2049, 2100, 3200])
def test_gates_of_a_long_sequence(case, n):
    """the running maximum goes from wave to wave every 64 tokens and from round to round every 1024, the third round into the first one's buffer:
    one sequence in one pass (whose rows the trace holds)"""
    K = case(U.config([U.parallel(right=U.mlstm(2, 16, 16, 9.0))], width=72, eps=0.05), options="piece_tokens=4096")
    t = K.tokens(n + 5, seed=n)
    want = K.want(t)
    K.lm.set_trace(True)
    s = K.lm.seq_open()
    got = K.lm.step([(s, t[:n], range(n))])
    K.lm.trace_rows(0, n)  # (an error if the last pass held fewer)
    assert U.err(got, want[:n]) < 3e-5
    assert U.err(K.lm.step([(s, t[n:], range(5))]), want[n:]) < 3e-5


def test_gates_of_long_sequences(case):
    """... and sequences of such lengths side by side, as passes of 2048 rows cut them"""
    check(case(U.config([U.parallel(right=U.mlstm(1, 16, 16, 9.0))], width=72, eps=0.05)), [63, 64, 65, 128, 1023, 1024, 1025, 1090])


def check(K, LENGTHS=LENGTHS):
    toks = [K.tokens(n + 5, seed=n) for n in LENGTHS]
    want = [K.want(t) for t in toks]
    seqs = [K.lm.seq_open() for _ in toks]
    got = K.lm.step([(s, t[:n], range(n)) for s, t, n in zip(seqs, toks, LENGTHS)])
    assert U.err(got, np.concatenate([w[:n] for w, n in zip(want, LENGTHS)])) < 3e-5  # (as the tests of single mechanisms)
    got = K.lm.step([(s, t[n:], range(5)) for s, t, n in zip(seqs, toks, LENGTHS)])
    assert U.err(got, np.concatenate([w[n:] for w, n in zip(want, LENGTHS)])) < 3e-5
