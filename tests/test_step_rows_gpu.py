"""Rows of decoding steps: the residual sum of a sandwich layer shared by several workgroups (join_device.h), and the launch that makes its rows
beside the product that reads them (kernels_enter.hip)."""
import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


def stack(width, ff=72, taps=4):
    return U.sandwich([dict(U.wkv(2, 16), mlp=U.dense(ff)), dict(U.head_delta(3, 3, 16, 20, 4), mlp=U.dense(ff)), U.no_ff(U.latent(2, 16, 8, 16, 12, 20, 6))],
                      width=width, taps=taps)


# one workgroup a row up to 1024, two up to 2048, four behind that, with one or two groups of four channels a thread; widths that do not divide evenly, ones
# that the general kernel takes (odd, wider, other taps); sums of one, two and eight parts
@pytest.mark.parametrize("width,ff,taps", [(32, 72, 4), (1020, 72, 4), (1024, 2100, 4), (1028, 72, 4), (2048, 4200, 4), (2052, 72, 4), (4100, 1100, 4), (8192, 72, 4),
                                           (8196, 72, 4), (1027, 72, 4), (1020, 72, 3), (2044, 72, 5)])
def test_rows_in_32_bits(ctx, tmp_path, width, ff, taps):
    K = U.Case(ctx, tmp_path, stack(width, ff, taps))
    t = K.tokens(9)
    assert U.err(K.got(t, range(1, 9)), K.want(t)) < U.F32


def steps(K, rows, n=7):
    """logits of n steps of single tokens (the second is captured, the others replay it), other work between them"""
    seqs, out = [K.lm.seq_open() for _ in range(rows)], []
    toks = [K.tokens(n, seed=r) for r in range(rows)]
    for i in range(n):
        out.append(K.lm.step([(s, t[i:i + 1], [0]) for s, t in zip(seqs, toks)]))
        if i % 2:
            K.got(toks[0][:5])
    for s in seqs:
        K.lm.seq_close(s)
    return np.array(out)


# the same sums in the same order as two launches: the same bits.  Rounds of 16 k tiles a wave: less than one, one, more; odd numbers of feature tiles
@pytest.mark.parametrize("rows", [1, 3, 8])
@pytest.mark.parametrize("width", [36, 1100, 2048])
@pytest.mark.parametrize("design", ["ranutar", "timerax"])
def test_rows_beside_their_product(ctx, tmp_path, design, width, rows):
    c = stack(width, 136) if design == "ranutar" else U.mixed(width)
    a, b = (U.Case(ctx, tmp_path / str(i), c, dtype="bfloat16", options=f"enter_ahead={i}") for i in (1, 0))
    x, y = steps(a, rows), steps(b, rows)
    assert a.lm.info("enter_launches") > 0 and b.lm.info("enter_launches") == 0
    assert np.isfinite(x).all() and np.array_equal(x, y)


# logits of some of a step's rows, in any place: the last launch makes those rows alone.  The norm by itself (the final one) in front of the output product
@pytest.mark.parametrize("want", [[0], [2], [1, 3], [0, 1, 2, 4]])
@pytest.mark.parametrize("design", ["ranutar", "timerax"])
def test_some_rows_beside_the_output_product(ctx, tmp_path, design, want):
    c = stack(1100, 136) if design == "ranutar" else U.mixed(1100)
    got = []
    for i in (1, 0):
        K = U.Case(ctx, tmp_path / str(i), c, dtype="bfloat16", options=f"enter_ahead={i}")
        toks, seqs = [K.tokens(5, seed=r) for r in range(5)], [K.lm.seq_open() for _ in range(5)]
        some = [K.lm.step([(s, t[n:n + 1], [0] if r in want else []) for r, (s, t) in enumerate(zip(seqs, toks))]).copy() for n in range(4)]  # (eager, captured, replayed)
        every = K.lm.step([(s, t[4:5], [0]) for s, t in zip(seqs, toks)]).copy()
        got.append((np.array(some), every))
        assert (K.lm.info("enter_launches") > 0) == bool(i)
    assert got[0][0].shape[1] == len(want) and np.isfinite(got[0][0]).all()
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    K = U.Case(ctx, tmp_path / "2", c, dtype="bfloat16")  # ... which are those of steps that want all
    seqs = [K.lm.seq_open() for _ in range(5)]
    for n in range(4):
        assert np.array_equal(K.lm.step([(s, t[n:n + 1], [0]) for s, t in zip(seqs, toks)])[want], got[0][0][n])


def test_a_wait_without_end_is_an_error(ctx, tmp_path):
    import dsk
    K = U.Case(ctx, tmp_path, stack(2048, 136), dtype="bfloat16", options="enter_spins=0")
    s = K.lm.seq_open()
    with pytest.raises(dsk.DskError, match="gave up"):
        for t in K.tokens(4):
            K.lm.step([(s, [t], [0])])


# Behind it: the step's sequences are closed to steps (their recurrent states were updated in place), others and new ones go on, in two launches; the model's
# own sequence starts anew at position 0
def test_a_step_that_gave_up_is_not_taken_again(ctx, tmp_path):
    import dsk
    K = U.Case(ctx, tmp_path / "0", stack(2048, 136), dtype="bfloat16", options="enter_spins=0")
    same = U.Case(ctx, tmp_path / "1", stack(2048, 136), dtype="bfloat16", options="enter_ahead=0")
    t, lone = K.tokens(6), K.lm.seq_open()
    a, b = K.lm.seq_open(), same.lm.seq_open()
    K.lm.step([(lone, t[:3], [])])
    n = 0
    with pytest.raises(dsk.DskError, match="gave up"):
        for n in range(6):
            K.lm.step([(a, t[n:n + 1], [0])])
    for _ in range(2):
        with pytest.raises(dsk.DskError, match="no valid state"):
            K.lm.step([(a, t[n:n + 1], [0])])
    with pytest.raises(dsk.DskError, match="no valid state"):
        K.lm.step([(lone, t[3:4], [0]), (a, t[n:n + 1], [0])])
    before = K.lm.info("enter_launches")
    K.lm.seq_close(a)
    a = K.lm.seq_open()
    for i in range(6):  # (eager, captured, replayed)
        assert np.array_equal(K.lm.step([(a, t[i:i + 1], [0])]), same.lm.step([(b, t[i:i + 1], [0])])), i
    assert K.lm.info("enter_launches") == before
    c = same.lm.seq_open()
    same.lm.step([(c, t[:3], [])])
    assert np.array_equal(K.lm.step([(lone, t[3:4], [0])]), same.lm.step([(c, t[3:4], [0])]))
