"""Logits in rows that the model lends (dsk_rows_lend): whose they are, what happens when none is left."""
import ctypes as C
import gc

import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


def model(ctx, tmp_path, dtype="bfloat16", vocab=208, **kw):
    return U.Case(ctx, tmp_path, U.sandwich([U.wkv(), U.no_ff(U.head_delta())], vocab=vocab), dtype=dtype, **kw)


def lent(a):
    return not a.flags.owndata


def run(K, rows, seed):
    """logits of two steps of `rows` sequences"""
    seqs, toks = [K.lm.seq_open() for _ in range(rows)], [K.tokens(2, seed=seed + r) for r in range(rows)]
    out = [K.lm.step([(s, t[i:i + 1], [0]) for s, t in zip(seqs, toks)]) for i in range(2)]
    for s in seqs:
        K.lm.seq_close(s)
    return out


@pytest.mark.parametrize("rows", [1, 3, 16])
def test_kept_rows_stay_what_they_are(ctx, tmp_path, rows):
    K = model(ctx, tmp_path)
    want = [a.copy() for seed in range(4) for a in run(K, rows, 100 * seed)]
    got = [a for seed in range(4) for a in run(K, rows, 100 * seed)]  # eight arrays held, the model lends four
    assert sum(map(lent, got)) == 4 and all(np.array_equal(a, b) for a, b in zip(got, want))
    t = K.tokens(150)  # a block of wanted rows of the model's own while others are held
    K.got(t)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    K.lm.close()
    assert all(np.array_equal(a, b) for a, b in zip(got, want))  # (and the model is gone)


def test_rows_come_back(ctx, tmp_path):
    K = model(ctx, tmp_path)
    whole = K.got(K.tokens(150))
    held = run(K, 2, 1) + run(K, 2, 2)
    assert all(map(lent, held)) and not any(map(lent, run(K, 2, 3)))
    part = held[0][1]  # a view keeps the rows
    value = part.copy()
    held.clear()
    gc.collect()
    again = run(K, 2, 4)
    assert lent(again[0]) and lent(again[1]) and np.array_equal(part, value)
    assert np.array_equal(K.got(K.tokens(150)), whole)


# 17 rows and vocabularies that are not whole tiles do not fit; prompts' last tokens do
@pytest.mark.parametrize("vocab,n", [(208, 17), (203, 2), (208, 16)])
def test_rows_of_prompts(ctx, tmp_path, vocab, n):
    K = model(ctx, tmp_path, vocab=vocab, dtype="float32")
    t = K.tokens(40)
    s = K.lm.seq_open()
    got = K.lm.step([(s, t, range(40 - n, 40))])
    assert lent(got) == (n <= 16 and vocab == 208) and U.err(got, K.want(t)[-n:]) < U.F32
    rows, hold = C.c_void_p(), C.c_void_p()
    import dsk
    with pytest.raises(dsk.DskError):
        dsk.check(dsk.lib().dsk_rows_lend(K.lm.h, 0, C.byref(rows), C.byref(hold)))


# Rows that are borrowed while a prompt's logits are on their way stay the borrower's: a prompt that wants many rows uses the borrowers' own room for
# them only if nobody has borrowed any, and lends none meanwhile
def test_rows_borrowed_beside_a_prompt(ctx, tmp_path):
    import threading

    import dsk
    K = model(ctx, tmp_path, vocab=4096)
    t, stop, seen = K.tokens(150), threading.Event(), []

    def borrow():
        n = 0
        while not stop.is_set():
            rows, hold = C.c_void_p(), C.c_void_p()
            dsk.check(dsk.lib().dsk_rows_lend(K.lm.h, 16, C.byref(rows), C.byref(hold)))
            if not hold.value:
                continue
            a = np.ctypeslib.as_array(C.cast(rows, C.POINTER(C.c_float)), (16, 4096))
            n += 1
            a[:] = n
            ok = True
            for _ in range(20):
                ok &= bool((a == n).all())
            seen.append(ok)
            dsk.lib().dsk_rows_return(hold)

    b = threading.Thread(target=borrow)
    want = K.got(t)
    b.start()
    try:
        for _ in range(40):
            assert np.array_equal(K.got(t), want)
    finally:
        stop.set()
        b.join()
    assert seen and all(seen)
