"""Products of prompts at the edges of their tiles (kernels_lin.hip), against the plain statement of the design (oracle/layered.py)."""
import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import dsk
    c = dsk.Ctx(0)
    yield c
    c.close()


def no_mixers(W):
    for k in W:
        if k.endswith("left.out") or k.endswith("right.out"):
            W[k][:] = 0


# one expert takes every row (and the shared one too), so a prompt's length is its number of rows: both sides of the 32-, 64- and 128-row
# forms; ff: feature tiles short of, at and behind a workgroup's 256 features (gate and up: 2 ff of them)
@pytest.mark.parametrize("ff,shared", [(40, 0), (128, 24), (136, 272)])
@pytest.mark.parametrize("dtype,tol", [("bfloat16", 0.02), ("float32", U.F32)])
def test_expert_products_at_the_edges_of_row_tiles(ctx, tmp_path, ff, shared, dtype, tol):
    # bf16: inputs, hidden values and outputs are each rounded to 2^-9, relative to values of about the result's size: 3 roundings of
    # independent terms, far below 0.02 of the rows' scale
    K = U.Case(ctx, tmp_path, U.config([U.parallel(mlp=U.moe(1, 1, ff, 0.8, shared, 1.2))], width=264), edit=no_mixers, dtype=dtype)
    t = K.tokens(257)
    want = []
    K.ref.run(U.O.Sequence(K.ref), t, want)
    K.lm.set_trace(True)
    for n in (17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 161, 193, 257):
        s = K.lm.seq_open()
        K.lm.step([(s, t[:n], [n - 1])])
        assert U.err(K.lm.trace_rows(0, n), want[0][:n]) < tol, n
        K.lm.seq_close(s)


# k tiles of 32 in a ring of four: 2, 4, 6, 8, 10 and 14 of them (gate and up: the width; down: ff), so that 2, 4 or 6 are left behind whole rounds
@pytest.mark.parametrize("width,ff", [(64, 448), (128, 320), (192, 256), (256, 192), (320, 128), (448, 64)])
def test_expert_products_of_few_rows_and_k_tiles(ctx, tmp_path, width, ff):
    K = U.Case(ctx, tmp_path, U.config([U.parallel(mlp=U.moe(1, 1, ff, 0.8, 0))], width=width), edit=no_mixers, dtype="bfloat16")
    t, want = K.tokens(64), []
    K.ref.run(U.O.Sequence(K.ref), t, want)
    K.lm.set_trace(True)
    for n in (17, 32, 33, 48, 64):
        s = K.lm.seq_open()
        K.lm.step([(s, t[:n], [n - 1])])
        assert U.err(K.lm.trace_rows(0, n), want[0][:n]) < 0.02, n
        K.lm.seq_close(s)


# several experts, rows spread unevenly: groups of four row tiles with and without neighbours of the same expert, a last group that is short
@pytest.mark.parametrize("experts,top", [(3, 1), (6, 2), (40, 7)])
def test_expert_products_over_many_experts(ctx, tmp_path, experts, top):
    K = U.Case(ctx, tmp_path, U.config([U.parallel(mlp=U.moe(experts, top, 72, 0.8, 40, 1.2))]), edit=no_mixers)
    K.check_trace(700, cuts=([129],))


# 32-bit activations are multiplied in three bf16 pieces.  Two pieces alone would be up to 2^-16 off; 32-bit sums, through the model's four
# products and a softmax, stay under a quarter of that (v_mfma_f32_16x16x4_f32 gave up to 2.2e-6 here, this gives up to 2.1e-6).
@pytest.mark.parametrize("width", [64, 328, 1000])
def test_32_bit_products_keep_32_bits(ctx, tmp_path, width):
    K = U.Case(ctx, tmp_path, U.sandwich([U.no_ff(U.latent())], width=width), dtype="float32")
    t = K.tokens(140)
    assert U.err(K.got(t), K.want(t)) < 2.0 ** -18


# decoding steps: from 9 rows and 1536 tiles on a workgroup takes four feature tiles.  Vocabulary, experts' hidden sizes and width leave a last group
# of 1, 2 or 3 tiles (pairs: of one); experts without a row, with one and with several.  A row's sums are added in the same order
# either way: the bits of steps of 8 rows.
@pytest.mark.parametrize("width,ff,vocab", [(400, 264, 24600), (432, 200, 24620), (264, 296, 24590)])
def test_steps_of_many_tiles_per_workgroup(ctx, tmp_path, width, ff, vocab):
    K = U.Case(ctx, tmp_path, U.config([U.parallel(mlp=U.moe(100, 7, ff, 0.8, 40, 1.2))], width=width, vocab=vocab), dtype="bfloat16")
    toks = [K.tokens(3, seed=n) for n in range(16)]

    def decode(sizes):
        seqs, out = [K.lm.seq_open() for _ in toks], []
        K.lm.step([(s, t[:2], []) for s, t in zip(seqs, toks)])
        for n in sizes:
            part = slice(len(out), len(out) + n)
            out.extend(K.lm.step([(s, t[2:], [0]) for s, t in zip(seqs[part], toks[part])]))
        for s in seqs:
            K.lm.seq_close(s)
        return np.array(out)

    few = decode([8, 8])
    assert np.array_equal(decode([16]), few)
    assert np.array_equal(decode([9, 7]), few)
    assert U.err(few[:1], K.want(toks[0])[-1:]) < K.tol


# Infinite weights and activations that overflow, in 32 bits: an infinite sum comes out, as it does of one 32-bit instruction, wherever its terms
# agree in sign (of an activation's three pieces the last is zero once in 256, and zero times infinity is no number)
@pytest.mark.parametrize("where", ["expert", "head", "hidden"])
def test_infinite_values_in_32_bit_products(ctx, tmp_path, where):
    width, ff, n = 120, 40, 60

    def edit(W):
        no_mixers(W)
        if where == "head":
            for v in range(203):
                W["head"][v, v % width] = np.inf * (-1) ** v
        elif where == "expert":
            for f in range(0, width, 2):
                W["l0.mlp.e0.down"][f, f % ff] = np.inf
        else:  # a hidden value of 1e25 x 1e25, times weights on both sides of 128
            W["l0.mlp.e0.gate"][3] *= 1e25
            W["l0.mlp.e0.up"][3] *= 1e25
            W["l0.mlp.e0.down"][:, 3] = np.resize([0.5, 300, -128, 2.0 ** 20, -1, 127], width)
    layer = U.parallel(mlp=U.moe(1, 1, ff, 3e38 if where == "hidden" else 0.8, 0))
    K = U.Case(ctx, tmp_path, U.config([layer], width=width), edit=edit)
    t, trace = K.tokens(n), []
    with np.errstate(all="ignore"):
        logits = K.ref.run(U.O.Sequence(K.ref), t, trace)
    K.lm.set_trace(True)
    s = K.lm.seq_open()
    got = K.lm.step([(s, t, range(n))])
    want = logits
    if where != "head":
        got = K.lm.trace_rows(0, n)
        with np.errstate(over="ignore"):
            want = trace[0].astype(np.float32)
        assert np.isinf(want).any()
    assert not np.isnan(want).any()
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]) and np.isfinite(got[~inf]).all()
    assert np.abs(got[~inf] - want[~inf]).max() < U.F32 * 20


# The decay of time mixing multiplies 32-bit activations in bfloat16 runs too, by the 32-bit matrix instruction: a pass of 20 single tokens (a
# prompt's kernels) and steps of 10 (a step's) give the same bits where every sum runs over one k tile.  Its terms nearly cancel in pairs, so that
# sums added up otherwise show behind the rounding to bfloat16.
def test_decay_of_prompts_and_steps_in_bfloat16(ctx, tmp_path):
    def edit(W):
        W["l0.mix.w1"][1::2] = W["l0.mix.w1"][::2] * (1 + 2.0 ** -6)
        W["l0.mix.w2"] *= 256
        W["l0.mix.w2"][:, 1::2] = -W["l0.mix.w2"][:, ::2]
    K = U.Case(ctx, tmp_path, U.sandwich([U.no_ff(U.wkv(2, 16))], width=32), edit=edit, dtype="bfloat16", options="fused_decode=0", rank_a=32)
    toks = [K.tokens(16, seed=n) for n in range(20)]
    K.lm.set_trace(True)

    def rows(size):
        seqs, out = [K.lm.seq_open() for _ in toks], []
        for i in range(16):
            for a in range(0, 20, size):
                K.lm.step([(s, t[i:i + 1], []) for s, t in zip(seqs[a:a + size], toks[a:a + size])])
                out.append(K.lm.trace_rows(0, size))
        for s in seqs:
            K.lm.seq_close(s)
        return np.concatenate(out)

    assert np.array_equal(rows(20), rows(10))


# its kernel: 64 features x 64 rows a workgroup, 32 x 32 a wave.  Feature tiles that end inside a wave's pair, a k of two and of four tiles
@pytest.mark.parametrize("heads,dim,rank", [(3, 20, 12), (5, 20, 70), (2, 52, 33), (1, 16, 100)])
def test_decay_at_the_edges_of_its_tiles(ctx, tmp_path, heads, dim, rank):
    K = U.Case(ctx, tmp_path, U.sandwich([U.no_ff(U.wkv(heads, dim))]), rank_a=rank)
    t, want = K.tokens(131), []
    K.ref.run(U.O.Sequence(K.ref), t, want)
    K.lm.set_trace(True)
    for n in (17, 31, 32, 33, 63, 64, 65, 97, 128, 131):
        s = K.lm.seq_open()
        K.lm.step([(s, t[:n], [n - 1])])
        assert U.err(K.lm.trace_rows(0, n), want[0][:n]) < U.F32, n
        K.lm.seq_close(s)


# Logits of up to 16 rows are stored into host memory by the product where the vocabulary is whole tiles of 16 (208), else copied behind it (203);
# more rows are copied.  Rows of prompts and of single tokens (eager, captured, replayed)
@pytest.mark.parametrize("vocab", [208, 203])
def test_logits_of_few_and_many_rows(ctx, tmp_path, vocab):
    K = U.Case(ctx, tmp_path, U.config([U.parallel(mlp=U.moe())], vocab=vocab), dtype="float32")
    t = K.tokens(26)
    want = K.want(t)
    for n in (1, 2, 15, 16, 17, 19):
        s = K.lm.seq_open()
        got = K.lm.step([(s, t[:20], range(20 - n, 20))])
        assert got.shape == (n, vocab) and U.err(got, want[20 - n:20]) < U.F32, n
        for i in range(20, 26):
            assert U.err(K.lm.step([(s, t[i:i + 1], [0])]), want[i:i + 1]) < U.F32, (n, i)
        K.lm.seq_close(s)
    seqs = [K.lm.seq_open() for _ in range(17)]
    for i in range(6):
        assert U.err(K.lm.step([(s, t[i:i + 1], [0]) for s in seqs]), np.repeat(want[i:i + 1], 17, 0)) < U.F32, i


# Stretches over several 256 x 256 tiles (LinStream): four to eight row tiles in 64 to 32 stretches of 67 feature tiles, a last tile of features that is not full, rows that end
# inside a tile, cuts at the first and last steps of a tile; blends (an operand per feature range) and xIELU.  The same rows by tiles of 128: sums in
# another order alone, 32 bits of a sum of up to 2048 products, bfloat16 behind it
@pytest.mark.parametrize("rows", [769, 1280, 1500, 1537, 2048])
def test_products_in_stretches(ctx, tmp_path, rows):
    c = U.sandwich([dict(U.wkv(32, 64), mlp=U.dense(16900))], width=2048, vocab=64)
    runs = [U.Case(ctx, tmp_path / str(tile), c, dtype="bfloat16", options=f"prompt_tile={tile}") for tile in (256, 128)]
    t = runs[0].tokens(rows)
    got = []
    for K in runs:
        K.lm.set_trace(True)
        for _ in range(2):  # (the words between the workgroups are zero again behind the first)
            s = K.lm.seq_open()
            K.lm.step([(s, t, [rows - 1])])
            got.append(K.lm.trace_rows(0, rows))
            K.lm.seq_close(s)
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1]) and np.array_equal(got[2], got[3])
    assert U.err(got[0], got[2]) < 0.02


# 32-bit products by workgroups of 64 and of 128 rows (whichever lin_cost finds the cheaper), bfloat16 products of workgroups with a compute unit each (one k
# step is less than their ring, a width of 64) and not: rows short of, at and behind a wave's 16 and a workgroup's
# 64 against the oracle, and, where 16 row tiles of 128 by 32 tiles of 128 features fill whole rounds of workgroups, the whole prompt at once against the
# same prompt in pieces of 64 rows.  Sums of up to 4096 products in another order of parts: the tolerance of 32 bits.
@pytest.mark.parametrize("dtype,tol", [("float32", U.F32), ("bfloat16", U.B16)])
@pytest.mark.parametrize("n", [17, 31, 33, 63, 64, 65, 129, 193, 1921, 2048])
def test_products_of_64_and_128_rows(ctx, tmp_path, n, dtype, tol):
    K = U.Case(ctx, tmp_path, U.sandwich([dict(U.wkv(4, 16), mlp=U.dense(4096))], width=64, vocab=72), dtype=dtype)
    t = K.tokens(n)
    s = K.lm.seq_open()
    got = K.lm.step([(s, t, range(n))])
    if n < 200:
        assert U.err(got, K.want(t)) < tol
        return
    p = K.lm.seq_open()
    cut = [K.lm.step([(p, t[i:i + 64], range(min(64, n - i)))]) for i in range(0, n, 64)]
    assert U.err(got, np.concatenate(cut)) < tol


# A sum has one order, that of k, whichever tiles make it: stretches (whose workgroups go on from each other's sums where they cut a tile), 256 x 256 and 128 x 128 tiles give
# the same bits, and those are near the oracle's values.  Stretches of one to two and a half tiles; a cut tile's front of one step up to all but one.
# A workgroup that does not find the front of its tile (at once, or as if it never did) adds up the whole: the same bits again
@pytest.mark.parametrize("rows,ff", [(257, 66000), (513, 40000), (769, 16900), (1280, 16900), (1500, 12300), (2048, 9000)])
def test_tiles_and_stretches_give_the_same_bits(ctx, tmp_path, rows, ff):
    c = U.sandwich([dict(U.wkv(2, 16), mlp=U.dense(ff))], width=256, vocab=64)
    got = []
    for i, options in enumerate(("prompt_tile=128", "prompt_tile=256", "prompt_tile=256,cut_looks=0", "prompt_tile=256,cut_looks=-1")):
        K = U.Case(ctx, tmp_path / str(i), c, dtype="bfloat16", options=options)
        K.lm.set_trace(True)
        for _ in range(2):  # (the words between the workgroups are zero again behind the first)
            s, t = K.lm.seq_open(), K.tokens(rows)
            K.lm.step([(s, t, [rows - 1])])
            got.append(K.lm.trace_rows(0, rows))
            K.lm.seq_close(s)
        K.lm.close()
    want = []
    K.ref.run(U.O.Sequence(K.ref), t, want)
    assert np.isfinite(got[0]).all() and all(np.array_equal(got[0], g) for g in got[1:]) and U.err(got[0], want[0]) < U.B16
