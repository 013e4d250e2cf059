"""Rows of float weights (rows_dot_f, gemv_device.h): scale blocks whose sides are powers of two and not, ragged rows, and per-head rows of the
attention launch over several row sets of a wave (head sizes on both sides of 8 sets), against the oracle."""
import numpy as np
import pytest

from tools import synth

pytestmark = pytest.mark.gpu


# f32 sums of n terms in another order: a few times sqrt(n) roundings of 6e-8, far below 2e-5 of the largest value
@pytest.mark.parametrize("block", [(128, 128), (64, 32), (96, 80), (16, 128)])
@pytest.mark.parametrize("rows,n", [(33, 1408), (100, 2048), (7, 272)])
def test_scale_blocks_of_any_size(ctx, oracle, block, rows, n):
    rng = np.random.default_rng(rows + n)
    w8, s8 = synth.encode_f8_blocks((rng.standard_normal((rows, n)) / np.sqrt(n)).astype(np.float32), block)
    x = rng.standard_normal(n).astype(np.float32)
    want = oracle.gemv(2, w8, rows, n, x, s8, block)
    assert np.abs(ctx.gemv(2, w8, rows, n, x, s8, block) - want).max() < 2e-5 * np.abs(want).max()


# 16 waves of 2 (F8), 1 (F16, F32) rows are a row set, up to 8 sets are taken at once: heads of fewer rows, of just as many and of more
@pytest.mark.parametrize("quant,nope,vd", [("f8e5m2", 128, 128), ("f8e5m2", 128, 256), ("fp16", 64, 64), ("fp16", 96, 64), ("fp32", 64, 64), ("fp32", 32, 160)])
def test_head_rows_over_row_sets(ctx, oracle, quant, nope, vd):
    check_head(ctx, oracle, quant, nope, vd)


# every number of sets at once (1, 2, 4, 6, 8), in one round and in more, the last set whole, ragged and past the head's end
@pytest.mark.parametrize("quant,nope,vd", [("f8e5m2", 16, 12), ("f8e5m2", 16, 16), ("f8e5m2", 20, 24), ("f8e5m2", 48, 48), ("f8e5m2", 64, 72), ("f8e5m2", 96, 96), ("f8e5m2", 112, 100),
                                           ("fp16", 8, 8), ("fp16", 64, 72), ("fp16", 96, 92), ("fp16", 128, 148), ("fp32", 8, 20), ("fp32", 40, 36), ("fp32", 96, 96)])
def test_head_rows_of_any_number_of_sets(ctx, oracle, quant, nope, vd):
    check_head(ctx, oracle, quant, nope, vd)


def check_head(ctx, oracle, quant, nope, vd):
    c = synth.preset("tiny_v2lite", quant, False, qk_nope_head_dim=nope, v_head_dim=vd, kv_lora_rank=512)
    T = synth.synth_model(c, seed=5)
    import dsk
    M, O = dsk.Model(ctx, c, T), oracle.model(c, T)
    for pos, t in enumerate((3, 14, 15, 92)):
        got, want = M.forward(t, pos), O.forward(t, pos)
        assert np.abs(got - want).max() < 1e-3 * np.abs(want).max(), pos
    M.close()
    O.close()
