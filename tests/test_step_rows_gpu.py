"""Rows of decoding steps: the residual sum of a sandwich layer shared by several workgroups (join_device.h)."""
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
