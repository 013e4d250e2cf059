"""Products of prompts at the edges of their tiles (kernels_lin.hip), against the plain statement of the design (oracle/layered.py)."""
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import dsk
    c = dsk.Ctx(0)
    yield c
    c.close()


# 32-bit activations are multiplied in three bf16 pieces.  Two pieces alone would be up to 2^-16 off; 32-bit sums, through the model's four
# products and a softmax, stay under a quarter of that (v_mfma_f32_16x16x4_f32 gave up to 2.2e-6 here, this gives up to 2.1e-6).
@pytest.mark.parametrize("width", [64, 328, 1000])
def test_32_bit_products_keep_32_bits(ctx, tmp_path, width):
    K = U.Case(ctx, tmp_path, U.sandwich([U.no_ff(U.latent())], width=width), dtype="float32")
    t = K.tokens(140)
    assert U.err(K.got(t), K.want(t)) < 2.0 ** -18
