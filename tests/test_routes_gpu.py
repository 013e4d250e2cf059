"""The router's choice for many rows (kernels_join.hip route_count_kernel, route_sort_kernel) against the plain statement, in 32 bits."""
import numpy as np
import pytest

from tests import layered_util as U

pytestmark = pytest.mark.gpu


# rows around whole workgroups of 16, counts of experts around whole waves up to the most, as many choices as a workgroup's slots hold, no shared expert
@pytest.mark.parametrize("experts,top,shared,n", [(7, 3, 72, 17), (64, 6, 72, 40), (65, 5, 0, 33), (128, 2, 0, 31), (130, 63, 72, 21), (512, 8, 72, 300), (512, 1, 0, 48)])
def test_rows_and_experts(case, experts, top, shared, n):
    case(U.config([U.channel_delta(mlp=U.moe(experts, top, shared=shared)), U.channel_delta(mlp=U.moe(5, 5))], width=64)).check_trace(n, cuts=([n - 17],))


@pytest.mark.parametrize("kind", ["all equal", "pairs", "zeros of both signs"])
def test_equal_logits_go_to_the_lowest_index(case, kind):
    def edit(W):
        for k in W:
            if k.endswith("router"):
                if kind == "pairs":
                    W[k][1::2] = W[k][0::2]
                else:
                    W[k][:] = 0
                    if kind != "all equal":
                        W[k][::3] = -0.0
    case(U.config([U.channel_delta(mlp=U.moe(70, 5))], width=64), edit=edit).check_trace(37, cuts=([20],))


# passes whose counts are summed by a launch of their own (workgroups of 16 rows, squared, times experts > 2^24): around that line, several of 64 runs empty, whole and
# broken ones, experts that are no whole workgroups of 16
@pytest.mark.parametrize("experts,top,shared,n", [(512, 2, 0, 2896), (512, 2, 0, 2897), (509, 3, 72, 3001), (130, 5, 0, 5900), (256, 8, 72, 8192)])
def test_long_passes(case, experts, top, shared, n):
    mixer = U.delta(heads=1, kv_heads=1, dim=16, vdim=16)
    m = case(U.config([U.channel_delta(mixer, mlp=U.moe(experts, top, ff=16, shared=shared))], width=64), options="piece_tokens=8192")
    assert m.lm.info("piece_tokens") == 8192
    m.check_trace(n)
