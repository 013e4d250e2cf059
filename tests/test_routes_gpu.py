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
