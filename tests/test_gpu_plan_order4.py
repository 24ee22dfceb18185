"""The coordinates given to a plan of order 4 only order its parts, as test_gpu_plan_order checks for orders 1-3: owner-only
plans, whose parts follow a curve through the nodes, and the others, through the elements."""

import pytest

from test_gpu_plan_order import test_ordering_coordinates as check_ordering

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["default", "deterministic", "residual", "owner"])
def test_order_4(fem, orc, torch_gpu, kind):
    check_ordering(fem, orc, torch_gpu, 4, 9, 8, kind)
