"""The carry-out on both sides of the line between its orders (all pairs compared,
two sorts) and at one workgroup's thread count, against the reference's loop."""
import pytest

from test_gpu_carry_out import test_carry_out as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [383, 384, 385, 512, 1023])
def test_order_edges(usap, B):
    _check(usap, B)
