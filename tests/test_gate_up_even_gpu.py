"""gate_up of one row of int8 weights in workgroups of four and of three blocks (csrc/norm_product.hip): the first and the last width that has both, the widths beside
them and widths that are left to workgroups of four, bit for bit the calls that it replaces."""
import pytest

from tests.test_norm_product_gpu import test_norm_product_gives_the_bits_of_the_calls_it_replaces as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,sk", [(24576, 2048, 1), (24704, 2048, 1), (24832, 4096, 4), (32640, 3072, 4), (32768, 2048, 2), (28672, 2048, 1), (28672, 3072, 4), (28800, 3072, 2)])
def test_widths(N, H, sk):
    check(2, 1, N, H, sk, True)
