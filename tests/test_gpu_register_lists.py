"""The register sort with eight keys a lane: lists of 2049 to 4096 entries, filled exactly, one short and one over."""
import pytest

import test_gpu_tile_lists as lists

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


@pytest.mark.parametrize("order", ["random", "falling", "equal"])
@pytest.mark.parametrize("P", [2049, 2560, 3583, 3584, 3585, 4095, 4096, 4097])
def test_list_lengths(orc, H, P, order):
    lists.test_list_lengths_at_the_edges_of_the_register_sort(orc, H, P, order)


@pytest.mark.parametrize("P", [2049, 4096])
def test_depths_that_agree_in_their_leading_bits(orc, H, P):
    lists.test_depths_that_agree_in_their_leading_bits(orc, H, P)
