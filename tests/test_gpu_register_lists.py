"""The register sort with eight keys a lane: lists of 2049 to 4096 entries, filled exactly, one short and one over; and views
whose lists take every number of keys a lane at once, with and without such long ones.  The same views with the register
sort's limit lowered, where the smaller kernel of the per-tile radix sort has what lies between the limit and 4096."""
import ctypes as C

import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("longest", [2048, 2049, 4096, 4097])
@pytest.mark.parametrize("bound,limits", [(None, None), (2048, None), (4096, None), (0, None), (None, (2048, 0)),
                                          (None, (256, 0)), (None, (1500, 0)), (0, (2048, 0))])
def test_lists_of_every_class_in_one_view(orc, H, longest, bound, limits):
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    lengths = [1, 64, 256, 257, 512, 0, 513, 1024, 1025, longest - 1, longest, 3]
    W, Hh = 16 * len(lengths), 16
    gen = torch.Generator().manual_seed(longest)
    tile = torch.repeat_interleave(torch.arange(len(lengths)), torch.tensor(lengths))
    tile = tile[torch.randperm(len(tile), generator=gen)]
    P = len(tile)
    means2D = torch.stack([tile * 16 + 8.0, torch.full((P,), 8.0)], 1)  # (radius 1: that tile and no other)
    radii = torch.ones(P, dtype=torch.int32)
    depths = torch.rand(P, generator=gen) * 50.0 + 0.25
    cl = torch.ones(1, len(lengths), dtype=torch.bool)
    n = lambda t: t.numpy()
    want = orc.bin_and_sort(n(radii), n(means2D), n(depths), n(cl).reshape(-1), W, Hh)
    assert (np.diff(want["ranges"].reshape(-1, 2).astype(np.int64)).ravel() == lengths).all()
    co = torch.tensor([0.02, 0.0, 0.02, 0.3]).repeat(P, 1).to(lists.DEV)
    dev = lambda t: t.to(lists.DEV)
    out, info = _C.render_gaussians_ex(
        torch.zeros(3, device=lists.DEV), Hh, W, dev(means2D), dev(depths), dev(radii), co,
        torch.zeros(P, 3, device=lists.DEV), dev(cl), torch.eye(4, device=lists.DEV), torch.zeros(3, device=lists.DEV), 1.0,
        1.0, torch.zeros(P, 5, device=lists.DEV), False, False, {"stats_collector": {}, "tile_sort_limits": limits},
        expected_instances=0 if bound is None else P + 100, expected_longest_list=bound or 0)
    assert out[0] == P and info["launched_ahead"] == (bound is not None and (bound == 0 or longest <= bound))
    binB = out[9]
    off = [C.c_size_t() for _ in range(5)]
    gn.check(gn.lib.gs_binning_state_layout(info["binning_capacity"], W, Hh, *[C.byref(x) for x in off]), "layout")
    b0 = (binB.data_ptr() + 255) // 256 * 256 - binB.data_ptr()
    assert np.array_equal(H.np_u32(binB[b0 + off[0].value: b0 + off[0].value + 4 * P].view(torch.int32)), want["point_list"])
    assert np.array_equal(H.np_u64(binB[b0 + off[1].value: b0 + off[1].value + 8 * P].view(torch.int64)), want["keys"])
