"""Lists of more entries than one workgroup of the per-tile radix sort holds: split by depth into groups first.  One tile, so
that the list is the Gaussians in the order of (depth bits, index)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def depths(kind, n, gen):
    if kind == "even":
        d = torch.rand(n, generator=gen) * 30 + 1
    elif kind == "equal":  # one group, and runs as long as the list
        d = torch.full((n,), 2.5)
    elif kind == "few":  # groups beyond a block
        d = torch.randint(1, 4, (n,), generator=gen).float()
    elif kind == "heavy":  # most of the list within a small part of the range
        d = torch.where(torch.rand(n, generator=gen) < 0.9, 5 + torch.rand(n, generator=gen) * 1e-3,
                        1 + torch.rand(n, generator=gen) * 1e3)
    else:  # "outliers": nearer and farther than anything that a sample of the list is likely to hold
        d = torch.rand(n, generator=gen) * 30 + 5
        d[n // 3 + 1], d[n // 2 + 1], d[n // 2 + 3] = 0.3, 1e30, 1e30
    return d


# 16384 records are sorted whole; 16385 are split; 140 000: a dozen groups; a block of 300 records: up to 64 groups, the
# last of them beyond a block
@pytest.mark.parametrize("kind", ["even", "equal", "few", "heavy", "outliers"])
@pytest.mark.parametrize("n,limits", [(16384, None), (16385, None), (20481, None), (140_000, None), (4097, (-1, 300)),
                                      (33_000, (-1, 300)), (9, (7, 7)), (65, (40, 64)), (5000, (100, 4096))])
def test_order_of_a_split_list(kind, n, limits):
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    if kind == "equal" and n > 40_000:
        n = 17_000  # (a run of L entries costs L reads an entry)
    if kind == "few" and n > 40_000:
        n = 40_000
    gen = torch.Generator().manual_seed(n)
    d = depths(kind, n, gen)
    W = H = 16
    m2 = (torch.rand(n, 2, generator=gen) * 15.9).to(DEV)
    co = torch.tensor([[0.5, 0.0, 0.5, 0.3]]).repeat(n, 1).to(DEV)
    args = {"stats_collector": {}}
    if limits is not None:
        args["tile_sort_limits"] = limits
    out = _C.render_gaussians(torch.zeros(3, device=DEV), H, W, m2, d.to(DEV),
                              torch.ones(n, dtype=torch.int32, device=DEV), co, torch.rand(n, 3, generator=gen).to(DEV),
                              torch.ones(1, 1, dtype=torch.bool, device=DEV), torch.eye(4, device=DEV),
                              torch.zeros(3, device=DEV), 0.5, 0.5, None, False, False, args)
    R, binning = out[0], out[9]
    assert R == n
    off = [C.c_size_t() for _ in range(5)]
    gn.check(gn.lib.gs_binning_state_layout(R, W, H, *[C.byref(x) for x in off]), "layout")
    base = (binning.data_ptr() + 255) // 256 * 256 - binning.data_ptr()
    point_list = binning[base + off[0].value: base + off[0].value + 4 * R].view(torch.int32).cpu().numpy()
    keys = binning[base + off[1].value: base + off[1].value + 8 * R].view(torch.int64).cpu().numpy()
    bits = d.numpy().view(np.uint32).astype(np.int64)
    want = np.argsort(bits, kind="stable")
    assert np.array_equal(point_list, want)
    assert np.array_equal(keys, bits[want])  # (tile 0)


# Several lists in one view, whose groups are jobs for the same workgroups: lists of one to a dozen groups (and of 64 with a
# block of 300 records), beside lists that are sorted whole, in registers, or empty.  300 tiles: as many workgroups as tiles;
# fewer than 256: up to 64 workgroups a tile.
@pytest.mark.parametrize("gx,gy,sizes,limits", [
    (3, 2, (20_000, 70_000, 17_000, 16_384, 4097, 100), None), (3, 2, (0, 16_385, 0, 140_000, 0, 33_000), None),
    (2, 1, (17_000, 70_000), None), (3, 2, (4097, 33_000, 5000, 300, 301, 0), (-1, 300)),
    (3, 2, (9, 8, 70, 500, 7, 64), (7, 7)), (20, 15, (17_000, 5000, 41_000) + (300,) * 297, None)])
@pytest.mark.parametrize("ahead", [False, True])
def test_order_of_several_split_lists(gx, gy, sizes, limits, ahead):
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    gen = torch.Generator().manual_seed(sum(sizes))
    W, H, n = 16 * gx, 16 * gy, sum(sizes)
    tile = torch.repeat_interleave(torch.arange(gx * gy), torch.tensor(sizes))
    d = torch.cat([depths(("even", "heavy", "outliers")[i % 3], k, gen) if k > 8 else torch.rand(k, generator=gen) + 1
                   for i, k in enumerate(sizes)])
    mix = torch.randperm(n, generator=gen)  # (a list's Gaussians lie anywhere)
    tile, d = tile[mix], d[mix]
    m2 = torch.stack([(tile % gx) * 16.0, (tile // gx) * 16.0], 1) + 3 + torch.rand(n, 2, generator=gen) * 9
    co = torch.tensor([[0.5, 0.0, 0.5, 0.3]]).repeat(n, 1).to(DEV)
    args = {"stats_collector": {}}
    if limits is not None:
        args["tile_sort_limits"] = limits
    out, info = _C.render_gaussians_ex(torch.zeros(3, device=DEV), H, W, m2.to(DEV), d.to(DEV),
                                       torch.full((n,), 2, dtype=torch.int32, device=DEV), co,
                                       torch.rand(n, 3, generator=gen).to(DEV),
                                       torch.ones(gy, gx, dtype=torch.bool, device=DEV), torch.eye(4, device=DEV),
                                       torch.zeros(3, device=DEV), 0.5, 0.5, None, False, False, args,
                                       expected_instances=n + 5 if ahead else 0)
    assert out[0] == n and info["launched_ahead"] == ahead and info["longest_list"] == max(sizes)
    capacity = info["binning_capacity"]
    off = [C.c_size_t() for _ in range(5)]
    gn.check(gn.lib.gs_binning_state_layout(capacity, W, H, *[C.byref(x) for x in off]), "layout")
    binning = out[9]
    base = -binning.data_ptr() % 256
    point_list = binning[base + off[0].value: base + off[0].value + 4 * n].view(torch.int32).cpu().numpy()
    keys = binning[base + off[1].value: base + off[1].value + 8 * n].view(torch.int64).cpu().numpy()
    key = tile.numpy().astype(np.int64) << 32 | d.numpy().view(np.uint32).astype(np.int64)
    want = np.argsort(key, kind="stable")
    assert np.array_equal(point_list, want)
    assert np.array_equal(keys, key[want])
