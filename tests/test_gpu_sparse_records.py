"""Backward blend of views with many Gaussians per pixel, whose instances without a blended pixel have no record: against
the oracle, and bit for bit against the stage entry point, which writes every record."""
import numpy as np
import pytest
import torch

from test_gpu_backward_view import DEV, oracle_gradients, scene, tiles, view

pytestmark = pytest.mark.gpu

NAMES = ("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity", "dL_dcolors", "dL_dall_map")


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


# Every view here has more than two instances a pixel.  scale 4: a 164 x 108 image of 77 tiles, with Gaussians
# of more than 32 instances, which a whole wave sums, and runs of more than 64 records for one wave.
@pytest.mark.parametrize("n,scale,masked", [(3874, 1, False), (3875, 1, False), (3875, 1, True), (9000, 1, False),
                                            (62_100, 4, False)])
@pytest.mark.parametrize("geo", [True, False])
def test_gradients(H, orc, n, scale, masked, geo):
    v = scene(n, True, seed=n + scale)
    gen = torch.Generator().manual_seed(n)
    if scale > 1:
        v["W"], v["H"] = 41 * scale, 27 * scale
        v["means2D"] = v["means2D"] * scale
        v["up"] = [torch.randn(k, v["H"], v["W"], generator=gen) for k in (3, 5, 1)]
        v["radii"][::997] = 130  # (rectangles of 33 tiles and more)
    v["co"][:, 3] = 0.05 + 0.9 * torch.rand(n, generator=gen)  # opaque: most instances lie behind the last blended one
    cl = tiles(v)
    if masked:
        cl[0, 1] = False
    b, f, want = oracle_gradients(orc, v, cl, geo)
    dev = lambda a: H.dev(a)
    dense = H.render_bwd(n, v["W"], v["H"], v["tan"], v["tan"], dev(v["bg"].numpy()), H.as_u32(b["ranges"]),
                         H.as_u32(b["point_list"]), *[dev(v[k].numpy()) for k in ("means2D", "co", "rgb", "am")],
                         dev(f["out_all_map"]), dev(f["final_T"]), H.as_u32(f["n_contrib"]), dev(cl.numpy().ravel()),
                         *[dev(u.numpy()) for u in v["up"]], H.as_u32(b["emission_sorted"]),
                         H.as_u32(b["point_offsets"]), **({} if geo else {"render_geo": False}))
    junk = torch.full((1 << 24,), float("nan"), device=DEV)  # (what the scratch memory may hold)
    del junk
    _, got = view(v, cl, geo)
    blended = 0
    for k, a, w in zip(NAMES, got, want):
        if k == "dL_dall_map" and not geo:
            assert not a.any()
            continue
        assert np.array_equal(a.view(np.int32), dense[k].cpu().numpy().view(np.int32)), k
        # A Gaussian's terms are its pixels', 17 712 at most, whose magnitudes add up to some ten times the sum:
        # sqrt(17712) * 2^-24 * 10 = 8e-5.
        assert H.rel_l2(a, w) <= 1e-4, (k, H.rel_l2(a, w))
        blended = max(blended, int(a.any(axis=1).sum()))
    assert 0 < blended < n // 2


# Two instances a pixel is where the records are left out: 6144 at 64 x 48.  What lies out of view does not count, nor does the
# number of Gaussians: 520 of them that are in every one of twelve tiles have enough.
@pytest.mark.parametrize("single,unseen,everywhere,sparse", [(6143, 0, 0, False), (6144, 0, 0, True), (6143, 20_000, 0, False),
                                                             (900, 40_000, 300, False), (0, 0, 511, False),
                                                             (0, 0, 520, True), (6132, 100, 1, True)])
def test_which_views_have_only_the_records_they_blend(single, unseen, everywhere, sparse):
    import ctypes as C
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    W, Hh, n = 64, 48, single + everywhere + unseen
    gen = torch.Generator().manual_seed(n)
    r = lambda *s: torch.rand(*s, generator=gen)
    radii = torch.full((n,), 2, dtype=torch.int32)
    radii[single:single + everywhere] = 300
    radii[single + everywhere:] = 0
    # (single tiles: centres three pixels and more from the tile's edges, radius 2)
    m2 = ((r(n, 2) * torch.tensor([4.0, 3.0])).floor() * 16 + 3 + r(n, 2) * 9).to(DEV)
    co = torch.stack([0.2 + r(n), r(n) * 0.1, 0.2 + r(n), 0.05 + 0.9 * r(n)], 1).to(DEV)
    depths, rgb, radii = (r(n) * 10 + 1).to(DEV), r(n, 3).to(DEV), radii.to(DEV)
    cl, zero3, args = torch.ones(3, 4, dtype=torch.bool, device=DEV), torch.zeros(3, device=DEV), {"stats_collector": {}}
    out = _C.render_gaussians(zero3, Hh, W, m2, depths, radii, co, rgb, cl, torch.eye(4, device=DEV), zero3, 0.5, 0.5, None,
                              False, False, args)
    R = out[0]
    assert R == single + 12 * everywhere and (R >= 2 * W * Hh) == sparse
    up = torch.randn(3, Hh, W, generator=gen).to(DEV)
    p = lambda t: C.c_void_p(t.data_ptr())

    def backward(size):
        grads = [torch.full((n, k), float("nan"), device=DEV) for k in (2, 3, 4, 3, 5)]
        ws = torch.full((size,), 0xAB, dtype=torch.uint8, device=DEV)
        gn.check(gn.lib.gs_render_backward(n, R, p(zero3), W, Hh, 0.5, 0.5, p(out[8]), p(out[9]), p(out[10]), p(cl), p(up), None,
                                           None, *[p(g) for g in grads], p(m2), p(co), p(rgb), None, None, 0, 0, p(ws), size,
                                           None, 0, None, C.c_void_p(torch.cuda.current_stream().cuda_stream)), "backward")
        flags = -ws.data_ptr() % 256 + 64 * R
        return grads, ws[flags:flags + R].cpu()

    dense, _ = backward(gn.lib.gs_render_backward_workspace_bytes(R))
    grads, flags = backward(gn.lib.gs_render_backward_sparse_workspace_bytes(R))
    assert bool((flags <= 1).all()) if sparse else bool((flags == 0xAB).all())
    assert not sparse or 0 < int(flags.sum()) < R
    for a, b in zip(grads, dense):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
