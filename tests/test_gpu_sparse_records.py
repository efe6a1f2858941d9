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


# 3.5 Gaussians a pixel is where records are left out: 3875 at 41 x 27.  scale 4: a 164 x 108 image of 77 tiles, with Gaussians
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
