"""Backward blend as a training view reaches it, through render_gaussians_ex and render_gaussians_backward: with the
forward kernel's hit words, the order of the tiles it left, packed, caller-written or gathered operands and lists
launched ahead of their count.  At the list lengths where the kernel's steps change, and with upstream gradients that
are not finite, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


def scene(n, thin, seed):
    """n Gaussians around a 41 x 27 image (its last tiles are cut off), as preprocess_gaussians would hand them on."""
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=gen)
    W, Hh = 41, 27
    s1 = torch.exp(r(n) * 2.5)
    s2 = s1 * torch.where(r(n) < 0.5, 0.05, 0.6) if thin else s1 * (0.4 + 0.6 * r(n))
    s2 = torch.clamp(s2, min=0.55)
    ang = r(n) * 3.14159
    c, s = torch.cos(ang), torch.sin(ang)
    i1, i2 = 1 / s1 ** 2, 1 / s2 ** 2
    opac = r(n) * (0.9 if n < 100 else 0.08) + 0.01
    am = torch.randn(n, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0  # faces the camera: the plane depth stays well conditioned
    am[:, 3] = 1.0
    return dict(W=W, H=Hh, tan=0.5, means2D=r(n, 2) * torch.tensor([W + 8.0, Hh + 8.0]) - 4.0,
                co=torch.stack([c * c * i1 + s * s * i2, c * s * (i1 - i2), s * s * i1 + c * c * i2, opac], 1).float(),
                radii=torch.ceil(3 * s1).int(), depths=r(n) * 10 + 1, rgb=r(n, 3), am=am,
                bg=torch.tensor([0.3, 0.6, 0.1]),
                up=[torch.randn(k, Hh, W, generator=gen) for k in (3, 5, 1)])


def oracle_gradients(orc, v, cl, geo):
    n = {k: t.numpy() for k, t in v.items() if isinstance(t, torch.Tensor)}
    W, Hh, tan = v["W"], v["H"], v["tan"]
    b = orc.bin_and_sort(n["radii"], n["means2D"], n["depths"], cl.numpy().ravel(), W, Hh)
    f = orc.render_fwd(b["ranges"], b["point_list"], n["means2D"], n["rgb"], n["am"], n["co"], cl.numpy().ravel(),
                       n["bg"], W, Hh, tan, tan, render_geo=geo)
    g = orc.render_bwd(b["ranges"], b["point_list"], n["means2D"], n["co"], n["rgb"], n["am"], f["out_all_map"],
                       f["final_T"], f["n_contrib"], cl.numpy().ravel(), n["bg"], *[u.numpy() for u in v["up"]], W, Hh,
                       tan, tan, render_geo=geo)
    return b, f, [g["dL_dmeans2D"][:, :2], g["dL_dmeans2D_abs"], g["dL_dconic_opacity"], g["dL_dcolors"],
                  g["dL_dall_map"]]


def view(v, cl, geo, ahead=False, records=False):
    """(colour, gradients) of the view's two calls."""
    from diff_gaussian_rasterization import _C
    d = {k: t.to(DEV) for k, t in v.items() if isinstance(t, torch.Tensor)}
    n = d["means2D"].shape[0]
    rec = None
    if records:
        rec = torch.cat([d["means2D"], d["co"], d["rgb"], d["am"], d["depths"][:, None], torch.zeros(n, 1, device=DEV)],
                        1).contiguous()
    eye, args = torch.eye(4, device=DEV), {"stats_collector": {}}
    out, info = _C.render_gaussians_ex(d["bg"], v["H"], v["W"], d["means2D"], d["depths"], d["radii"], d["co"], d["rgb"],
                                       cl.to(DEV), eye, torch.zeros(3, device=DEV), v["tan"], v["tan"], d["am"], geo,
                                       False, args, expected_instances=50 * n + 100 if ahead else 0,
                                       expected_longest_list=0, blend_records=rec)
    assert info["launched_ahead"] == ahead
    color, oam, (geom, binning, img) = out[1], out[6], out[8:11]
    up = [u.to(DEV) for u in v["up"]]
    run = lambda: _C.render_gaussians_backward(d["bg"], v["tan"], v["tan"], oam, d["am"], out[0], geom, binning, img,
                                               cl.to(DEV), *up, d["means2D"], d["co"], d["rgb"], geo, False, args,
                                               binning_capacity=info["binning_capacity"], blend_records=rec)
    a, b = run(), run()
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    return color.cpu().numpy(), [x.cpu().numpy() for x in a]


def tiles(v):
    return torch.ones((v["H"] + 15) // 16, (v["W"] + 15) // 16, dtype=torch.bool)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 127, 128, 129, 256, 257, 700])
@pytest.mark.parametrize("thin,geo", [(False, True), (True, True), (True, False)])
def test_list_lengths(H, orc, n, thin, geo):
    v = scene(n, thin, seed=n)
    cl = tiles(v)
    b, f, want = oracle_gradients(orc, v, cl, geo)
    if n == 1:
        cl[0, 0] = False  # (a masked tile, whatever its list would hold)
        b, f, want = oracle_gradients(orc, v, cl, geo)
    first = None
    for ahead, records in ((False, False), (True, False), (False, True), (True, True)):
        color, got = view(v, cl, geo, ahead, records)
        assert np.array_equal(color, f["color"])
        # every route stages the same operands in the same order: the same bits
        if first is None:
            first = got
        for a, c in zip(first, got):
            assert np.array_equal(a, c)
    # At most 700 x 256 terms, added in another order: an error of sqrt(terms) * 2^-24 = 2.5e-5 of the sum of their
    # magnitudes if all fell on one Gaussian; a Gaussian's own terms are its pixels', at most 41 x 27 of them, whose
    # magnitudes add up to some ten times the sum: sqrt(1107) * 2^-24 * 10 = 2e-5.
    for k, a, w in zip(("means2D", "means2D_abs", "conic_opacity", "colors", "all_map"), first, want):
        if k == "all_map" and not geo:
            assert not a.any()
            continue
        assert H.rel_l2(a, w) <= 1e-4, (k, H.rel_l2(a, w))


@pytest.mark.parametrize("what", ["colour", "channel", "depth", "all"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("n,thin", [(40, False), (300, False), (300, True)])
def test_upstream_gradients_that_are_not_finite(H, orc, what, value, n, thin):
    """They reach the Gaussians that the pixel blended and no other, as in the reference, which adds nothing for the
    rest (cuda_rasterizer/backward.cu:463-563); everything else stays what it is without them."""
    v = scene(n, thin, seed=1000 + n)
    cl = tiles(v)
    for y, x in ((3, 5), (3, 6), (20, 33), (26, 40)):
        if what in ("colour", "all"):
            v["up"][0][1, y, x] = value
        if what in ("channel", "all"):
            v["up"][1][0, y, x] = value
        if what in ("depth", "all"):
            v["up"][2][0, y, x] = value
    b, f, want = oracle_gradients(orc, v, cl, True)
    _, got = view(v, cl, True)
    dev = lambda a: H.dev(a)
    tile_entry = H.render_bwd(n, v["W"], v["H"], v["tan"], v["tan"], dev(v["bg"].numpy()), H.as_u32(b["ranges"]),
                              H.as_u32(b["point_list"]), *[dev(v[k].numpy()) for k in ("means2D", "co", "rgb", "am")],
                              dev(f["out_all_map"]), dev(f["final_T"]), H.as_u32(f["n_contrib"]),
                              dev(cl.numpy().ravel()), *[dev(u.numpy()) for u in v["up"]],
                              H.as_u32(b["emission_sorted"]), H.as_u32(b["point_offsets"]))
    hit = 0
    for k, a, w in zip(("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity", "dL_dcolors", "dL_dall_map"), got, want):
        for x in (a, tile_entry[k].cpu().numpy()):
            bad = ~np.isfinite(w)
            assert np.array_equal(~np.isfinite(x), bad), k
            hit += int(bad.sum())
            assert H.rel_l2(x[~bad], w[~bad]) <= 1e-4, k  # (the bound of the test above)
    assert 0 < hit
