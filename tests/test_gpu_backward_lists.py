"""Backward blend by itself (the entry point that is handed finished lists and neither hit words nor an order of the
tiles; tests/test_gpu_backward_view.py has the whole view) at the list lengths where its steps change: four entries per
pass, 56 slots per wave without the geometry channels and 64 with them, windows and scans of 256 positions, runs of 64;
with and without thin Gaussians (whose sums keep a fixed order), on an image whose last tiles are cut off, against the
oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


@pytest.mark.parametrize("n", [1, 3, 4, 5, 55, 56, 57, 63, 64, 65, 111, 112, 113, 127, 128, 129, 256, 257, 700])
@pytest.mark.parametrize("thin,geo", [(False, True), (True, True), (True, False)])
def test_list_lengths(H, orc, n, thin, geo):
    gen = torch.Generator().manual_seed(n)
    r = lambda *s: torch.rand(*s, generator=gen)
    W, Hh, tan = 41, 27, 0.5
    means2D = (r(n, 2) * torch.tensor([W + 8.0, Hh + 8.0]) - 4.0).numpy()
    s1 = torch.exp(r(n) * 2.5)
    s2 = s1 * torch.where(r(n) < 0.5, 0.05, 0.6) if thin else s1 * (0.4 + 0.6 * r(n))
    s2 = torch.clamp(s2, min=0.55)
    ang = r(n) * 3.14159
    c, s = torch.cos(ang), torch.sin(ang)
    i1, i2 = 1 / s1 ** 2, 1 / s2 ** 2
    opac = r(n) * (0.9 if n < 100 else 0.08) + 0.01
    co = torch.stack([c * c * i1 + s * s * i2, c * s * (i1 - i2), s * s * i1 + c * c * i2, opac], 1).float().numpy()
    radii = torch.ceil(3 * s1).int().numpy()
    depths = (r(n) * 10 + 1).numpy()
    rgb = r(n, 3).numpy()
    am = torch.randn(n, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0  # faces the camera: the plane depth stays well conditioned
    am[:, 3] = 1.0
    am = am.numpy()
    gx, gy = H.grid(W, Hh)
    cl = np.ones(gx * gy, bool)
    bg = np.array([0.3, 0.6, 0.1], np.float32)
    b = orc.bin_and_sort(radii, means2D, depths, cl, W, Hh)
    f = orc.render_fwd(b["ranges"], b["point_list"], means2D, rgb, am, co, cl, bg, W, Hh, tan, tan, render_geo=geo)
    gpix, gmap, gdep = (torch.randn(k, Hh, W, generator=gen).numpy() for k in (3, 5, 1))
    ref = orc.render_bwd(b["ranges"], b["point_list"], means2D, co, rgb, am, f["out_all_map"], f["final_T"],
                         f["n_contrib"], cl, bg, gpix, gmap, gdep, W, Hh, tan, tan, render_geo=geo)

    def run():
        return H.render_bwd(n, W, Hh, tan, tan, H.dev(bg), H.as_u32(b["ranges"]), H.as_u32(b["point_list"]),
                            H.dev(means2D), H.dev(co), H.dev(rgb), H.dev(am), H.dev(f["out_all_map"]),
                            H.dev(f["final_T"]), H.as_u32(f["n_contrib"]), H.dev(cl), H.dev(gpix), H.dev(gmap),
                            H.dev(gdep), H.as_u32(b["emission_sorted"]), H.as_u32(b["point_offsets"]), render_geo=geo)

    got, again = run(), run()
    # 24-bit sums in another order: about sqrt(terms) * 2^-24 of the sum of magnitudes, which is some ten times the sum
    # itself.  A Gaussian's terms are its pixels', at most 41 x 27 of them: sqrt(1107) * 2^-24 * 10 = 2e-5.
    for k, want in (("dL_dmeans2D", ref["dL_dmeans2D"][:, :2]), ("dL_dmeans2D_abs", ref["dL_dmeans2D_abs"]),
                    ("dL_dconic_opacity", ref["dL_dconic_opacity"]), ("dL_dcolors", ref["dL_dcolors"]),
                    ("dL_dall_map", ref["dL_dall_map"])):
        if k == "dL_dall_map" and not geo:
            continue
        assert torch.equal(got[k], again[k]), k
        assert H.rel_l2(got[k].cpu().numpy(), want) <= 1e-4, (k, H.rel_l2(got[k].cpu().numpy(), want))


def _covering_view(H, orc, n, small):
    """Gaussians that cover the whole image, three in ten of them thin: every wave stages every entry, so the windows end at
    the waves' slots (56 or 64), and a run of 64 positions spans two of them.  small: so many of a pixel's size among them,
    that touch one row or two, so that the rows' lists are of different lengths where a run is carried on."""
    gen = torch.Generator().manual_seed(1000 + n)
    r = lambda *s: torch.rand(*s, generator=gen)
    W, Hh, tan = 33, 17, 0.5
    means2D = (r(n, 2) * torch.tensor([float(W), float(Hh)])).numpy()
    thin = r(n) < 0.3
    s1 = (40.0 + 20.0 * r(n)) * torch.where(thin, 10.0, 1.0)
    s2 = s1 * torch.where(thin, 0.1, 0.8)
    ang = torch.where(thin, 0.5 + 0.5 * r(n), r(n) * 3.14159)
    tiny = r(n) < small
    s1, s2 = torch.where(tiny, 0.6, s1), torch.where(tiny, 0.55, s2)
    c, s = torch.cos(ang), torch.sin(ang)
    i1, i2 = 1 / s1 ** 2, 1 / s2 ** 2
    co = torch.stack([c * c * i1 + s * s * i2, c * s * (i1 - i2), s * s * i1 + c * c * i2, 0.01 + 0.01 * r(n)],
                     1).float().numpy()
    is_thin = co[:, 1] ** 2 >= 0.8 * co[:, 0] * co[:, 2]  # (the kernel's own test)
    assert is_thin.sum() > n // 8 and not is_thin[tiny.numpy()].any() and tiny.sum() >= n * small / 2
    radii, depths, rgb = torch.ceil(3 * s1).int().numpy(), (r(n) * 10 + 1).numpy(), r(n, 3).numpy()
    am = torch.randn(n, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0
    am = am.numpy()
    gx, gy = H.grid(W, Hh)
    cl = np.ones(gx * gy, bool)
    bg = np.array([0.3, 0.6, 0.1], np.float32)
    b = orc.bin_and_sort(radii, means2D, depths, cl, W, Hh)
    f = orc.render_fwd(b["ranges"], b["point_list"], means2D, rgb, am, co, cl, bg, W, Hh, tan, tan, render_geo=True)
    assert f["n_contrib2loss"].min() == (~tiny).sum()  # (they do cover it, every pixel)
    gpix, gmap, gdep = (torch.randn(k, Hh, W, generator=gen).numpy() for k in (3, 5, 1))

    def reference(geo):
        return orc.render_bwd(b["ranges"], b["point_list"], means2D, co, rgb, am, f["out_all_map"], f["final_T"],
                              f["n_contrib"], cl, bg, gpix, gmap, gdep, W, Hh, tan, tan, render_geo=geo)

    def run(geo, map_scale=1.0):
        return H.render_bwd(n, W, Hh, tan, tan, H.dev(bg), H.as_u32(b["ranges"]), H.as_u32(b["point_list"]),
                            H.dev(means2D), H.dev(co), H.dev(rgb), H.dev(am), H.dev(f["out_all_map"]),
                            H.dev(f["final_T"]), H.as_u32(f["n_contrib"]), H.dev(cl), H.dev(gpix),
                            H.dev(gmap * np.float32(map_scale)), H.dev(gdep * np.float32(map_scale)),
                            H.as_u32(b["emission_sorted"]), H.as_u32(b["point_offsets"]), render_geo=geo)

    return run, reference, is_thin


@pytest.mark.parametrize("n", [55, 56, 57, 63, 64, 65, 112, 113, 255, 256, 257, 321])
@pytest.mark.parametrize("geo", [True, False])
@pytest.mark.parametrize("small", [0.0, 0.3])
def test_every_wave_needs_every_slot(H, orc, n, geo, small):
    run, reference, _ = _covering_view(H, orc, n, small)
    got, again, ref = run(geo), run(geo), reference(geo)
    # the bound of the test above (561 pixels here)
    for k, want in (("dL_dmeans2D", ref["dL_dmeans2D"][:, :2]), ("dL_dmeans2D_abs", ref["dL_dmeans2D_abs"]),
                    ("dL_dconic_opacity", ref["dL_dconic_opacity"]), ("dL_dcolors", ref["dL_dcolors"]),
                    ("dL_dall_map", ref["dL_dall_map"])):
        if k != "dL_dall_map" or geo:
            assert torch.equal(got[k], again[k]), k
            assert H.rel_l2(got[k].cpu().numpy(), want) <= 1e-4, (k, H.rel_l2(got[k].cpu().numpy(), want))


@pytest.mark.parametrize("n", [57, 65, 113, 129, 257, 321])
@pytest.mark.parametrize("small", [0.0, 0.3])
def test_the_order_of_thin_gaussians_sums_does_not_depend_on_the_windows(H, orc, n, small):
    # With no gradients of the channels the kernels with 64 and with 56 slots per wave add the same terms, in windows that
    # end at different places.
    run, _, is_thin = _covering_view(H, orc, n, small)
    a, b = run(True, 0.0), run(False, 0.0)
    thin = torch.from_numpy(is_thin).to(H.DEV)
    for k in ("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity"):
        assert a[k][thin].abs().amax() > 0.0 and torch.equal(a[k][thin], b[k][thin]), k


@pytest.mark.parametrize("P", [1_499_999, 1_500_000, 1_500_001, 1_500_063])
@pytest.mark.parametrize("geo", [True, False])
def test_results_of_a_large_view_are_streamed(H, orc, P, geo):
    """From 1.5 M Gaussians on the sums over a Gaussian's instances leave past the caches and turned through LDS, the last
    wave partly filled.  A small view's Gaussians, half of them at the start and half at the end of a large view that has
    nothing between them: the same bits, and zeros for everybody else."""
    n, half = 300, 150
    gen = torch.Generator().manual_seed(3)
    r = lambda *s: torch.rand(*s, generator=gen)
    W, Hh, tan = 41, 27, 0.5
    means2D = (r(n, 2) * torch.tensor([W + 8.0, Hh + 8.0]) - 4.0).numpy()
    s1 = torch.exp(r(n) * 2.5)
    i1 = 1 / s1 ** 2
    co = torch.stack([i1, torch.zeros(n), i1, r(n) * 0.1 + 0.01], 1).float().numpy()
    radii = torch.ceil(3 * s1).int().numpy()
    depths, rgb = (r(n) * 10 + 1).numpy(), r(n, 3).numpy()
    am = torch.randn(n, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0
    am[:, 3] = 1.0
    am = am.numpy()
    gx, gy = H.grid(W, Hh)
    cl = np.ones(gx * gy, bool)
    bg = np.array([0.3, 0.6, 0.1], np.float32)
    b = orc.bin_and_sort(radii, means2D, depths, cl, W, Hh)
    f = orc.render_fwd(b["ranges"], b["point_list"], means2D, rgb, am, co, cl, bg, W, Hh, tan, tan, render_geo=geo)
    gpix, gmap, gdep = (torch.randn(k, Hh, W, generator=gen).numpy() for k in (3, 5, 1))

    def run(count, place, point_offsets):
        def spread(a):
            out = np.zeros((count,) + a.shape[1:], a.dtype)
            out[place] = a
            return H.dev(out)
        point_list = place.astype(np.uint32)[b["point_list"].astype(np.int64)]
        return H.render_bwd(count, W, Hh, tan, tan, H.dev(bg), H.as_u32(b["ranges"]), H.as_u32(point_list),
                            spread(means2D), spread(co), spread(rgb), spread(am), H.dev(f["out_all_map"]),
                            H.dev(f["final_T"]), H.as_u32(f["n_contrib"]), H.dev(cl), H.dev(gpix), H.dev(gmap),
                            H.dev(gdep), H.as_u32(b["emission_sorted"]), H.as_u32(point_offsets), render_geo=geo)

    offsets = np.asarray(b["point_offsets"])
    small = run(n, np.arange(n), offsets)
    place = np.concatenate([np.arange(half), np.arange(P - (n - half), P)])
    large = run(P, place, np.concatenate([offsets[:half], np.full(P - n, offsets[half - 1], offsets.dtype), offsets[half:]]))
    index = torch.from_numpy(place).cuda()
    for k in ("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity", "dL_dcolors", "dL_dall_map"):
        assert large[k].shape[0] == P
        assert torch.equal(large[k][index], small[k]), k
        assert not large[k][half:P - (n - half)].any(), k


# With the geometry channels a wave has 60 slots: windows that hold one Gaussian less, as many and one more.  (With three in
# ten of them small, 59 and 61 are not the view that _covering_view wants.)
@pytest.mark.parametrize("n,small", [(59, 0.0), (60, 0.0), (61, 0.0), (58, 0.3), (60, 0.3), (62, 0.3), (119, 0.3), (120, 0.0),
                                     (120, 0.3), (121, 0.3), (181, 0.3)])
def test_sixty_slots(H, orc, n, small):
    run, reference, is_thin = _covering_view(H, orc, n, small)
    got, ref = run(True), reference(True)
    # the bound of test_list_lengths (561 pixels here)
    for k, want in (("dL_dmeans2D", ref["dL_dmeans2D"][:, :2]), ("dL_dmeans2D_abs", ref["dL_dmeans2D_abs"]),
                    ("dL_dconic_opacity", ref["dL_dconic_opacity"]), ("dL_dcolors", ref["dL_dcolors"]),
                    ("dL_dall_map", ref["dL_dall_map"])):
        assert H.rel_l2(got[k].cpu().numpy(), want) <= 1e-4, (k, H.rel_l2(got[k].cpu().numpy(), want))
    a, b = run(True, 0.0), run(False, 0.0)
    thin = torch.from_numpy(is_thin).to(H.DEV)
    for k in ("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity"):
        assert torch.equal(a[k][thin], b[k][thin]), k
