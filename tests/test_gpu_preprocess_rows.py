"""The rows of colours and clamping flags that the forward preprocess kernel stores as whole words per wave: numbers of
Gaussians around its waves and workgroups, flags that start at any byte, with and without the blend records, against the
oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("P", [1, 63, 64, 65, 127, 255, 256, 257, 1000])
@pytest.mark.parametrize("shift", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("records", [False, True])
def test_colours_and_flags(orc, P, shift, records):
    import gpu_harness as H
    import gs_scenes
    g, cams = gs_scenes.make_scene(0, P=P, n_views=1)
    g["shs"] = g["shs"] * 8.0  # (many colours below 0)
    cam = cams[0]
    W, Hh = cam.image_width, cam.image_height
    gd = {k: H.dev(v) for k, v in g.items() if torch.is_tensor(v)}
    f = lambda *s: torch.full(s, 77.0, device=DEV)
    means2D, depths, co, rgb = f(P, 2), f(P), f(P, 4), f(P, 3)
    radii = torch.full((P,), 77, dtype=torch.int32, device=DEV)
    flags = torch.full((3 * P + shift + 8,), 77, dtype=torch.uint8, device=DEV)
    rec = f(P, 16) if records else None
    V, PM, cp = H.dev(cam.world_view_transform), H.dev(cam.full_proj_transform), H.dev(cam.camera_center)
    H.gn.check(H.lib.gs_preprocess_forward(
        H.ptr(means2D), H.ptr(depths), H.ptr(radii), None, H.ptr(co), H.ptr(rgb), H.ptr(flags[shift:]), None, P, 3, 16, W,
        Hh, H.ptr(gd["means3D"]), H.ptr(gd["scales"]), H.ptr(gd["rotations"]), H.ptr(gd["shs"]), H.ptr(gd["opacities"]),
        1.0, H.ptr(V), H.ptr(PM), H.ptr(cp), cam.tanfovx, cam.tanfovy, 0, 1, None, H.ptr(rec), H.stream()),
        "gs_preprocess_forward")
    torch.cuda.synchronize()
    want = H.oracle_preprocess(orc, g, cam)
    n = lambda t: t.cpu().numpy()
    for got, k in ((radii, "radii"), (depths, "depths"), (means2D, "means2D"), (co, "conic_opacity"), (rgb, "rgb")):
        assert np.array_equal(n(got), want[k].reshape(n(got).shape)), k
    got = n(flags)
    assert np.array_equal(got[shift:shift + 3 * P].reshape(P, 3), want["clamped"].reshape(P, 3))
    assert (got[:shift] == 77).all() and (got[shift + 3 * P:] == 77).all()
    if records:
        ok = want["radii"] > 0
        r = n(rec)[ok]
        assert np.array_equal(r[:, :2], want["means2D"][ok]) and np.array_equal(r[:, 2:6], want["conic_opacity"][ok])
        assert np.array_equal(r[:, 6:9], want["rgb"][ok]) and np.array_equal(r[:, 14], want["depths"][ok])


@pytest.mark.parametrize("P,channels", [((2 << 20) + 77, False), ((4 << 20) + 77, True)])
def test_backward_of_many_gaussians(P, channels):
    """The backward kernel for large steps against the one for small ones, bit for bit: a Gaussian's gradients do not depend
    on the others, so the step in parts gives the same."""
    import gs_scenes
    from diff_gaussian_rasterization import _C
    _, cams = gs_scenes.make_scene(0, P=8, n_views=1)
    cam = cams[0]
    W, Hh = cam.image_width, cam.image_height
    gen = torch.Generator(device=DEV).manual_seed(P)
    n = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    means, scales, rots = n(P, 3) * 6, torch.exp(n(P, 3) * 0.5 - 4), torch.nn.functional.normalize(n(P, 4))
    sh, op = n(P, 16, 3) * 0.3, torch.sigmoid(n(P, 1))
    view = [t.to(DEV) for t in (cam.world_view_transform, cam.full_proj_transform, cam.camera_center)]
    args = {"stats_collector": {}}
    (_, _, _, radii, _, _, _, clamped), ddir = _C.preprocess_gaussians_ex(
        means, scales, rots, sh, op, 1.0, view[0], view[1], cam.tanfovx, cam.tanfovy, Hh, W, 3, view[2], False, False, args,
        want_direction_derivative=True, want_cov3D=False)
    live = int((radii > 0).sum())
    assert 0 < live < P and bool(clamped.bool().any())
    up = [n(P, 2), n(P, 4), n(P, 3)]
    am = n(P, 5) if channels else None
    if channels:
        am[::3] = 0.0

    def backward(a, b):
        return _C.preprocess_gaussians_backward(
            radii[a:b].contiguous(), None, clamped[a:b].contiguous(), means[a:b], scales[a:b], rots[a:b], sh[a:b], 1.0,
            view[0], view[1], cam.tanfovx, cam.tanfovy, Hh, W, 3, view[2], up[0][a:b], up[1][a:b], up[2][a:b], live, False,
            args, dcolor_ddir=ddir[a:b].contiguous(), dL_dall_map=None if am is None else am[a:b])

    whole = backward(0, P)
    for a, b in ((0, P // 2 + 3), (P // 2 + 3, P)):
        for k, (w, part) in enumerate(zip(whole, backward(a, b))):
            assert torch.equal(w[a:b], part), k
