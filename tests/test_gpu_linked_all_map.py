"""Geometry channels formed by preprocess_gaussians itself (build_all_map(..., blend_records_of=means2D) from the second
view on) against the separate operator: the same bits, forward and backward, also where the channels are used
outside the blend and where only some of the outputs are differentiated.  (tests/test_linked_channels_cpu.py looks at the
autograd graph around them.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("P", [1, 63, 64, 65, 257, 5000])
@pytest.mark.parametrize("sh", [True, False])
@pytest.mark.parametrize("use", ["all", "channels", "colour"])
def test_channels_of_the_preprocess_node(P, sh, use):
    import diff_gaussian_rasterization as dgr
    import gs_scenes
    g, cams = gs_scenes.make_scene(1, P=P, n_views=1)
    cam = cams[0]
    half = P // 2  # some Gaussians behind the camera: culled, but with channels and a gradient of their own
    g["means3D"][:half] = 2.5 * cam.camera_center + g["means3D"][:half] * 0.01
    if not sh:
        g["shs"] = g["shs"][:, 0].contiguous()
    rs = dgr.GaussianRasterizationSettings(
        image_height=cam.image_height, image_width=cam.image_width, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy,
        bg=torch.zeros(3, device=DEV), scale_modifier=1.0, viewmatrix=cam.world_view_transform.to(DEV),
        projmatrix=cam.full_proj_transform.to(DEV), sh_degree=3, campos=cam.camera_center.to(DEV), prefiltered=False,
        render_geo=True, debug=False)
    gen = torch.Generator(device=DEV).manual_seed(P)
    r = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    ups = [r(P, 2), r(P, 3), r(P, 4), r(P, 5)]
    ups[3][P // 3:P // 2] = 0.0  # (a zero row is skipped by the kernel)

    def run(linked, grad=True):
        dgr._linked_all_map_seen[0] = linked
        leaf = {k: g[k].to(DEV).requires_grad_(grad) for k in ("means3D", "scales", "rotations", "opacities", "shs")}
        means2D, rgb, co, radii, depths = dgr.preprocess_gaussians(leaf["means3D"], leaf["scales"], leaf["rotations"],
                                                                   leaf["shs"], leaf["opacities"], rs, None)
        am = dgr.build_all_map(leaf["means3D"], leaf["scales"], leaf["rotations"], rs.viewmatrix, rs.campos,
                               blend_records_of=means2D if linked else None)
        if grad:
            outs = {"all": [means2D, rgb, co, am], "channels": [am], "colour": [rgb]}[use]
            if use == "colour" and not sh:
                outs = [co]
            which = {id(means2D): 0, id(rgb): 1, id(co): 2, id(am): 3}
            torch.autograd.backward(outs, [ups[which[id(o)]] for o in outs])
        return am.detach(), [leaf[k].grad for k in sorted(leaf)]

    try:
        want, want_grads = run(False)
        got, got_grads = run(True)
        assert torch.equal(want, got)
        for a, b in zip(want_grads, got_grads):
            assert (a is None) == (b is None)
            assert a is None or torch.equal(a, b)
        assert torch.equal(want, run(True, grad=False)[0])
        # channels asked for without gradients of an output that has them, and twice from one view
        dgr._linked_all_map_seen[0] = True
        m = g["means3D"].to(DEV).requires_grad_()
        s, q, o, c = (g[k].to(DEV) for k in ("scales", "rotations", "opacities", "shs"))
        means2D = dgr.preprocess_gaussians(m, s, q, c, o, rs, None)[0]
        with torch.no_grad():
            first = dgr.build_all_map(m, s, q, rs.viewmatrix, rs.campos, blend_records_of=means2D)
        second = dgr.build_all_map(m, s, q, rs.viewmatrix, rs.campos, blend_records_of=means2D)
        assert not first.requires_grad and second.requires_grad and first.data_ptr() != second.data_ptr()
        assert torch.equal(first, second) and torch.equal(first, want)
    finally:
        dgr._linked_all_map_seen[0] = False


def test_a_loss_on_the_channels_beside_a_loss_on_the_image():
    """Differentiated in one pass, with the channels on the view's stream or built on one of their own, or (a loss that
    does not go through the channels) one after the other: the gradients of the unlinked view, from the first linked
    view on."""
    import diff_gaussian_rasterization as dgr
    import gs_scenes
    g, cams = gs_scenes.make_scene(1, P=3000, n_views=1)
    cam = cams[0]
    rs = dgr.GaussianRasterizationSettings(
        image_height=cam.image_height, image_width=cam.image_width, tanfovx=cam.tanfovx, tanfovy=cam.tanfovy,
        bg=torch.zeros(3, device=DEV), scale_modifier=1.0, viewmatrix=cam.world_view_transform.to(DEV),
        projmatrix=cam.full_proj_transform.to(DEV), sh_degree=3, campos=cam.camera_center.to(DEV), prefiltered=False,
        render_geo=True, debug=False)
    cl = torch.ones((cam.image_height + 15) // 16, (cam.image_width + 15) // 16, dtype=torch.bool, device=DEV)
    ug = {k: v.to(DEV) for k, v in gs_scenes.upstream_grads(cam).items()}
    g_am = torch.randn(3000, 5, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    side = torch.cuda.Stream()

    def run(linked, how):
        leaf = {k: g[k].to(DEV).requires_grad_() for k in ("means3D", "scales", "rotations", "opacities", "shs")}
        m2abs = torch.zeros(3000, 3, device=DEV, requires_grad=True)
        rast, args = dgr.GaussianRasterizer(rs), {"stats_collector": {}}
        if how == "side stream":
            side.wait_stream(torch.cuda.current_stream())  # (for the leaves)
        means2D, rgb, co, radii, depths = rast.preprocess_gaussians(leaf["means3D"], leaf["scales"], leaf["rotations"],
                                                                    leaf["shs"], leaf["opacities"], args)
        build = lambda: dgr.build_all_map(leaf["means3D"], leaf["scales"], leaf["rotations"], rs.viewmatrix, rs.campos,
                                          blend_records_of=means2D if linked else None)
        if how == "side stream":
            with torch.cuda.stream(side):
                am = build()
            torch.cuda.current_stream().wait_stream(side)
        else:
            am = build()
        out = rast.render_gaussians(means2D, m2abs, co, rgb, am, depths, radii, cl, cl, args)
        image = [out[0], out[5], out[6]], [ug["color"], ug["all_map"], ug["plane_depth"]]
        if how == "one after the other":
            torch.autograd.backward([am], [g_am])
            torch.autograd.backward([means2D, rgb, co], [g_am[:, :2], g_am[:, :3], g_am[:, :4]])
        else:
            torch.autograd.backward(image[0] + [am], image[1] + [g_am])
        torch.cuda.synchronize()
        return am.detach(), [leaf[k].grad for k in sorted(leaf)]

    dgr._linked_all_map_seen[0] = False
    try:
        for how in ("one pass", "one after the other", "side stream"):
            dgr._linked_all_map_seen[0] = False
            am, want = run(False, how)
            for n in range(3):
                got_am, got = run(True, how)
                assert torch.equal(am, got_am)
                for a, b in zip(want, got):
                    # (three terms per gradient, added in another order)
                    assert float((a - b).norm()) <= 1e-6 * float(a.norm()), (how, n)
    finally:
        dgr._linked_all_map_seen[0] = False
