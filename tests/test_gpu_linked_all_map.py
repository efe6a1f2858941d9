"""Geometry channels formed by preprocess_gaussians itself (build_all_map(..., blend_records_of=means2D) from the second
view on) against the separate operator: the same bits, forward and backward, also where the channels are used
outside the blend and where only some of the node's outputs are differentiated."""
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
