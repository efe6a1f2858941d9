"""Outputs that are zeros without being computed, whatever the memory held: the images of the geometry channels where these
are not rendered, and the gradient of colours that are no spherical-harmonics coefficients."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _dirty(n):
    """Leaves NaNs in the memory that torch hands out next."""
    junk = [torch.full((k,), float("nan"), device=DEV) for k in (n, 5 * n, 3 * n, 16)]
    del junk


# images of fewer floats than a 16-byte word, of none left over, of one to three; more than one round of 511 workgroups
@pytest.mark.parametrize("W,H", [(1, 1), (3, 1), (41, 27), (16, 16), (333, 217), (1701, 1303)])
@pytest.mark.parametrize("limits,ahead", [(None, False), (None, True), ((0, 0), False)])
def test_images_that_are_not_rendered(W, H, limits, ahead):
    from diff_gaussian_rasterization import _C
    n = 200
    gen = torch.Generator().manual_seed(W)
    m2 = (torch.rand(n, 2, generator=gen) * torch.tensor([float(W), float(H)])).to(DEV)
    co = torch.tensor([[0.5, 0.0, 0.5, 0.3]]).repeat(n, 1).to(DEV)
    gx, gy = (W + 15) // 16, (H + 15) // 16
    args = {"stats_collector": {}}
    if limits is not None:
        args["tile_sort_limits"] = limits
    _dirty(W * H)
    out, info = _C.render_gaussians_ex(
        torch.zeros(3, device=DEV), H, W, m2, torch.rand(n, generator=gen).to(DEV) + 1,
        torch.ones(n, dtype=torch.int32, device=DEV), co, torch.rand(n, 3, generator=gen).to(DEV),
        torch.ones(gy, gx, dtype=torch.bool, device=DEV), torch.eye(4, device=DEV), torch.zeros(3, device=DEV), 0.5, 0.5,
        None, False, False, args, expected_instances=20 * n if ahead else 0)
    assert info["launched_ahead"] == ahead
    assert out[6].shape == (5, H, W) and not out[6].view(torch.int32).any()
    assert out[7].shape == (1, H, W) and not out[7].view(torch.int32).any()


@pytest.mark.parametrize("P", [1, 63, 64, 65, 255, 256, 257, 1000])
def test_gradient_of_plain_colours(P):
    from diff_gaussian_rasterization import _C
    gen = torch.Generator().manual_seed(P)
    r = lambda *s: torch.randn(*s, generator=gen).to(DEV)
    means = r(P, 3) * 0.5
    means[:, 2] = means[:, 2].abs() + 2.0
    scales, rots = r(P, 3).abs() * 0.1 + 0.01, torch.nn.functional.normalize(r(P, 4))
    proj = torch.tensor([[1., 0, 0, 0], [0, 1, 0, 0], [0, 0, 1, 1], [0, 0, -0.01, 0]], device=DEV)
    cam = (torch.eye(4, device=DEV), proj)
    radii = torch.ones(P, dtype=torch.int32, device=DEV)
    clamped = torch.zeros(P, 3, dtype=torch.bool, device=DEV)
    g2, gco = r(P, 2), r(P, 4)

    def run(grad_colours):
        _dirty(P)
        return _C.preprocess_gaussians_backward(radii, None, clamped, means, scales, rots, r(P, 3), 1.0, *cam, 0.5, 0.5, 64,
                                                64, 0, torch.zeros(3, device=DEV), g2, gco, grad_colours, 0, False, {})

    got, want = run(None), run(torch.ones(P, 3, device=DEV))
    for a, b in zip(got, want):
        assert torch.equal(a, b) and torch.isfinite(a).all()
    assert got[3].shape == (P, 3) and not got[3].view(torch.int32).any()
    assert torch.equal(got[4], gco[:, 3:])


# A caller that was compiled before the field, one that leaves it at its default (0, or below zero as in any field), and one
# that asks for it.  The other fields hold either way: lists launched ahead, the caller's operand records.
@pytest.mark.parametrize("older,clear,images", [(False, 1, True), (False, 0, True), (False, 0, False), (False, -1, True),
                                                (False, -1, False), (True, 1, True), (True, 1, False)])
def test_who_has_the_images_cleared(older, clear, images):
    import ctypes as C
    import gsrast_native as gn
    n, W, H = 300, 41, 27
    gen = torch.Generator().manual_seed(n)
    r = lambda *s: torch.rand(*s, generator=gen).to(DEV)
    m2, co = r(n, 2) * torch.tensor([W, H], device=DEV), torch.tensor([[0.5, 0.0, 0.5, 0.3]], device=DEV).repeat(n, 1)
    depths, rgb, radii = r(n) + 1, r(n, 3), torch.ones(n, dtype=torch.int32, device=DEV)
    records = torch.cat([m2, co, rgb, torch.zeros(n, 5, device=DEV), depths[:, None], torch.zeros(n, 1, device=DEV)], 1).contiguous()
    cl, zero3 = torch.ones(2, 3, dtype=torch.bool, device=DEV), torch.zeros(3, device=DEV)
    p = lambda t: None if t is None else C.c_void_p(t.data_ptr())

    def run(options):
        kept = []

        def buffer(size, user):
            kept.append(torch.zeros(size, dtype=torch.uint8, device=DEV))
            return kept[-1].data_ptr()
        fn, result, count = gn.RESIZE_FN(buffer), gn.RenderResult(), C.c_int()
        color = torch.full((3, H, W), float("nan"), device=DEV)
        stats = [torch.zeros(k, dtype=torch.int32, device=DEV) for k in (6, 6, 6, n)]
        geo = [torch.full((k, H, W), 7.0, device=DEV) if images else None for k in (5, 1)]
        gn.stage_timing(True)
        status = gn.lib.gs_render_forward(fn, None, fn, None, fn, None, n, p(zero3), W, H, 41.0, 27.0, W / 2, H / 2, None, None,
                                          None, p(m2), p(depths), p(radii), p(co), p(rgb), p(cl), p(color),
                                          *[p(s) for s in stats], p(geo[0]), p(geo[1]), None, 0, 0, C.byref(count), None,
                                          C.byref(options) if options else None, C.byref(result),
                                          C.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        gn.stage_timing(False)
        gn.check(status, "gs_render_forward")
        return color, geo, result, gn.stage_timing_collect().get("pack_operands", (0.0, 0))[1], count.value

    options = gn.RenderOptions(expected_instances=20 * n, blend_records=records.data_ptr())
    options.clear_geo_images = clear
    if older:
        options.struct_bytes = gn.RenderOptions.clear_geo_images.offset
        options.recent_longest_list = -559038737
    color, geo, result, packs, R = run(options)
    assert result.launched_ahead == 1 and packs == 0 and R * 5 > n * 4
    want, _, _, packs, _ = run(None)
    assert packs == 1 and torch.equal(color.view(torch.int32), want.view(torch.int32))
    for image in geo:
        assert image is None or bool((image == (0.0 if clear > 0 and not older else 7.0)).all())
