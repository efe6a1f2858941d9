"""Which views the forward call packs operand records for: by their own figures, also where a view launched ahead of its
instance count did not fit and had been taken for one that needs none.  The results are the gathered operands' bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
W, H = 80, 48  # 5 x 3 tiles


def view(n, everywhere, unseen, seed):
    """n Gaussians of one tile each, `everywhere` that are in every tile's list, `unseen` of radius 0."""
    gen = torch.Generator().manual_seed(seed)
    P = n + everywhere + unseen
    r = lambda *s: torch.rand(*s, generator=gen)
    # (single tiles: their centres three pixels and more from the tile's edges, radius 2)
    tile = (r(P, 2) * torch.tensor([5.0, 3.0])).floor()
    radii = torch.full((P,), 2, dtype=torch.int32)
    radii[n:n + everywhere] = 300
    radii[n + everywhere:] = 0
    am = torch.randn(P, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0
    return {k: v.to(DEV) for k, v in dict(
        means2D=tile * 16 + 3 + r(P, 2) * 9, radii=radii, depths=r(P) * 10 + 1, rgb=r(P, 3), am=am,
        co=torch.stack([0.2 + r(P), r(P) * 0.1, 0.2 + r(P), r(P) * 0.2], 1), bg=torch.tensor([0.3, 0.6, 0.1]),
        u3=torch.randn(3, H, W, generator=gen), u5=torch.randn(5, H, W, generator=gen),
        u1=torch.randn(1, H, W, generator=gen)).items()}


def render(d, instances, longest, recent=0):
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    cl = torch.ones(3, 5, dtype=torch.bool, device=DEV)
    args = {"stats_collector": {}}
    gn.stage_timing(True)
    out, info = _C.render_gaussians_ex(d["bg"], H, W, d["means2D"], d["depths"], d["radii"], d["co"], d["rgb"], cl,
                                       torch.eye(4, device=DEV), torch.zeros(3, device=DEV), 0.5, 0.5, d["am"], True,
                                       False, args, expected_instances=instances, expected_longest_list=longest,
                                       recent_longest_list=recent)
    torch.cuda.synchronize()
    gn.stage_timing(False)
    packs = gn.stage_timing_collect().get("pack_operands", (0.0, 0))[1]
    back = _C.render_gaussians_backward(d["bg"], 0.5, 0.5, out[6], d["am"], out[0], out[8], out[9], out[10], cl,
                                        d["u3"], d["u5"], d["u1"], d["means2D"], d["co"], d["rgb"], True, False, args,
                                        binning_capacity=info["binning_capacity"])
    return packs, info, out[0], [*out[1:8], *back]


# instances per Gaussian and longest list: beyond the register sort's 4096 records pay from 0.4 on, else from 0.8
@pytest.mark.parametrize("n,everywhere,unseen,packed", [(0, 4097, 0, True), (0, 4097, 149000, True),
                                                        (0, 4097, 150000, False), (0, 4096, 100000, False),
                                                        (3000, 100, 2500, True), (3000, 100, 2600, False)])
def test_by_the_views_own_figures(n, everywhere, unseen, packed):
    d = view(n, everywhere, unseen, seed=n + everywhere + unseen)
    P, R = n + everywhere + unseen, n + 15 * everywhere
    packs, info, got_R, want = render(d, 0, 0)
    assert got_R == R and packs == (1 if packed else 0)
    longest = info["longest_list"]
    assert (R * 5 > P * (2 if longest > 4096 else 4)) == packed
    # launched ahead: what is expected decides (less the margin a caller adds), then, where that does not hold, the view
    for instances, bound, ahead in ((R + R // 4, 0, True), (R // 4, 0, False), (R + R // 4, longest - 1, False),
                                    (max(4 * P, R), 0, True), (max(4 * P, R), longest - 1, False)):
        packs, info, _, got = render(d, instances, bound)
        assert info["launched_ahead"] == ahead
        expected = (instances - instances // 5) * 5 > P * (2 if bound == 0 or bound > 4096 else 4)
        assert packs == (1 if ahead and expected else 0 if ahead else 2 if expected else 1 if packed else 0)
        for a, b in zip(want, got):
            assert np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)


# launched for lists of any length: the views that the expectation comes from say how long they are
@pytest.mark.parametrize("instances,recent,packed", [(0.7, 0, True), (0.7, -1, True), (0.7, 100, False), (0.7, 4096, False),
                                                     (0.7, 4097, True), (0.39, 4097, False), (0.9, 100, True)])
def test_by_the_lists_of_the_views_before(instances, recent, packed):
    d = view(3000, 100, 2600, seed=3)
    want = render(d, 0, 0)[3]
    packs, info, _, got = render(d, int(instances * 5700 * 1.25), 0, recent)
    assert info["launched_ahead"] == (instances * 5700 * 1.25 >= 4500)
    assert packs == (1 if packed else 0)  # (the view's own figures, 4500 instances and a list of 300: none)
    for a, b in zip(want, got):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)


# launched ahead on a buffer that turns out too small, or on too short a bound: whatever was launched leaves it alone, the
# operand records too
@pytest.mark.parametrize("instances,longest", [(5000, 0), (100_000, 299)])
def test_a_view_that_does_not_fit_leaves_the_buffer_it_was_launched_on(instances, longest):
    import ctypes as C
    import gsrast_native as gn
    d = view(4500, 300, 100, seed=9)
    P, R = 4900, 4500 + 15 * 300
    want = render(d, 0, 0)[3]
    p, kept = (lambda t: C.c_void_p(t.data_ptr())), []

    def buffer(fill):
        def resize(size, user):
            kept.append(torch.full((size,), fill, dtype=torch.uint8, device=DEV))
            return kept[-1].data_ptr()
        return gn.RESIZE_FN(resize)
    other, binning = buffer(0), buffer(0xAB)
    color, omap, depth = (torch.full((k, H, W), float("nan"), device=DEV) for k in (3, 5, 1))
    stats = [torch.zeros(k, dtype=torch.int32, device=DEV) for k in (15, 15, 15, P)]
    cl, zero3 = torch.ones(3, 5, dtype=torch.bool, device=DEV), torch.zeros(3, device=DEV)
    options, result, count = gn.RenderOptions(-1, -1, instances, longest), gn.RenderResult(), C.c_int()
    gn.check(gn.lib.gs_render_forward(other, None, binning, None, other, None, P, p(d["bg"]), W, H, W / 1.0, H / 1.0, W / 2, H / 2,
                                      None, None, p(d["am"]), p(d["means2D"]), p(d["depths"]),
                                      p(d["radii"]), p(d["co"]), p(d["rgb"]), p(cl), p(color), *[p(s) for s in stats], p(omap),
                                      p(depth), None, 1, 0, C.byref(count), None, C.byref(options), C.byref(result),
                                      C.c_void_p(torch.cuda.current_stream().cuda_stream)), "gs_render_forward")
    torch.cuda.synchronize()
    assert count.value == R and result.launched_ahead == 0
    first, second = [b for b in kept if bool((b[-1:] == 0xAB).all())]
    assert first.numel() >= 64 * P and bool((first == 0xAB).all())
    assert torch.equal(color.view(torch.int32), want[0].view(torch.int32))
