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
