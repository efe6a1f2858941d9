"""The per-pixel loss maps of the reference, utils/loss_utils.py:88-132, as one fused call each way into
libgsrast.so.  `pixelwise_l1_with_mask` and `pixelwise_ssim_with_mask` keep the reference's names and
arguments; `pixelwise_l1_ssim_with_mask` returns both maps from a single pass, which is what
gaussian_renderer/loss_distribution.py:267-279 needs."""
import torch

import gsrast_native as _n

_ops = _n.ops


class _L1SsimMaps(torch.autograd.Function):
    @staticmethod
    def forward(ctx, img1, img2, pixel_mask):
        need = ctx.needs_input_grad[0]
        l1, ss, *saved = _ops.ssim_l1_forward(img1, img2, pixel_mask, need, _n.stream_handle(img1.device))
        if need:
            ctx.save_for_backward(*saved)
        ctx.set_materialize_grads(False)
        return l1, ss

    @staticmethod
    def backward(ctx, g_l1, g_ssim):
        a, b, m, d_mu, d_xx, d_xy = ctx.saved_tensors
        if g_l1 is None and g_ssim is None:
            return torch.zeros_like(a), None, None
        return (_ops.ssim_l1_backward(a, b, m, g_l1, g_ssim, d_mu, d_xx, d_xy, _n.stream_handle(a.device)), None,
                None)


def pixelwise_l1_ssim_with_mask(img1, img2, pixel_mask=None):
    """(|img1 - img2| * mask, SSIM(img1, img2) * mask), both (3, H, W); differentiable in img1 (img2 is the
    ground truth and gets no gradient)."""
    return _L1SsimMaps.apply(img1, img2, pixel_mask)


def pixelwise_l1_with_mask(img1, img2, pixel_mask):
    """utils/loss_utils.py:88-94."""
    return _L1SsimMaps.apply(img1, img2, pixel_mask)[0]


def pixelwise_ssim_with_mask(img1, img2, pixel_mask):
    """utils/loss_utils.py:97-132."""
    return _L1SsimMaps.apply(img1, img2, pixel_mask)[1]
