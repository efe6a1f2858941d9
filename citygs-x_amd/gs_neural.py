"""Neural-Gaussian generation of the reference, generate_neural_gaussians (gaussian_renderer/__init__.py:789-899),
as three kernel launches forward (opacity MLP, scan, color/cov MLPs with the post-processing) and two backward,
in libgsrast.so.  The fused operator is the reference's default model configuration (arguments/__init__.py:94-124):
feat_dim 32, inputs [feature, view direction]; the operator also takes the optional distance and level inputs of the
three MLPs (add_opacity_dist, add_color_dist, add_cov_dist, add_level) and the per-anchor opacity factor of dist2level
'progressive'; the drop-in function also serves the appearance embedding and the feature bank, which reduce to it."""
import torch

import gsrast_native as _n

_ops = _n.ops


class _NeuralGaussians(torch.autograd.Function):
    @staticmethod
    def forward(ctx, anchor, feat, offsets, scaling, campos, opacity_scale, level, input_flags, *params):
        if len(params) != 12:
            raise RuntimeError("expected W1, b1, W2, b2 of the opacity, color and cov MLPs (12 tensors)")
        if offsets.dim() != 3:
            raise RuntimeError("offsets must be (anchors, n_offsets, 3)")
        k = offsets.shape[1]
        if not _n.lib.gs_neural_supported(k):
            raise NotImplementedError(f"n_offsets = {k} is not among the values the kernels are built for")
        out, saved, params, ctx.opacity_scale, ctx.level, ctx.opacity_tanh = _ops.neural_forward(
            anchor, feat, offsets, scaling, campos, opacity_scale, level, input_flags, params,
            _n.stream_handle(anchor.device))
        # (opacity_scale carries no gradient: a buffer of the model)
        ctx.save_for_backward(*saved, *params)
        ctx.input_flags = input_flags
        neural_opacity, mask = out[5:]
        ctx.mark_non_differentiable(neural_opacity, mask)
        ctx.set_materialize_grads(False)
        return out

    @staticmethod
    def backward(ctx, g_xyz, g_color, g_opacity, g_scal, g_rot, _g_nop, _g_mask):
        saved = ctx.saved_tensors
        d_inputs = _ops.neural_backward(*saved[:10], saved[10:], ctx.opacity_scale, ctx.level, ctx.input_flags,
                                          ctx.opacity_tanh, (g_xyz, g_color, g_opacity, g_scal, g_rot),
                                          _n.stream_handle(saved[0].device))
        return (*d_inputs[:4], None, None, None, None, *d_inputs[4:])


def neural_gaussians(anchor, feat, offsets, scaling, camera_center, mlp_opacity, mlp_color, mlp_cov,
                     opacity_scale=None, level=None, input_flags=0):
    """The body of generate_neural_gaussians after the visible_mask gathers (gaussian_renderer/__init__.py:800-896).
    anchor (N,3), feat (N,32), offsets (N,k,3), scaling (N,6) = get_scaling, camera_center (3); each mlp_* is
    (W1, b1, W2, b2) as nn.Linear holds them; opacity_scale (N), if given, multiplies the opacity MLP's output per
    anchor (:844-848); input_flags (add_opacity_dist = 1, add_color_dist = 2, add_cov_dist = 4: that MLP's W1 has a
    column for the distance; add_level = 8: all three have a last column for level (N), :824-877).
    Returns (xyz, color, opacity, scaling, rot, neural_opacity, mask);
    differentiable in everything but the camera centre; neural_opacity and mask carry no gradient (the reference
    uses them detached, scene/gaussian_model.py:1183)."""
    return _NeuralGaussians.apply(anchor, feat, offsets, scaling, camera_center, opacity_scale, level, input_flags,
                                  *mlp_opacity, *mlp_color, *mlp_cov)


class _VisibleRows(torch.autograd.Function):
    """The rows of anchor, feat, offsets and scaling that a bool mask selects (gaussian_renderer/__init__.py:794-798)
    and their numbers: what nonzero() and four index_select()s give."""

    @staticmethod
    def forward(ctx, mask, anchor, feat, offsets, scaling, want_index):
        *out, index, rank = _ops.visible_rows(mask, anchor, feat, offsets, scaling, want_index,
                                                _n.stream_handle(anchor.device))
        ctx.save_for_backward(rank)
        ctx.k = offsets.shape[1]
        ctx.set_materialize_grads(False)
        # rows of an array without a gradient carry none either
        ctx.mark_non_differentiable(*[t for t, need in zip(out, ctx.needs_input_grad[1:5]) if not need],
                                    *([index] if want_index else []))
        return (*out, index)

    @staticmethod
    def backward(ctx, *grads):
        rank, = ctx.saved_tensors
        grads = [g if need else None for g, need in zip(grads[:4], ctx.needs_input_grad[1:5])]
        if torch.is_grad_enabled():  # a graph of the backward pass is asked for
            A = rank.shape[0]
            idx = (rank >= 0).nonzero(as_tuple=True)[0]
            return (None, *[None if g is None else g.new_zeros(A, *g.shape[1:]).index_add(0, idx, g) for g in grads],
                    None)
        return (None, *_ops.visible_rows_backward(rank, ctx.k, grads, _n.stream_handle(rank.device)), None)


def _visible_rows(mask, anchor, feat, offsets, scaling, want_index):
    """anchor[mask], feat[mask], offsets[mask], scaling[mask] and, if wanted, mask.nonzero(): one pass over the arrays
    where they are the dense float32 arrays of a model on the current device with 16-byte rows of features, torch's
    gathers for everything else (other types, strides, devices and mask shapes, n_offsets without a kernel, a stream
    under capture)."""
    t4 = (anchor, feat, offsets, scaling)
    if (mask.dtype is torch.bool and mask.is_cuda and mask.dim() == 1 and mask.is_contiguous()
            and all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.dtype is torch.float32
                    and t.device == mask.device and t.is_contiguous() and t.shape[0] == mask.shape[0] for t in t4)
            and anchor.shape[1:] == (3,) and feat.shape[1:] == (32,) and scaling.shape[1:] == (6,)
            and offsets.dim() == 3 and offsets.shape[2] == 3 and _n.lib.gs_neural_supported(offsets.shape[1])
            and feat.data_ptr() % 16 == 0 and mask.shape[0] > 0
            and mask.device.index == torch.cuda.current_device()
            and not torch.cuda.is_current_stream_capturing()):
        return _VisibleRows.apply(mask, anchor, feat, offsets, scaling, want_index)
    # one nonzero() (one host synchronisation) serves the four gathers; x[visible_mask] would run it four times
    idx = mask.nonzero(as_tuple=True)[0]
    return (*[t.index_select(0, idx) for t in t4], idx)


def _linear_pair(seq):
    """(W1, b1, W2, b2) of a Sequential(Linear, ReLU, Linear[, activation]) (scene/gaussian_model.py:131-149)."""
    first, second = seq[0], seq[2]
    return first.weight, first.bias, second.weight, second.bias


def generate_neural_gaussians(viewpoint_camera, pc, visible_mask=None, is_training=False, ape_code=-1):
    """Same signature and results as gaussian_renderer/__init__.py:789-899.  Served: the default configuration,
    the appearance embedding (appearance_dim > 0: every anchor of a view gets the same embedding row, :830-836,
    :866-868, so its part of the first color layer is a per-view addition to that layer's bias) and the feature
    bank (use_feat_bank, :809-823: the view-dependent mix of the feature's resolutions is a few torch lines ahead
    of the fused operator), dist2level 'progressive' (:844-848: the opacity of an anchor in transition is scaled
    by its progress ratio) and the distance / level inputs of the MLPs (add_opacity_dist, add_color_dist,
    add_cov_dist, add_level, :824-829, :839-877)."""
    input_flags = ((1 if pc.add_opacity_dist else 0) | (2 if pc.add_color_dist else 0) | (4 if pc.add_cov_dist else 0)
                   | (8 if pc.add_level else 0))
    level = None
    progressive = pc.dist2level == "progressive"
    opacity_scale = None
    if visible_mask is None:
        anchor, feat, offsets, scaling = pc.get_anchor, pc.get_anchor_feat, pc._offset, pc.get_scaling
        if pc.add_level:
            level = pc.get_level.reshape(-1).float()
        if progressive:
            opacity_scale = torch.where(pc.transition_mask, pc._prog_ratio.reshape(-1),
                                        torch.ones_like(pc._prog_ratio.reshape(-1)))
    else:
        anchor, feat, offsets, scaling, idx = _visible_rows(
            visible_mask, pc.get_anchor, pc.get_anchor_feat, pc._offset, pc.get_scaling, pc.add_level or progressive)
        if pc.add_level:
            level = pc.get_level.reshape(-1).index_select(0, idx).float()
        if progressive:
            prog = pc._prog_ratio.reshape(-1).index_select(0, idx)
            opacity_scale = torch.where(pc.transition_mask.index_select(0, idx), prog, torch.ones_like(prog))
    if pc.use_feat_bank:
        ob_view = anchor - viewpoint_camera.camera_center
        ob_view = ob_view / ob_view.norm(dim=1, keepdim=True)
        cat_view = torch.cat([ob_view, level.unsqueeze(1)], dim=1) if pc.add_level else ob_view
        bank_weight = pc.get_featurebank_mlp(cat_view).unsqueeze(dim=1)  # [n, 1, 3]
        f = feat.unsqueeze(dim=-1)
        f = f[:, ::4, :1].repeat([1, 4, 1]) * bank_weight[:, :, :1] + \
            f[:, ::2, :1].repeat([1, 2, 1]) * bank_weight[:, :, 1:2] + \
            f[:, ::1, :1] * bank_weight[:, :, 2:]
        feat = f.squeeze(dim=-1)
    color_mlp = _linear_pair(pc.get_color_mlp)
    if pc.appearance_dim > 0:
        cam_id = viewpoint_camera.uid if (is_training or ape_code < 0) else ape_code[0]
        row = pc.get_appearance(torch.tensor([cam_id], dtype=torch.long, device=anchor.device))[0]
        W1 = color_mlp[0]
        base = 35 + (1 if pc.add_color_dist else 0) + (1 if pc.add_level else 0)  # the embedding's first column
        color_mlp = (W1[:, :base].contiguous(), color_mlp[1] + W1[:, base:] @ row, color_mlp[2], color_mlp[3])
    out = neural_gaussians(anchor, feat, offsets, scaling, viewpoint_camera.camera_center,
                           _linear_pair(pc.get_opacity_mlp), color_mlp, _linear_pair(pc.get_cov_mlp), opacity_scale,
                           level, input_flags)
    return out if is_training else out[:5]
