"""Operator API of CityGS-X's differentiable Gaussian rasterizer on MI355X.

Same names, argument order, shapes, dtypes and gradient contracts as
submodule_cityx/diff-gaussian-rasterization/diff_gaussian_rasterization/__init__.py
(GaussianRasterizationSettings :314-327, GaussianRasterizer :329-405,
preprocess op :46-146, render op :182-303), so gaussian_renderer/__init__.py
and train.py can call it unchanged.  The native side is libgsrast.so
(hand-written gfx950 kernels) reached through `_C`.

One addition: passing SH coefficients shaped (P, M, 3) as `shs` makes
preprocess evaluate colour from spherical harmonics at `sh_degree` and return
the matching dL/dshs; any other `shs` shape keeps the reference behaviour
(colour output zero, zero gradient of the same shape as `shs`).
"""
import weakref
from typing import NamedTuple

import torch
import torch.nn as nn

import gsrast_native as _n

from . import _C

__all__ = ["GaussianRasterizationSettings", "GaussianRasterizer", "preprocess_gaussians", "render_gaussians",
           "build_all_map"]


class GaussianRasterizationSettings(NamedTuple):
    image_height: int
    image_width: int
    tanfovx: float
    tanfovy: float
    bg: torch.Tensor
    scale_modifier: float
    viewmatrix: torch.Tensor
    projmatrix: torch.Tensor
    sh_degree: int
    campos: torch.Tensor
    prefiltered: bool
    render_geo: bool
    debug: bool


# ------------------------------------------------------------ blend records --

# The blend kernels read a Gaussian's operands (centre, conic, opacity, colour, geometry channels, depth) as one
# 64-byte record.  The library packs those records itself from the separate tensors, one more pass per view, unless
# preprocess_gaussians has written them on the way: it has every value but the geometry channels at hand, and
# those it forms as build_all_map does, from the same parameters and camera.  The records travel as an attribute
# of the means2D tensor.  render_gaussians uses them only if every tensor it is given is the very tensor the
# records were written from, unmodified since (tensor identity and version counters), and, with geometry channels
# to render, if all_map is what build_all_map(..., blend_records_of=means2D) returned for the very parameter
# tensors and camera preprocess_gaussians had; otherwise the library packs.  Nothing a caller sees changes: same
# tensors, same values.

# In the same way preprocess_gaussians forms the channels themselves once a caller builds all_map through
# build_all_map(..., blend_records_of=means2D): that call then hands out what the preprocess kernel left instead of
# launching one of its own.  The autograd graph is the same with and without: build_all_map's result belongs to a node
# of its own, with its own saved tensors, so that a loss on the channels and one that does not go through them can be
# differentiated one after the other.  Where both nodes run in one backward pass the channels' node leaves its gradient
# to the preprocess node (_ChannelGradients), whose kernel has means and rotations in registers.

class _BlendRecords:
    """What one preprocess call leaves for build_all_map and render_gaussians, beside its outputs."""
    __slots__ = ("records", "all_map", "gradients", "stream", "refs", "versions", "sources", "source_versions",
                 "all_map_ref", "all_map_version")

    def __init__(self):
        self.records = None    # the blend kernels' operand records
        self.all_map = None    # the channels, until build_all_map hands them out
        self.gradients = None  # the node's _ChannelGradients
        self.stream = 0        # what the kernel that writes the two was launched on
        self.all_map_ref = None
        self.all_map_version = -1

    def written_from(self, parts, sources):
        """parts: the outputs the records repeat; sources: means3D, scales, rotations, viewmatrix, campos."""
        self.refs = [weakref.ref(t) for t in parts]
        self.versions = [t._version for t in parts]
        self.sources = [weakref.ref(t) for t in sources]
        self.source_versions = [t._version for t in sources]

    def on_this_stream(self, device):
        """Both tensors were allocated for the stream that writes them, and only work on it is ordered behind that."""
        return self.stream == _n.stream_handle(device)

    def same_sources(self, sources):
        return all(ref() is t and t._version == v for ref, v, t in zip(self.sources, self.source_versions, sources))

    def take_all_map(self, sources):
        """The channels preprocess_gaussians formed, if they are those of `sources` and this stream's; once (two
        callers must not share a tensor either may modify)."""
        if self.all_map is None or not self.same_sources(sources) or not self.on_this_stream(sources[0].device):
            return None
        all_map, self.all_map = self.all_map, None
        return all_map

    def usable(self, parts, all_maps, render_geo):
        if self.records is None or not self.on_this_stream(parts[0].device):
            return False
        for ref, version, t in zip(self.refs, self.versions, parts):
            if ref() is not t or t._version != version:
                return False
        if render_geo and (self.all_map_ref is None or self.all_map_ref() is not all_maps
                           or all_maps._version != self.all_map_version):
            return False
        return True


class _ChannelGradients:
    """Carries the gradient of the channels from their node to the preprocess node, which adds what it makes of it to
    its own results, if the preprocess node is still to run in the same backward pass and passes its gradients of
    means and rotations on to where the channels' node would have passed them.  Everything is kept per backward pass
    (the autograd engine numbers them): a pass that failed half way leaves nothing for another one, and passes over a
    retained graph do not meet."""
    __slots__ = ("node", "handed", "done")

    def __init__(self, node):
        self.node = weakref.ref(node)
        self.handed = {}  # pass: gradient
        self.done = set()  # passes in which the preprocess node has run

    def leave(self, channels_node, grad):
        node = self.node()
        if node is None or torch.is_grad_enabled():  # (a graph of the backward pass is asked for)
            return False
        this_pass = torch._C._current_graph_task_id()
        if this_pass < 0 or this_pass in self.done or not torch._C._will_engine_execute_node(node):
            return False
        here, there = channels_node.next_functions, node.next_functions
        if here[0] != there[0] or here[2] != there[2]:
            return False
        self.handed[this_pass] = grad
        return True

    def take(self):
        this_pass = torch._C._current_graph_task_id()
        self.done.add(this_pass)
        return self.handed.pop(this_pass, None)


# The caller builds all_map with blend_records_of=...: records and channels are worth writing.  Only the time depends
# on it, never a result or the graph.
_linked_all_map_seen = [False]


def _have_versions(sources):
    """Whether the link between the calls can be checked: tensors of inference mode have no version counter."""
    return not (torch.is_inference_mode_enabled() or any(t.is_inference() for t in sources))


def _records_wanted(rs, P, device):
    """Whether preprocess should write the records: one of the last views of this image size had enough instances per
    Gaussian for records to pay (written on the way they cost about a third of the library's packing pass, which
    pays from 0.8 instances per Gaussian, 0.4 with long lists), and render_gaussians will be able to use them (no geometry channels to
    render, or the caller builds them through build_all_map(..., blend_records_of=means2D))."""
    seen = _expectations.get((rs.image_height, rs.image_width, device))
    if seen is None or _most_instances(seen) * 10 <= P * 3:
        return False
    return (not rs.render_geo) or _linked_all_map_seen[0]


# --------------------------------------------------------------- preprocess --

class _PreprocessGaussians(torch.autograd.Function):
    @staticmethod
    def forward(ctx, means3D, scales, rotations, sh, opacities, raster_settings, cuda_args, blend):
        rs = raster_settings
        # (when a backward pass can follow, the forward kernel also leaves the colours' derivative with respect to
        # the view direction, nine numbers per Gaussian, which is all the backward kernel needs the coefficients for)
        P = means3D.shape[0]
        linkable = P > 0 and _have_versions((means3D, scales, rotations, rs.viewmatrix, rs.campos))
        records = (torch.empty(P, 16, dtype=torch.float32, device=means3D.device)
                   if linkable and _records_wanted(rs, P, means3D.device) else None)
        all_map = (torch.empty(P, 5, dtype=torch.float32, device=means3D.device)
                   if linkable and rs.render_geo and _linked_all_map_seen[0] else None)
        (num_rendered, means2D, depths, radii, cov3D, conic_opacity, rgb, clamped), ddir = _C.preprocess_gaussians_ex(
            means3D, scales, rotations, sh, opacities, rs.scale_modifier, rs.viewmatrix, rs.projmatrix, rs.tanfovx,
            rs.tanfovy, rs.image_height, rs.image_width, rs.sh_degree, rs.campos, rs.prefiltered, rs.debug, cuda_args,
            want_direction_derivative=any(ctx.needs_input_grad[:5]), want_cov3D=False, blend_records=records,
            all_map=all_map)
        blend.records, blend.all_map = records, all_map
        if records is not None or all_map is not None:
            blend.stream = _n.stream_handle(means3D.device)
        ctx.channel_gradients = blend.gradients = _ChannelGradients(ctx) if all_map is not None else None
        # (cov3D is None: the backward kernel forms the covariances again from scales and rotations, which it reads
        # anyway, instead of both passes moving 24 bytes per Gaussian)
        ctx.raster_settings = rs
        ctx.cuda_args = cuda_args
        ctx.num_rendered = num_rendered
        ctx.has_ddir = ddir is not None
        ctx.save_for_backward(means3D, scales, rotations, sh, radii, cov3D, clamped,
                              *([ddir] if ddir is not None else []))
        ctx.mark_non_differentiable(radii, depths)
        # no zero tensors for the outputs nobody differentiates (radii, depths): backward fills in what it needs
        ctx.set_materialize_grads(False)
        return means2D, rgb, conic_opacity, radii, depths

    @staticmethod
    def backward(ctx, grad_means2D, grad_rgb, grad_conic_opacity, grad_radii, grad_depths):
        rs = ctx.raster_settings
        means3D, scales, rotations, sh, radii, cov3D, clamped, *ddir = ctx.saved_tensors
        grad_all_map = ctx.channel_gradients.take() if ctx.channel_gradients is not None else None
        ddir = ddir[0] if ctx.has_ddir else None
        P = means3D.shape[0]
        if grad_means2D is None:
            grad_means2D = means3D.new_zeros(P, 2)
        if grad_conic_opacity is None:
            grad_conic_opacity = means3D.new_zeros(P, 4)
        dL_dmeans3D, dL_dscales, dL_drotations, dL_dsh, dL_dopacity = _C.preprocess_gaussians_backward(
            radii, cov3D, clamped, means3D, scales, rotations, sh, rs.scale_modifier, rs.viewmatrix, rs.projmatrix,
            rs.tanfovx, rs.tanfovy, rs.image_height, rs.image_width, rs.sh_degree, rs.campos, grad_means2D,
            grad_conic_opacity, grad_rgb, ctx.num_rendered, rs.debug, ctx.cuda_args, dcolor_ddir=ddir,
            dL_dall_map=grad_all_map)
        if dL_dsh.shape != sh.shape:
            dL_dsh = torch.zeros_like(sh)
        return dL_dmeans3D, dL_dscales, dL_drotations, dL_dsh, dL_dopacity, None, None, None


def preprocess_gaussians(means3D, scales, rotations, sh, opacities, raster_settings, cuda_args):
    blend = _BlendRecords()
    means2D, rgb, conic_opacity, radii, depths = _PreprocessGaussians.apply(
        means3D, scales, rotations, sh, opacities, raster_settings, cuda_args, blend)
    if blend.records is not None or blend.all_map is not None:
        blend.written_from((means2D, conic_opacity, rgb, depths),
                           (means3D, scales, rotations, raster_settings.viewmatrix, raster_settings.campos))
        means2D._gs_blend = blend
    return means2D, rgb, conic_opacity, radii, depths


# ------------------------------------------------------------------- render --

# What the last views of a given image size needed, (instances, longest list, whether any view of the size had a list
# beyond _LONG_LIST, the first two of the _RECENT_VIEWS last ones) keyed by (height, width, device): the
# next view of that size is launched without waiting for its instance count, on buffers sized for the most instances of
# those views and the longest list of the last one plus
# a margin (a training loop renders thousands of similar views; the number of Gaussians changes at every
# densification, so it is not part of the key).  A scene's cameras differ by more than the margin: in a loop over views of
# 6.2 M and 2.7 M instances every view of the larger kind missed an expectation taken from the view before it.
# Only the time and the memory depend on it, never a result; a stale or missing entry costs one ordinary call, and the
# binning buffer of a view that fits has the expected size until its backward pass has run.
# Behind a dense view the next seven of its size pack or write operand records for its sake, sparse ones too.  One dense
# view in eight, us a training view with this expectation and with that of the last view alone (channels linked; built
# apart; colour only): 1 M Gaussians obliquely and through a narrow lens 387 and 387; 425 and 436; 353 and 353; 4 M from the
# air, 0.8 and 0.1 instances a Gaussian, 736 and 740; 902 and 888; 696 and 688; 10 M at street level, 0.6 and 0.02, 1371 and
# 1373; 1753 and 1735; 1303 and 1288.  Peak memory 288 MB for 258 (1 M), else the same.  Against that stands a dense view of
# 10 M that is launched on a buffer that fits but without its records: 350 us of that view.
# A handful of image sizes at most are alive in a run: the oldest entry goes
# when there are more than _MAX_EXPECTATIONS.
_expectations = {}
_MARGIN = 1.25
_MAX_EXPECTATIONS = 16
_RECENT_VIEWS = 8
_LONG_LIST = 4096  # the longest list that is sorted in registers
_LONG_TILE = 3072  # a list from which on the forward blend splits its tile


def _most_instances(seen):
    """Of the last views that an entry of _expectations tells of."""
    return max(n for n, _ in seen[3]) if len(seen) > 3 else seen[0]


def _recent_longest(key):
    """The longest list of the views that the expectation of a size comes from."""
    seen = _expectations.get(key, (0, 0))
    return max(n for _, n in seen[3]) if len(seen) > 3 else seen[1]


def _expectation(key):
    seen = _expectations.get(key)
    if seen is None:
        return 0, 0
    longest, long = seen[1], seen[2:3]
    if longest <= 0:
        return 0, 0  # a view without per-tile lists (a tile grid too large for them): nothing to gain
    # whole variants of the register sort (256 ... 4096 records per list), so that a slightly longer list still fits; beyond
    # it any length (0): the radix sort is launched as well.  So it is for its longest lists wherever a view of this size
    # has had a longer one: cameras on both sides of that length would miss the bound at every other view, for the 4.6 us
    # of an empty launch.
    cap = 256
    while cap < longest * _MARGIN:
        cap *= 2
    return int(_most_instances(seen) * _MARGIN) + 65536, (0 if cap > _LONG_LIST or (cap == _LONG_LIST and any(long)) else cap)


def _launch_bounds(key):
    """The expectation as a view is launched with it: where the longest list, margin included, leaves no tile to split, the
    bound says so (views that may have such tiles have a forward blend of their own, 2 us slower where there are none)."""
    instances, bound = _expectation(key)
    seen = _expectations.get(key)
    if bound == _LONG_LIST and seen is not None and seen[1] * _MARGIN < _LONG_TILE:
        bound = _LONG_TILE - 1
    return instances, bound


def _remember(key, instances, longest):
    seen = _expectations.pop(key, ())  # (re-inserted at the end: the dict keeps insertion order)
    recent = ((instances, longest), *(seen[3] if len(seen) > 3 else (seen[:2],) if seen else ()))[:_RECENT_VIEWS]
    _expectations[key] = (instances, longest, longest > _LONG_LIST or any(seen[2:3]), recent)
    while len(_expectations) > _MAX_EXPECTATIONS:
        # (a copy to look at: another thread may be adding entries, or have removed this one)
        _expectations.pop(list(_expectations)[0], None)


class _RenderGaussians(torch.autograd.Function):
    @staticmethod
    def forward(ctx, means2D, means2D_abs, conic_opacity, rgb, all_maps, depths, radii, compute_locally,
                extended_compute_locally, raster_settings, cuda_args):
        rs = raster_settings
        avoid = bool(cuda_args.get("avoid_pixel_all2all", False)) if cuda_args is not None else False
        mask = extended_compute_locally if avoid else compute_locally
        key = (rs.image_height, rs.image_width, means2D.device)
        expected_instances, expected_longest = _launch_bounds(key)
        blend = getattr(means2D, "_gs_blend", None)
        records = (blend.records if blend is not None and blend.usable((means2D, conic_opacity, rgb, depths), all_maps,
                                                                       rs.render_geo) else None)
        if (blend is not None and records is None and rs.render_geo
                and (blend.records is not None or blend.all_map is not None)):
            # records or channels were written and cannot be used: the caller does not (or no longer) build all_map
            # through build_all_map(..., blend_records_of=means2D); stop writing them until it does
            _linked_all_map_seen[0] = False
        ((num_rendered, color, n_render, n_consider, n_contrib, out_observe, out_all_map, out_plane_depth, geomBuffer,
          binningBuffer, imgBuffer), info) = _C.render_gaussians_ex(
            rs.bg, rs.image_height, rs.image_width, means2D, depths, radii, conic_opacity, rgb, mask, rs.viewmatrix,
            rs.campos, rs.tanfovx, rs.tanfovy, all_maps, rs.render_geo, rs.debug, cuda_args,
            expected_instances=expected_instances, expected_longest_list=expected_longest, blend_records=records,
            recent_longest_list=_recent_longest(key))
        ctx.blend_records = records
        if means2D.shape[0] > 0:
            _remember(key, num_rendered, info["longest_list"])
        if isinstance(cuda_args, dict) and isinstance(cuda_args.get("stats_collector"), dict):
            # (beside the reference's timing keys: whether this view's list kernels ran ahead of its instance count)
            cuda_args["stats_collector"]["launched_ahead"] = info["launched_ahead"]
            cuda_args["stats_collector"]["num_rendered"] = num_rendered
        ctx.binning_capacity = info["binning_capacity"]
        ctx.raster_settings = rs
        ctx.cuda_args = cuda_args
        ctx.num_rendered = num_rendered
        ctx.save_for_backward(means2D, conic_opacity, rgb, all_maps, out_all_map, geomBuffer, binningBuffer, imgBuffer,
                              compute_locally)
        ctx.mark_non_differentiable(n_render, n_consider, n_contrib, out_observe)
        ctx.set_materialize_grads(False)  # the four integer outputs never get a zero "gradient" allocated
        return color, n_render, n_consider, n_contrib, out_observe, out_all_map, out_plane_depth

    @staticmethod
    def backward(ctx, grad_color, grad_n_render, grad_n_consider, grad_n_contrib, grad_out_observe, grad_out_all_map,
                 grad_out_plane_depth):
        rs = ctx.raster_settings
        (means2D, conic_opacity, rgb, all_maps, all_map_pixels, geomBuffer, binningBuffer, imgBuffer,
         compute_locally) = ctx.saved_tensors
        if grad_color is None:
            grad_color = torch.zeros_like(all_map_pixels[:3])
        if rs.render_geo:
            if grad_out_all_map is None:
                grad_out_all_map = torch.zeros_like(all_map_pixels)
            if grad_out_plane_depth is None:
                grad_out_plane_depth = torch.zeros_like(all_map_pixels[:1])
        dL_dmeans2D, dL_dmeans2D_abs, dL_dconic_opacity, dL_dcolors, dL_dall_map = _C.render_gaussians_backward(
            rs.bg, rs.tanfovx, rs.tanfovy, all_map_pixels, all_maps, ctx.num_rendered, geomBuffer, binningBuffer,
            imgBuffer, compute_locally, grad_color, grad_out_all_map, grad_out_plane_depth, means2D, conic_opacity,
            rgb, rs.render_geo, rs.debug, ctx.cuda_args, binning_capacity=ctx.binning_capacity,
            blend_records=ctx.blend_records)
        return (dL_dmeans2D, dL_dmeans2D_abs, dL_dconic_opacity, dL_dcolors, dL_dall_map, None, None, None, None, None,
                None)


def render_gaussians(means2D, means2D_abs, conic_opacity, rgb, all_map, depths, radii, compute_locally,
                     extended_compute_locally, raster_settings, cuda_args):
    return _RenderGaussians.apply(means2D, means2D_abs, conic_opacity, rgb, all_map, depths, radii, compute_locally,
                                  extended_compute_locally, raster_settings, cuda_args)


# ------------------------------------------------------------------ all_map --

class _BuildAllMap(torch.autograd.Function):
    @staticmethod
    def forward(ctx, means3D, scales, rotations, viewmatrix, campos, blend):
        sources = (means3D, scales, rotations, viewmatrix, campos)
        ctx.save_for_backward(*sources)
        all_map = blend.take_all_map(sources) if blend is not None else None
        ctx.gradients = blend.gradients if all_map is not None else None
        return all_map if all_map is not None else _C.build_all_map(*sources)

    @staticmethod
    def backward(ctx, grad_all_map):
        means3D, scales, rotations, viewmatrix, campos = ctx.saved_tensors
        if ctx.gradients is not None and ctx.gradients.leave(ctx, grad_all_map):
            return (None,) * 6
        dL_dmeans3D, dL_drotations = _C.build_all_map_backward(means3D, scales, rotations, viewmatrix, campos,
                                                               grad_all_map)
        return dL_dmeans3D, None, dL_drotations, None, None, None


def build_all_map(means3D, scales, rotations, viewmatrix, campos, blend_records_of=None):
    """[normal in the camera frame, 1, |normal . p_cam|] per Gaussian: a drop-in for the torch lines
    gaussian_renderer/__init__.py:1501-1518 (pass the camera's world_view_transform and camera_center).
    Differentiable in means3D and rotations, like those lines; `scales` only picks the axis.
    blend_records_of (optional): the means2D tensor preprocess_gaussians returned for the same parameter tensors
    and camera (the settings' viewmatrix and campos tensors).  preprocess_gaussians then writes the blend kernels'
    operand records with these very channels in them (from the next view on), and render_gaussians, given these
    very tensors, skips the pass that packs them; it also forms this tensor's values and, where one backward pass runs
    through both, takes its gradient.  The returned values, the gradients and the autograd graph are the same either
    way, except that through the link a Gaussian whose channels get a gradient of zero gets zero from them whatever its
    parameters are (build_all_map's own kernel makes a NaN of it where they are not finite).  Both are used on the
    stream preprocess_gaussians ran on only."""
    sources = (means3D, scales, rotations, viewmatrix, campos)
    if blend_records_of is None:
        return _BuildAllMap.apply(*sources, None)
    _linked_all_map_seen[0] = True
    blend = getattr(blend_records_of, "_gs_blend", None)
    all_map = _BuildAllMap.apply(*sources, blend)
    if blend is not None and blend.same_sources(sources) and not all_map.is_inference():
        blend.all_map_ref = weakref.ref(all_map)
        blend.all_map_version = all_map._version
    return all_map


# ------------------------------------------------------------------- module --

class GaussianRasterizer(nn.Module):
    def __init__(self, raster_settings):
        super().__init__()
        self.raster_settings = raster_settings

    def markVisible(self, positions):
        """Boolean mask of points in front of the camera."""
        with torch.no_grad():
            rs = self.raster_settings
            return _C.mark_visible(positions, rs.viewmatrix, rs.projmatrix)

    def preprocess_gaussians(self, means3D, scales, rotations, shs, opacities, cuda_args=None):
        return preprocess_gaussians(means3D, scales, rotations, shs, opacities, self.raster_settings, cuda_args)

    def visible_filter(self, means3D, scales=None, rotations=None, cov3D_precomp=None):
        rs = self.raster_settings
        return _C.rasterize_aussians_filter(means3D, scales, rotations, rs.scale_modifier, cov3D_precomp, rs.viewmatrix,
                                            rs.projmatrix, rs.tanfovx, rs.tanfovy, rs.image_height, rs.image_width,
                                            rs.prefiltered, rs.debug)

    def render_gaussians(self, means2D, means2D_abs, conic_opacity, rgb, all_map, depths, radii, compute_locally,
                         extended_compute_locally, cuda_args=None):
        return render_gaussians(means2D, means2D_abs, conic_opacity, rgb, all_map, depths, radii, compute_locally,
                                extended_compute_locally, self.raster_settings, cuda_args)
