// Host side of the hot entry points for torch: checks, output allocation and the call into libgsrast.so, without the
// interpreter.  The autograd nodes stay in Python; what they call lands here.
//
// A training view makes four such calls with some forty tensors in and thirty out.  As Python over ctypes (a pointer
// object per tensor, an interpreter round trip per allocation, callbacks for the growing buffers) they cost 150 us of
// a view, the backward half of it on autograd's own thread, whose core has none of the interpreter's state in its
// caches: small views waited for the host.
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>

#include <algorithm>
#include <exception>
#include <optional>
#include <vector>

#include "../../include/gsrast.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

constexpr int64_t CHANNELS = 3, MAP_CHANNELS = 5, TILE = 16;

void check(int status, const char* what) {
  if (status != 0) {
    const char* why = gs_last_error();
    TORCH_CHECK(false, what, ": ", why ? why : "");
  }
}

Tensor f32c(const Tensor& t, const char* name) {
  TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, name, " must be float32, got ", t.scalar_type());
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor: this rasterizer has no CPU path");
  return t.contiguous();
}

Tensor f32c(const OptTensor& t, const char* name) { return t.has_value() ? f32c(*t, name) : Tensor(); }

Tensor contiguous_or_none(const OptTensor& t) { return t.has_value() ? t->contiguous() : Tensor(); }

py::object some(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

template <typename T = float>
T* ptr(const Tensor& t) {
  return t.defined() ? (T*)t.data_ptr() : nullptr;
}

gs_stream_t stream_of(uintptr_t s) { return (gs_stream_t)s; }

// A tensor that a kernel reads or writes as P rows where it lies: there is no copy that would put it right.
void check_rows(const OptTensor& t, const char* name, const Tensor& like, at::IntArrayRef shape) {
  TORCH_CHECK(!t.has_value() || (t->scalar_type() == at::kFloat && t->sizes() == shape && t->is_contiguous() &&
                                 t->device() == like.device()),
              name, " must be a contiguous ", shape, " float32 tensor on the same device");
}

struct Options {
  at::TensorOptions f32, i32, u8, b8, i64;
  explicit Options(const at::Device& d)
      : f32(at::TensorOptions().dtype(at::kFloat).device(d)),
        i32(f32.dtype(at::kInt)),
        u8(f32.dtype(at::kByte)),
        b8(f32.dtype(at::kBool)),
        i64(f32.dtype(at::kLong)) {}
};

// A byte tensor that the library grows on demand (resizeFunctional, rasterize_points.cu:31-37).  The library is called
// through its C interface, so an allocation that fails is kept here and thrown once the call is back.
struct GrowBuffer {
  Tensor tensor;
  std::exception_ptr failure;

  explicit GrowBuffer(const at::TensorOptions& u8) : tensor(at::empty({0}, u8)) {}

  static char* resize(size_t nbytes, void* user) noexcept {
    auto* self = (GrowBuffer*)user;
    try {
      if ((size_t)self->tensor.numel() < nbytes)
        self->tensor = at::empty({(int64_t)nbytes}, self->tensor.options());
      return (char*)self->tensor.data_ptr();
    } catch (...) {
      self->failure = std::current_exception();
      return nullptr;
    }
  }
};

py::tuple preprocess_forward(const Tensor& means3D_, const Tensor& scales_, const Tensor& rotations_,
                             const OptTensor& sh, const Tensor& opacity_, float scale_modifier,
                             const Tensor& viewmatrix, const Tensor& projmatrix, const Tensor& campos, float tan_fovx,
                             float tan_fovy, int height, int width, int degree, bool prefiltered, bool debug,
                             bool want_ddir, bool want_cov3D, const OptTensor& blend_records,
                             const OptTensor& all_map, uintptr_t stream) {
  const int64_t P = means3D_.size(0);
  check_rows(blend_records, "blend_records", means3D_, {P, 16});
  check_rows(all_map, "all_map", means3D_, {P, 5});
  const Tensor means3D = f32c(means3D_, "means3D");
  const Options o(means3D.device());
  const c10::DeviceGuard guard(means3D.device());
  const Tensor scales = f32c(scales_, "scales"), rotations = f32c(rotations_, "rotations"),
               opacity = f32c(opacity_, "opacity");
  const Tensor vm = f32c(viewmatrix, "viewmatrix"), pm = f32c(projmatrix, "projmatrix"), cp = f32c(campos, "campos");
  const bool sh_mode = sh.has_value() && sh->dim() == 3 && sh->size(0) == P;
  const int64_t M = sh_mode ? sh->size(1) : 0;
  const Tensor shc = sh_mode ? f32c(*sh, "sh") : Tensor();
  Tensor means2D = at::empty({P, 2}, o.f32), depths = at::empty({P}, o.f32), radii = at::empty({P}, o.i32),
         conic_opacity = at::empty({P, 4}, o.f32), rgb = at::empty({P, 3}, o.f32), clamped = at::empty({P, 3}, o.b8);
  Tensor cov3D = want_cov3D ? at::empty({P, 6}, o.f32) : Tensor();
  Tensor ddir = sh_mode && want_ddir ? at::empty({P, 3, 3}, o.f32) : Tensor();
  int status;
  {
    py::gil_scoped_release nogil;
    status = gs_preprocess_channels_forward(
        ptr(means2D), ptr(depths), ptr<int>(radii), ptr(cov3D), ptr(conic_opacity), ptr(rgb), ptr<uint8_t>(clamped),
        nullptr, (int)P, degree, (int)M, width, height, ptr(means3D), ptr(scales), ptr(rotations), ptr(shc),
        ptr(opacity), scale_modifier, ptr(vm), ptr(pm), ptr(cp), tan_fovx, tan_fovy, prefiltered, debug, ptr(ddir),
        blend_records ? ptr(*blend_records) : nullptr, all_map ? ptr(*all_map) : nullptr, stream_of(stream));
  }
  check(status, "preprocess_gaussians");
  return py::make_tuple(means2D, depths, radii, some(cov3D), conic_opacity, rgb,
                        clamped, some(ddir));
}

py::tuple preprocess_backward(const Tensor& radii, const OptTensor& cov3D_, const Tensor& clamped,
                              const Tensor& means3D_, const Tensor& scales_, const Tensor& rotations_,
                              const OptTensor& sh, float scale_modifier, const Tensor& viewmatrix,
                              const Tensor& projmatrix, float tan_fovx, float tan_fovy, int height, int width,
                              int degree, const Tensor& campos, const Tensor& dL_dmeans2D,
                              const Tensor& dL_dconic_opacity, const OptTensor& dL_dcolors, bool debug,
                              const OptTensor& dcolor_ddir, const OptTensor& dL_dall_map, uintptr_t stream) {
  const int64_t P = means3D_.size(0);
  const bool sh_mode = sh.has_value() && sh->dim() == 3 && sh->size(0) == P;
  if (sh_mode) check_rows(dcolor_ddir, "dcolor_ddir", means3D_, {P, 3, 3});  // (not used otherwise)
  TORCH_CHECK(!dL_dall_map.has_value() || (dL_dall_map->sizes() == at::IntArrayRef({P, 5}) &&
                                           dL_dall_map->device() == means3D_.device()),
              "dL_dall_map must have shape [", P, ", 5] and be on the same device");
  const Tensor means3D = f32c(means3D_, "means3D");
  const Options o(means3D.device());
  const c10::DeviceGuard guard(means3D.device());
  const int64_t M = sh_mode ? sh->size(1) : 0;
  Tensor dL_dsh = sh_mode ? at::empty({P, M, 3}, o.f32) : at::empty({P, 3}, o.f32);  // (the latter: zeros)
  Tensor dmeans = at::empty({P, 3}, o.f32), dscales = at::empty({P, 3}, o.f32), drot = at::empty({P, 4}, o.f32),
         dopacity = at::empty({P, 1}, o.f32);
  const Tensor g2 = f32c(dL_dmeans2D, "dL_dmeans2D"), gco = f32c(dL_dconic_opacity, "dL_dconic_opacity");
  Tensor gcol = sh_mode ? f32c(dL_dcolors, "dL_dcolors") : Tensor();
  if (sh_mode && !gcol.defined()) gcol = at::zeros({P, 3}, o.f32);
  const Tensor scales = f32c(scales_, "scales"), rotations = f32c(rotations_, "rotations");
  const Tensor vm = f32c(viewmatrix, "viewmatrix"), pm = f32c(projmatrix, "projmatrix"), cp = f32c(campos, "campos");
  const Tensor shc = sh_mode ? f32c(*sh, "sh") : Tensor();
  const Tensor cov3D = contiguous_or_none(cov3D_), rad = radii.contiguous(), cl = clamped.contiguous();
  const Tensor gmap = f32c(dL_dall_map, "dL_dall_map");
  int status;
  {
    py::gil_scoped_release nogil;
    status = gs_preprocess_rows_backward(
        ptr<int>(rad), ptr(cov3D), ptr<uint8_t>(cl), (int)P, degree, (int)M, width, height, ptr(means3D), ptr(scales),
        ptr(rotations), ptr(shc), scale_modifier, ptr(vm), ptr(pm), ptr(cp), tan_fovx, tan_fovy, ptr(g2),
        (int)g2.size(1), ptr(gco), ptr(gcol), ptr(dmeans), nullptr, ptr(dscales), ptr(drot),
        sh_mode ? ptr(dL_dsh) : nullptr, ptr(dopacity), debug,
        sh_mode && dcolor_ddir.has_value() ? ptr(*dcolor_ddir) : nullptr, ptr(gmap),
        sh_mode ? nullptr : ptr(dL_dsh), stream_of(stream));
  }
  check(status, "preprocess_gaussians_backward");
  return py::make_tuple(dmeans, dscales, drot, dL_dsh, dopacity);
}

// What the caller passes for "not given": None or an empty tensor, of whatever type.
OptTensor given(const OptTensor& t) { return t.has_value() && t->numel() != 0 ? t : OptTensor(); }

// Radii only.  Scales may be the first columns of wider rows, as the anchor model holds them: they are read where they lie.
Tensor visible_filter(const Tensor& means3D_, const OptTensor& scales_, const OptTensor& rotations_,
                      float scale_modifier, const OptTensor& cov3D_, const Tensor& viewmatrix, const Tensor& projmatrix,
                      float tan_fovx, float tan_fovy, int height, int width, bool prefiltered, bool debug,
                      uintptr_t stream) {
  const at::AutoDispatchBelowADInplaceOrView no_grad;  // (a copy made here is no part of a graph)
  const Tensor means3D = f32c(means3D_, "means3D");
  const int64_t P = means3D.size(0);
  const Options o(means3D.device());
  const c10::DeviceGuard guard(means3D.device());
  Tensor radii = at::empty({P}, o.i32);
  if (P == 0) return radii;
  OptTensor scales = given(scales_);
  int64_t stride = 3;
  if (scales.has_value()) {
    const Tensor& s = *scales;
    const bool in_place = s.scalar_type() == at::kFloat && s.is_cuda() && s.dim() == 2 && s.size(0) == P && s.size(1) == 3 &&
                          s.stride(1) == 1 && s.stride(0) >= 3 && s.stride(0) <= 1024;
    if (in_place) stride = s.stride(0);
    else scales = f32c(s, "scales");
  }
  const Tensor rot = f32c(given(rotations_), "rotations"), cov = f32c(given(cov3D_), "cov3D_precomp");
  const Tensor vm = f32c(viewmatrix, "viewmatrix"), pm = f32c(projmatrix, "projmatrix");
  int status;
  {
    py::gil_scoped_release nogil;  // (with debug the call waits for the kernel)
    status = gs_visible_filter_rows((int)P, (int)stride, width, height, ptr(means3D), scales ? ptr(*scales) : nullptr,
                                    scale_modifier, ptr(rot), ptr(cov), ptr(vm), ptr(pm), tan_fovx, tan_fovy, prefiltered,
                                    ptr<int>(radii), debug, stream_of(stream));
  }
  check(status, "rasterize_aussians_filter");
  return radii;
}

py::tuple render_forward(const Tensor& background, int H, int W, const Tensor& means2D_, const Tensor& depths_,
                         const Tensor& radii_, const Tensor& conic_opacity, const Tensor& rgb, const Tensor& locally,
                         float tan_fovx, float tan_fovy, const OptTensor& all_map, bool geo, bool debug,
                         bool want_max_weight_depth, bool timing, int small_limit, int block_records,
                         int64_t expected_instances, int expected_longest_list, int recent_longest_list,
                         const OptTensor& blend_records, uintptr_t stream) {
  const Tensor means2D = f32c(means2D_, "means2D");
  const int64_t P = means2D.size(0);
  const Options o(means2D.device());
  const c10::DeviceGuard guard(means2D.device());
  const int64_t tiles = ((H + TILE - 1) / TILE) * ((W + TILE - 1) / TILE);
  const Tensor bg = f32c(background, "background"), depths = f32c(depths_, "depths"),
               co = f32c(conic_opacity, "conic_opacity"), col = f32c(rgb, "rgb");
  const Tensor radii = radii_.contiguous();
  TORCH_CHECK_TYPE(radii.scalar_type() == at::kInt, "radii must be int32");
  const Tensor cl = locally.contiguous();
  TORCH_CHECK(cl.scalar_type() == at::kBool && cl.numel() == tiles, "compute_locally must be a bool tensor with ",
              tiles, " elements");
  TORCH_CHECK_TYPE(!geo || all_map.has_value(), "all_map must be a tensor where geometry channels are rendered");
  const Tensor am = geo ? f32c(*all_map, "all_map") : Tensor();
  check_rows(blend_records, "blend_records", means2D, {P, 16});
  Tensor color = at::empty({CHANNELS, H, W}, o.f32), observe = at::empty({P}, o.i32);
  // (zeros without geometry channels, cleared in the call)
  Tensor map = at::empty({MAP_CHANNELS, H, W}, o.f32), depth = at::empty({1, H, W}, o.f32);
  Tensor n_render = at::empty({tiles}, o.i32), n_consider = at::empty({tiles}, o.i32),
         n_contrib = at::empty({tiles}, o.i32);
  Tensor mwd = want_max_weight_depth ? at::empty({1, H, W}, o.f32) : Tensor();
  GrowBuffer geom(o.u8), binning(o.u8), img(o.u8);
  gs_render_options options = {};
  options.struct_bytes = sizeof(options);
  options.tile_sort_small_limit = small_limit;
  options.tile_sort_block_records = block_records;
  options.expected_longest_list = expected_longest_list;
  options.expected_instances = expected_instances;
  options.blend_records = blend_records.has_value() ? ptr(*blend_records) : nullptr;
  options.clear_geo_images = 1;
  options.recent_longest_list = recent_longest_list;
  gs_render_result result = {};
  result.struct_bytes = sizeof(result);
  // fp32 arithmetic, as `H / (2.0f * tan_fovy)` at rasterize_points.cu:328-329
  const float focal_x = (float)W / (2.0f * tan_fovx), focal_y = (float)H / (2.0f * tan_fovy);
  int num_rendered = 0, status;
  float elapsed = 0.f;
  {
    py::gil_scoped_release nogil;
    status = gs_render_forward(
        &GrowBuffer::resize, &geom, &GrowBuffer::resize, &binning, &GrowBuffer::resize, &img, (int)P, ptr(bg), W, H,
        focal_x, focal_y, (float)(W * 0.5), (float)(H * 0.5), nullptr, nullptr, ptr(am), ptr(means2D), ptr(depths),
        ptr<int>(radii), ptr(co), ptr(col), ptr<uint8_t>(cl), ptr(color), ptr<int>(n_render), ptr<int>(n_consider),
        ptr<int>(n_contrib), ptr<int>(observe), ptr(map), ptr(depth), ptr(mwd), geo, debug, &num_rendered,
        timing ? &elapsed : nullptr, &options, &result, stream_of(stream));
  }
  for (const GrowBuffer* b : {&geom, &binning, &img})
    if (b->failure) std::rethrow_exception(b->failure);
  check(status, "render_gaussians");
  return py::make_tuple(num_rendered, color, n_render, n_consider, n_contrib, observe, map, depth, geom.tensor,
                        binning.tensor, img.tensor, result.longest_list, result.binning_capacity,
                        result.launched_ahead != 0, elapsed, some(mwd));
}

py::tuple render_backward(const Tensor& background, float tan_fovx, float tan_fovy, const OptTensor& all_map_pixels,
                          const OptTensor& all_maps, int R, const Tensor& geom, const Tensor& binning,
                          const Tensor& img, const Tensor& locally, const Tensor& dL_dout_color,
                          const OptTensor& dL_dout_all_map, const OptTensor& dL_dout_plane_depth,
                          const Tensor& means2D_, const Tensor& conic_opacity, const Tensor& rgb, bool geo, bool debug,
                          bool timing, int64_t binning_capacity, const OptTensor& blend_records, uintptr_t stream) {
  const int64_t P = means2D_.size(0);
  check_rows(blend_records, "blend_records", means2D_, {P, 16});
  const Tensor means2D = f32c(means2D_, "means2D");
  const Options o(means2D.device());
  const c10::DeviceGuard guard(means2D.device());
  const int H = (int)dL_dout_color.size(1), W = (int)dL_dout_color.size(2);
  Tensor d2 = at::empty({P, 2}, o.f32), dabs = at::empty({P, 3}, o.f32), dco = at::empty({P, 4}, o.f32),
         dcol = at::empty({P, CHANNELS}, o.f32), dmap = at::empty({P, MAP_CHANNELS}, o.f32);
  const size_t ws_bytes = gs_render_backward_sparse_workspace_bytes(R);
  const Tensor workspace = at::empty({(int64_t)ws_bytes}, o.u8);
  const Tensor bg = f32c(background, "background"), gpix = f32c(dL_dout_color, "dL_dout_color");
  TORCH_CHECK_TYPE(!geo || (dL_dout_all_map && dL_dout_plane_depth && all_map_pixels && all_maps),
                   "geometry channels need all_maps, all_map_pixels and their gradients");
  const Tensor gmap = geo ? f32c(dL_dout_all_map, "dL_dout_all_map") : Tensor(),
               gdep = geo ? f32c(dL_dout_plane_depth, "dL_dout_plane_depth") : Tensor(),
               amp = geo ? f32c(all_map_pixels, "all_map_pixels") : Tensor(),
               am = geo ? f32c(all_maps, "all_maps") : Tensor();
  const Tensor co = f32c(conic_opacity, "conic_opacity"), col = f32c(rgb, "rgb"), cl = locally.contiguous();
  int status;
  float elapsed = 0.f;
  {
    py::gil_scoped_release nogil;
    status = gs_render_backward(
        (int)P, R, ptr(bg), W, H, tan_fovx, tan_fovy, ptr<char>(geom), ptr<char>(binning), ptr<char>(img),
        ptr<uint8_t>(cl), ptr(gpix), ptr(gmap), ptr(gdep), ptr(d2), ptr(dabs), ptr(dco), ptr(dcol), ptr(dmap),
        ptr(means2D), ptr(co), ptr(col), ptr(am), ptr(amp), geo, debug, ptr(workspace), ws_bytes,
        timing ? &elapsed : nullptr, binning_capacity, blend_records.has_value() ? ptr(*blend_records) : nullptr,
        stream_of(stream));
  }
  check(status, "render_gaussians_backward");
  return py::make_tuple(d2, dabs, dco, dcol, dmap, elapsed);
}

// ---------------------------------------------------------------- loss maps --

Tensor image(const Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 3, name, " must be (channels, height, width)");
  TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, name, " must be float32, got ", t.scalar_type());
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor: there is no CPU path");
  return t.contiguous();
}

py::tuple ssim_l1_forward(const Tensor& img1, const Tensor& img2, const OptTensor& pixel_mask, bool need,
                          uintptr_t stream) {
  const Tensor a = image(img1, "img1"), b = image(img2, "img2");
  TORCH_CHECK(a.sizes() == b.sizes(), "img1 and img2 must have the same shape");
  const int64_t C = a.size(0), H = a.size(1), W = a.size(2);
  Tensor m;
  if (pixel_mask.has_value()) {
    TORCH_CHECK(pixel_mask->dim() == 2 && pixel_mask->size(0) == H && pixel_mask->size(1) == W &&
                    (pixel_mask->scalar_type() == at::kBool || pixel_mask->scalar_type() == at::kByte) &&
                    pixel_mask->is_cuda(),
                "pixel_mask must be a (height, width) bool GPU tensor");
    m = pixel_mask->contiguous();
  }
  Tensor l1 = at::empty_like(a), ssim = at::empty_like(a), d_mu, d_xx, d_xy;
  if (need) {
    d_mu = at::empty_like(a);
    d_xx = at::empty_like(a);
    d_xy = at::empty_like(a);
  }
  check(gs_ssim_l1_forward((int)C, (int)H, (int)W, ptr(a), ptr(b), ptr<uint8_t>(m), ptr(l1), ptr(ssim), ptr(d_mu),
                           ptr(d_xx), ptr(d_xy), stream_of(stream)),
        "pixelwise_l1_ssim_with_mask");
  return py::make_tuple(l1, ssim, a, b, some(m), some(d_mu), some(d_xx), some(d_xy));
}

Tensor ssim_l1_backward(const Tensor& a, const Tensor& b, const OptTensor& m, const OptTensor& g_l1,
                        const OptTensor& g_ssim, const Tensor& d_mu, const Tensor& d_xx, const Tensor& d_xy,
                        uintptr_t stream) {
  const Tensor g1 = g_l1.has_value() ? image(*g_l1, "grad of l1 map") : Tensor(),
               g2 = g_ssim.has_value() ? image(*g_ssim, "grad of ssim map") : Tensor();
  Tensor out = at::empty_like(a);
  check(gs_ssim_l1_backward((int)a.size(0), (int)a.size(1), (int)a.size(2), ptr(a), ptr(b),
                            m.has_value() ? ptr<uint8_t>(*m) : nullptr, ptr(g1), ptr(g2), ptr(d_mu), ptr(d_xx),
                            ptr(d_xy), ptr(out), stream_of(stream)),
        "pixelwise_l1_ssim_with_mask backward");
  return out;
}

// ----------------------------------------------------------- neural Gaussians --

Tensor shaped(const Tensor& t, const char* name, at::IntArrayRef shape) {
  TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, name, " must be float32, got ", t.scalar_type());
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor: there is no CPU path");
  TORCH_CHECK(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes());
  return t.contiguous();
}

// W1, b1, W2, b2 of the opacity, color and cov MLPs
std::vector<Tensor> mlp_params(const std::vector<Tensor>& params, int64_t k, int input_flags) {
  TORCH_CHECK(params.size() == 12, "expected W1, b1, W2, b2 of the opacity, color and cov MLPs (12 tensors)");
  const int64_t outs[3] = {k, 3 * k, 7 * k};
  std::vector<Tensor> r;
  r.reserve(12);
  for (int m = 0; m < 3; m++) {
    const int64_t in = 35 + ((input_flags >> m) & 1) + ((input_flags >> 3) & 1);
    r.push_back(shaped(params[4 * m], "MLP W1", {32, in}));
    r.push_back(shaped(params[4 * m + 1], "MLP b1", {32}));
    r.push_back(shaped(params[4 * m + 2], "MLP W2", {outs[m], 32}));
    r.push_back(shaped(params[4 * m + 3], "MLP b2", {outs[m]}));
  }
  return r;
}

std::vector<float*> table(const std::vector<Tensor>& ts) {
  std::vector<float*> r;
  r.reserve(ts.size());
  for (const Tensor& t : ts) r.push_back(ptr(t));
  return r;
}

py::tuple neural_forward(const Tensor& anchor_, const Tensor& feat_, const Tensor& offsets_, const Tensor& scaling_,
                         const Tensor& campos_, const OptTensor& opacity_scale_, const OptTensor& level_,
                         int input_flags, const std::vector<Tensor>& params_, uintptr_t stream) {
  const int64_t N = anchor_.size(0), k = offsets_.size(1);
  const Tensor anchor = shaped(anchor_, "anchor", {N, 3}), feat = shaped(feat_, "feat", {N, 32}),
               offsets = shaped(offsets_, "offsets", {N, k, 3}), scaling = shaped(scaling_, "scaling", {N, 6}),
               campos = shaped(campos_, "camera_center", {3});
  const Tensor opacity_scale = opacity_scale_ ? shaped(opacity_scale_->detach(), "opacity_scale", {N}) : Tensor();
  TORCH_CHECK(!(input_flags & 8) || level_.has_value(), "input_flags asks for the level input");
  const Tensor level = input_flags & 8 ? shaped(level_->detach().reshape(-1), "level", {N}) : Tensor();
  const std::vector<Tensor> params = mlp_params(params_, k, input_flags);
  const Options o(anchor.device());
  Tensor neural_opacity = at::empty({N * k, 1}, o.f32), mask = at::empty({N * k}, o.b8),
         first = at::empty({std::max<int64_t>(N, 1)}, o.i32);
  // with a factor on the opacity the backward pass needs the MLP's own output as well
  Tensor opacity_tanh = opacity_scale.defined() ? at::empty({N * k}, o.f32) : Tensor();
  const size_t ws_bytes = gs_neural_workspace_bytes(N, (int)k);
  const Tensor ws = at::empty({(int64_t)ws_bytes}, o.u8);
  const std::vector<float*> weights = table(params);
  int64_t S = 0;
  int status;
  {
    py::gil_scoped_release nogil;  // (waits for the number of selected offsets)
    status = gs_neural_opacity_forward(N, (int)k, ptr(anchor), ptr(feat), ptr(campos), weights.data(),
                                       ptr(opacity_scale), ptr(level), input_flags, ptr(neural_opacity),
                                       ptr(opacity_tanh), ptr<uint8_t>(mask), ptr<uint32_t>(first), ptr<void>(ws),
                                       ws_bytes, &S, stream_of(stream));
  }
  check(status, "generate_neural_gaussians");
  Tensor xyz = at::empty({S, 3}, o.f32), color = at::empty({S, 3}, o.f32), opacity = at::empty({S, 1}, o.f32),
         scal = at::empty({S, 3}, o.f32), rot = at::empty({S, 4}, o.f32), aux = at::empty({S, 4}, o.f32);
  check(gs_neural_gaussians_forward(N, (int)k, S, ptr(anchor), ptr(feat), ptr(offsets), ptr(scaling), ptr(campos),
                                    ptr(level), ptr(neural_opacity), ptr<uint32_t>(first), ptr<void>(ws), ws_bytes,
                                    ptr(xyz), ptr(color), ptr(opacity), ptr(scal), ptr(rot), ptr(aux),
                                    stream_of(stream)),
        "generate_neural_gaussians");
  return py::make_tuple(py::make_tuple(xyz, color, opacity, scal, rot, neural_opacity, mask),
                        py::make_tuple(anchor, feat, offsets, scaling, campos, neural_opacity, first, color, rot, aux),
                        params, some(opacity_scale), some(level), some(opacity_tanh));
}

py::tuple neural_backward(const Tensor& anchor, const Tensor& feat, const Tensor& offsets, const Tensor& scaling,
                          const Tensor& campos, const Tensor& neural_opacity, const Tensor& first, const Tensor& color,
                          const Tensor& rot, const Tensor& aux, const std::vector<Tensor>& params,
                          const OptTensor& opacity_scale, const OptTensor& level, int input_flags,
                          const OptTensor& opacity_tanh, const std::vector<OptTensor>& grads, uintptr_t stream) {
  const int64_t N = anchor.size(0), k = offsets.size(1), S = color.size(0);
  const Options o(anchor.device());
  const int64_t widths[5] = {3, 3, 1, 3, 4};
  TORCH_CHECK(grads.size() == 5, "expected five upstream gradients");
  Tensor g[5];
  for (int i = 0; i < 5; i++)
    g[i] = grads[i].has_value() ? shaped(*grads[i], "upstream gradient", {S, widths[i]})
                                : at::zeros({S, widths[i]}, o.f32);
  Tensor d_anchor = at::empty_like(anchor), d_feat = at::empty_like(feat), d_offsets = at::empty_like(offsets),
         d_scaling = at::empty_like(scaling);
  std::vector<Tensor> d_params;
  d_params.reserve(12);
  for (const Tensor& p : params) d_params.push_back(at::empty_like(p));
  const size_t ws_bytes = gs_neural_backward_workspace_bytes(N, (int)k);
  const Tensor ws = at::empty({(int64_t)ws_bytes}, o.u8);
  const std::vector<float*> weights = table(params), d_weights = table(d_params);
  const auto given = [](const OptTensor& t) { return t.has_value() ? ptr(*t) : nullptr; };
  check(gs_neural_backward(N, (int)k, S, ptr(anchor), ptr(feat), ptr(offsets), ptr(scaling), ptr(campos),
                           weights.data(), given(opacity_scale), given(level), input_flags, ptr(neural_opacity),
                           given(opacity_tanh), ptr<uint32_t>(first), ptr(color), ptr(rot), ptr(aux), ptr(g[0]),
                           ptr(g[1]), ptr(g[2]), ptr(g[3]), ptr(g[4]), ptr(d_anchor), ptr(d_feat), ptr(d_offsets),
                           ptr(d_scaling), d_weights.data(), ptr<void>(ws), ws_bytes, stream_of(stream)),
        "generate_neural_gaussians backward");
  py::tuple out(4 + d_params.size());
  const Tensor first4[4] = {d_anchor, d_feat, d_offsets, d_scaling};
  for (size_t i = 0; i < 4; i++) out[i] = py::cast(first4[i]);
  for (size_t i = 0; i < d_params.size(); i++) out[4 + i] = py::cast(d_params[i]);
  return out;
}

// (the caller has looked at types, shapes and strides)
py::tuple visible_rows(const Tensor& mask, const Tensor& anchor, const Tensor& feat, const Tensor& offsets,
                       const Tensor& scaling, bool want_index, uintptr_t stream) {
  const int64_t A = offsets.size(0), k = offsets.size(1);
  const Options o(anchor.device());
  const size_t nb = gs_visible_rows_workspace_bytes(A);
  const Tensor ws = at::empty({(int64_t)nb / 4}, o.i32);
  int64_t N = 0;
  int status;
  {
    py::gil_scoped_release nogil;  // (waits for the number of rows)
    status = gs_visible_rows_count(A, ptr<uint8_t>(mask), ptr<void>(ws), nb, &N, stream_of(stream));
  }
  check(status, "visible rows");
  Tensor a = at::empty({N, 3}, o.f32), f = at::empty({N, 32}, o.f32), d = at::empty({N, k, 3}, o.f32),
         s = at::empty({N, 6}, o.f32), rank = at::empty({A}, o.i32);
  Tensor index = want_index ? at::empty({N}, o.i64) : Tensor();
  check(gs_visible_rows_gather(A, (int)k, N, ptr<uint8_t>(mask), ptr<void>(ws), nb, ptr(anchor), ptr(feat),
                               ptr(offsets), ptr(scaling), ptr(a), ptr(f), ptr(d), ptr(s), ptr<uint32_t>(rank),
                               ptr<int64_t>(index), stream_of(stream)),
        "visible rows");
  return py::make_tuple(a, f, d, s, some(index), rank);
}

py::tuple visible_rows_backward(const Tensor& rank, int64_t k, const std::vector<OptTensor>& grads,
                                uintptr_t stream) {
  const int64_t A = rank.size(0);
  const Options o(rank.device());
  const std::vector<int64_t> shapes[4] = {{A, 3}, {A, 32}, {A, k, 3}, {A, 6}};
  TORCH_CHECK(grads.size() == 4, "expected four gradients");
  Tensor g[4], d[4];
  for (int i = 0; i < 4; i++) {
    if (!grads[i].has_value()) continue;
    g[i] = f32c(*grads[i], "gradient");
    d[i] = at::empty(shapes[i], o.f32);
  }
  if (g[1].defined() && ((uintptr_t)g[1].data_ptr() & 15)) g[1] = g[1].clone();  // (read 16 bytes at a time)
  check(gs_visible_rows_spread(A, (int)k, ptr<uint32_t>(rank), ptr(g[0]), ptr(g[1]), ptr(g[2]), ptr(g[3]), ptr(d[0]),
                               ptr(d[1]), ptr(d[2]), ptr(d[3]), stream_of(stream)),
        "visible rows backward");
  return py::make_tuple(some(d[0]), some(d[1]), some(d[2]), some(d[3]));
}

}  // namespace

PYBIND11_MODULE(gsrast_ops, m) {
  m.def("preprocess_forward", &preprocess_forward);
  m.def("preprocess_backward", &preprocess_backward);
  m.def("visible_filter", &visible_filter);
  m.def("render_forward", &render_forward);
  m.def("render_backward", &render_backward);
  m.def("ssim_l1_forward", &ssim_l1_forward);
  m.def("ssim_l1_backward", &ssim_l1_backward);
  m.def("neural_forward", &neural_forward);
  m.def("neural_backward", &neural_backward);
  m.def("visible_rows", &visible_rows);
  m.def("visible_rows_backward", &visible_rows_backward);
}
