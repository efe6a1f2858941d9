"""The work a user of this framework has it do, as measurable cases: training views (forward and backward), rendering,
neural-Gaussian generation, the loss maps, the optimizer step, the densification statistics and the k-NN
initialiser, each through its public entry points.

Scenes are synthetic, made on the GPU from the seed: the five layouts of the repository's benchmark configurations
(a block of Gaussians, an oblique aerial view, high aerial views over a city, street level, and the 20 M city from
600 m), with the Gaussians' size following their number so that a layout is covered alike at every size.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "citygs-x_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda:0"

# layout: number of Gaussians its figures are quoted for, mean and sigma of the log scale, horizontal field of view,
# and the Gaussians a pixel blends (measured, for the operation counts below)
LAYOUTS = {
    "block": (50_000, -4.0, 0.5, 60.0, 2.4),
    "oblique": (1_000_000, -2.5, 0.7, 70.0, 18.5),
    "aerial": (4_000_000, -2.0, 0.8, 70.0, 22.0),
    "street": (10_000_000, -2.0, 0.8, 90.0, 14.0),
    "city": (20_000_000, -2.0, 0.8, 70.0, 30.0),
}


def listed():
    return [
        # the first iterations of a small scene, or a preview: launches and latency count
        dict(name="train_50k_640x480", kind="train", layout="block", P=50_000, W=640, H=480, geo=True, sh=True),
        # the headline workload: one view of a training step, geometry channels built inside it
        dict(name="train_1m_1152x864", kind="train", layout="oblique", P=1_000_000, W=1152, H=864, geo=True, sh=True),
        # a grown scene seen from the air, lists of several thousand Gaussians per tile
        dict(name="train_4m_1152x864", kind="train", layout="aerial", P=4_000_000, W=1152, H=864, geo=True, sh=True),
        # street level at full HD: most Gaussians out of view, a few covering thousands of tiles
        dict(name="train_10m_1920x1080", kind="train", layout="street", P=10_000_000, W=1920, H=1080, geo=True,
             sh=True),
        # the early iterations of a run before the geometry losses set in, colours from the caller (an MLP's), an
        # image that is no multiple of the tile
        dict(name="train_rgb_300k_1237x822", kind="train", layout="oblique", P=300_000, W=1237, H=822, geo=False,
             sh=False),
        # evaluation: a view rendered without gradients
        dict(name="render_1m_1152x864", kind="render", layout="oblique", P=1_000_000, W=1152, H=864, geo=True,
             sh=True),
        # the largest scene, rendered from 600 m, colour only, as a viewer does
        dict(name="render_20m_1152x864", kind="render", layout="city", P=20_000_000, W=1152, H=864, geo=False,
             sh=True),
        # anchors of a scaffold model: the visible ones, their neural Gaussians and the gradients of both
        dict(name="neural_500k_anchors", kind="neural", A=500_000, k=10, W=1152, H=864),
        # the two loss maps of one training image and their gradient
        dict(name="loss_1152x864", kind="loss", W=1152, H=864),
        # one optimizer step over all parameters of 1 M Gaussians
        dict(name="adam_1m", kind="adam", P=1_000_000),
        # densification statistics after one view of 1 M anchors
        dict(name="stats_1m_anchors", kind="stats", A=1_000_000, k=10),
        # the initial scale of every point of an SfM cloud
        dict(name="knn_1m", kind="knn", P=1_000_000),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("train", "train", "train", "render", "neural", "loss", "adam", "stats", "knn"))
    if kind in ("train", "render"):
        layout = rng.choice(("block", "oblique", "aerial", "street"))
        top = {"block": 300_000, "oblique": 3_000_000, "aerial": 5_000_000, "street": 8_000_000}[layout]
        return dict(kind=kind, layout=layout, P=_log_uniform(rng, 20_000, top), W=rng.randint(320, 1920),
                    H=rng.randint(240, 1080), geo=rng.random() < 0.7, sh=rng.random() < 0.7)
    if kind == "neural":
        return dict(kind=kind, A=_log_uniform(rng, 10_000, 1_000_000), k=rng.choice((4, 10)), W=rng.randint(320, 1920),
                    H=rng.randint(240, 1080))
    if kind == "loss":
        return dict(kind=kind, W=rng.randint(160, 1920), H=rng.randint(120, 1080))
    if kind == "adam":
        return dict(kind=kind, P=_log_uniform(rng, 20_000, 3_000_000))
    if kind == "stats":
        return dict(kind=kind, A=_log_uniform(rng, 20_000, 2_000_000), k=rng.choice((5, 10)))
    return dict(kind=kind, P=_log_uniform(rng, 10_000, 4_000_000))


# ------------------------------------------------------------------ inputs --

class _Draws:
    """Random tensors on the GPU from one seeded generator."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)

    def u(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=DEV)

    def n(self, *shape):
        return torch.randn(*shape, generator=self.gen, device=DEV)


def _camera(eye, target, W, H, fovx_deg, up):
    """World-to-camera and projection in the row-vector convention of the operator, and the settings' scalars."""
    d = torch.float64
    eye, target, up = (torch.tensor(v, dtype=d) for v in (eye, target, up))
    f = torch.nn.functional.normalize(target - eye, dim=0)
    x = torch.nn.functional.normalize(torch.linalg.cross(f, up), dim=0)
    y = torch.linalg.cross(f, x)
    view = torch.eye(4, dtype=d)
    view[:3, 0], view[:3, 1], view[:3, 2] = x, y, f
    view[3, :3] = -(eye @ view[:3, :3])
    tanx = math.tan(math.radians(fovx_deg) / 2)
    tany = tanx * H / W
    near, far = 0.01, 100.0
    proj = torch.zeros(4, 4, dtype=d)
    proj[0, 0], proj[1, 1] = 1 / tanx, 1 / tany
    proj[2, 2], proj[2, 3], proj[3, 2] = far / (far - near), 1.0, -far * near / (far - near)
    return (view.float().to(DEV), (view @ proj).float().to(DEV), eye.float().to(DEV), tanx, tany)


def _view(layout, seed, W, H):
    """One camera of the layout; its place on the layout's path follows the seed, as the views of a batch do."""
    fov = LAYOUTS[layout][3]
    a = 2 * math.pi * ((int(seed) * 0.618033988749895) % 1.0)
    if layout == "block":
        return _camera((30 * math.sin(a), 0.0, -30 * math.cos(a)), (0.0, 0.0, 0.0), W, H, fov, (0.0, -1.0, 0.0))
    if layout == "oblique":
        return _camera((120 * math.sin(a), -120 * math.cos(a), 120.0), (0.0, 0.0, 0.0), W, H, fov, (0.0, 0.0, 1.0))
    if layout == "aerial":
        return _camera((300 * math.cos(a), 300 * math.sin(a), 175 + 25 * math.sin(a)), (0.0, 0.0, 0.0), W, H, fov,
                       (0.0, 0.0, 1.0))
    if layout == "street":
        p = (300 * math.cos(3 * a), 300 * math.sin(5 * a), 2.0)
        return _camera(p, (p[0] + math.cos(a), p[1] + math.sin(a), 2.0), W, H, fov, (0.0, 0.0, 1.0))
    return _camera((600 * math.cos(a), 600 * math.sin(a), 200.0), (0.0, 0.0, 0.0), W, H, fov, (0.0, 0.0, 1.0))


def _means(r, layout, P):
    u = r.u(P, 3)
    if layout == "block":
        return (u * 2 - 1) * 10.0
    if layout == "oblique":
        return (u - torch.tensor([0.5, 0.5, 0.0], device=DEV)) * torch.tensor([200.0, 200.0, 30.0], device=DEV)
    if layout == "aerial":
        z = torch.where(r.u(P) < 0.7, r.n(P) * 3.0 + 2.0, u[:, 2] * 60.0)
        return torch.stack([(u[:, 0] - 0.5) * 1000.0, (u[:, 1] - 0.5) * 1000.0, z], 1)
    z = u[:, 2] * torch.where(r.u(P) < 1.0 / 9.0, 10.0, 80.0)
    return torch.stack([(u[:, 0] - 0.5) * 2000.0, (u[:, 1] - 0.5) * 2000.0, z], 1)


def _gaussians(r, layout, P, sh):
    P0, mu, sigma = LAYOUTS[layout][:3]
    g = {"means3D": _means(r, layout, P),
         "scales": torch.exp(r.n(P, 3) * sigma + (mu + 0.5 * math.log(P0 / P))),
         "rotations": torch.nn.functional.normalize(r.n(P, 4)),
         "opacities": torch.sigmoid(r.n(P, 1) * (1.0 if layout == "block" else 1.5))}
    if sh:
        g["shs"] = torch.cat([r.n(P, 1, 3) * 0.3, r.n(P, 15, 3) * 0.05], 1)
    else:
        g["colors"] = r.u(P, 3)
    return g


# ----------------------------------------------------------- rasterizer views --

def _prepare_view(c, seed, train):
    from diff_gaussian_rasterization import GaussianRasterizationSettings, GaussianRasterizer
    r = _Draws(seed)
    P, W, H = c["P"], c["W"], c["H"]
    g = _gaussians(r, c["layout"], P, c["sh"])
    vm, pm, pos, tanx, tany = _view(c["layout"], seed, W, H)
    rs = GaussianRasterizationSettings(
        image_height=H, image_width=W, tanfovx=tanx, tanfovy=tany, bg=torch.zeros(3, device=DEV), scale_modifier=1.0,
        viewmatrix=vm, projmatrix=pm, sh_degree=3, campos=pos, prefiltered=False, render_geo=c["geo"], debug=False)
    s = {"geo": c["geo"], "sh": c["sh"], "rs": rs, "rast": GaussianRasterizer(rs),
         "mask": torch.ones((H + 15) // 16, (W + 15) // 16, dtype=torch.bool, device=DEV),
         "args": {"avoid_pixel_all2all": False, "stats_collector": {}}, "train": train}
    s["leaf"] = {k: v.contiguous().requires_grad_(train) for k, v in g.items()}
    s["m2abs"] = torch.zeros(P, 3, device=DEV, requires_grad=train)
    s["no_map"] = torch.zeros(P, 5, device=DEV)
    if train:
        # what the losses leave on the images: gradients of unit size on colour and channels, and on the depth those
        # of a loss on inverse depth (the depth itself is unbounded where a surface is seen edge-on)
        s["up"] = [r.n(3, H, W)]
        if c["geo"]:
            with torch.no_grad():
                z = _forward(s)["depth"]
            w = torch.where(z.abs() > 1e-2, z, torch.full_like(z, math.inf))
            s["up"] += [r.n(5, H, W), r.n(1, H, W) / (w * w)]
    return s


def _forward(s):
    from diff_gaussian_rasterization import build_all_map
    leaf, rast, rs = s["leaf"], s["rast"], s["rs"]
    means2D, rgb, co, radii, depths = rast.preprocess_gaussians(
        leaf["means3D"], leaf["scales"], leaf["rotations"], leaf["shs"] if s["sh"] else leaf["colors"],
        leaf["opacities"], s["args"])
    all_map = (build_all_map(leaf["means3D"], leaf["scales"], leaf["rotations"], rs.viewmatrix, rs.campos,
                             blend_records_of=means2D) if s["geo"] else s["no_map"])
    color, n_render, n_consider, n_contrib, observe, omap, depth = rast.render_gaussians(
        means2D, s["m2abs"], co, rgb if s["sh"] else leaf["colors"], all_map, depths, radii, s["mask"], s["mask"],
        s["args"])
    out = {"color": color, "radii": radii, "n_render": n_render, "n_contrib": n_contrib, "observe": observe}
    if s["geo"]:
        out["all_map"], out["depth"] = omap, depth
    return out


def _run_view(s):
    if not s["train"]:
        with torch.no_grad():
            return _forward(s)
    for t in list(s["leaf"].values()) + [s["m2abs"]]:
        t.grad = None
    out = _forward(s)
    images = [out["color"]] + ([out["all_map"], out["depth"]] if s["geo"] else [])
    torch.autograd.backward(images, s["up"])
    out = {k: v.detach() for k, v in out.items()}
    out.update({"d_" + k: t.grad for k, t in s["leaf"].items()})
    out["d_means2D_abs"] = s["m2abs"].grad
    return out


# --------------------------------------------------------- neural Gaussians --

class _Anchors:
    """The parts of the anchor model that the generation step reads."""
    add_opacity_dist = add_color_dist = add_cov_dist = add_level = use_feat_bank = False
    dist2level, appearance_dim = "round", 0

    def __init__(self, r, A, k):
        self.get_anchor = ((r.u(A, 3) - 0.5) * torch.tensor([400.0, 400.0, 40.0], device=DEV)).requires_grad_()
        self.get_anchor_feat = (r.n(A, 32) * 0.7).requires_grad_()
        self._offset = (r.n(A, k, 3) * 0.5).requires_grad_()
        self.get_scaling = torch.exp(r.n(A, 6) * 0.4 - 1.0).requires_grad_()
        self.rotations = torch.zeros(A, 4, device=DEV)
        self.rotations[:, 0] = 1.0

        def mlp(out):
            m = torch.nn.Sequential(torch.nn.Linear(35, 32), torch.nn.ReLU(), torch.nn.Linear(32, out)).to(DEV)
            with torch.no_grad():
                for p, fan in zip(m.parameters(), (35, 35, 32, 32)):
                    p.copy_((r.u(*p.shape) * 2 - 1) / math.sqrt(fan))
            return m

        self.get_opacity_mlp, self.get_color_mlp, self.get_cov_mlp = mlp(k), mlp(3 * k), mlp(7 * k)
        # half of a visible anchor's candidates end up opaque, as in a trained model (about 45 %); with the second
        # half of the opacities the negatives of the first it is exactly half, so that outputs have one shape
        with torch.no_grad():
            for p in (self.get_opacity_mlp[2].weight, self.get_opacity_mlp[2].bias):
                p[k // 2:] = -p[:k // 2]

    def parameters(self):
        return [self.get_anchor, self.get_anchor_feat, self._offset, self.get_scaling] + [
            p for m in (self.get_opacity_mlp, self.get_color_mlp, self.get_cov_mlp) for p in m.parameters()]


class _Viewpoint:
    uid = 0

    def __init__(self, camera_center):
        self.camera_center = camera_center


def _visible(c):
    return int(0.35 * c["A"])


def _prepare_neural(c, seed):
    from diff_gaussian_rasterization import GaussianRasterizationSettings, GaussianRasterizer
    r = _Draws(seed)
    vm, pm, pos, tanx, tany = _view("oblique", seed, c["W"], c["H"])
    rs = GaussianRasterizationSettings(
        image_height=c["H"], image_width=c["W"], tanfovx=tanx, tanfovy=tany, bg=torch.zeros(3, device=DEV),
        scale_modifier=1.0, viewmatrix=vm, projmatrix=pm, sh_degree=3, campos=pos, prefiltered=False, render_geo=True,
        debug=False)
    model = _Anchors(r, c["A"], c["k"])
    # the anchors the view shows: the 35 % nearest to its axis
    p = model.get_anchor.detach() @ vm[:3, :3] + vm[3, :3]
    off_axis = torch.where(p[:, 2] > 0.1, p[:, :2].norm(dim=1) / p[:, 2], torch.full_like(p[:, 2], math.inf))
    visible = torch.zeros(c["A"], dtype=torch.bool, device=DEV)
    visible[off_axis.argsort(stable=True)[:_visible(c)]] = True
    n = _visible(c) * c["k"] // 2
    return {"model": model, "visible": visible, "camera": _Viewpoint(pos), "rast": GaussianRasterizer(rs),
            "up": [r.n(n, w) for w in (3, 3, 1, 3, 4)]}


def _run_neural(s):
    from gs_neural import generate_neural_gaussians
    m = s["model"]
    for p in m.parameters():
        p.grad = None
    radii = s["rast"].visible_filter(m.get_anchor, m.get_scaling[:, :3], m.rotations)
    out = generate_neural_gaussians(s["camera"], m, s["visible"], is_training=True)
    torch.autograd.backward(list(out[:5]), s["up"])
    return [radii] + [t.detach() for t in out] + [p.grad for p in m.parameters()]


# --------------------------------------------- loss, optimizer, statistics, k-NN --

def _prepare_loss(c, seed):
    r = _Draws(seed)
    W, H = c["W"], c["H"]
    coarse = r.u(1, 3, H // 16 + 2, W // 16 + 2)
    gt = torch.nn.functional.interpolate(coarse, size=(H, W), mode="bilinear", align_corners=False)[0]
    gt = (gt + r.n(3, H, W) * 0.03).clamp(0, 1).contiguous()
    img = (gt + r.n(3, H, W) * 0.05).clamp(0, 1).contiguous().requires_grad_()
    return {"img": img, "gt": gt, "mask": r.u(H, W) < 0.9,
            "up": [torch.full((3, H, W), 0.8 / (3 * H * W), device=DEV),
                   torch.full((3, H, W), -0.2 / (3 * H * W), device=DEV)]}


def _run_loss(s):
    from gs_loss import pixelwise_l1_ssim_with_mask
    s["img"].grad = None
    l1, ssim = pixelwise_l1_ssim_with_mask(s["img"], s["gt"], s["mask"])
    torch.autograd.backward([l1, ssim], s["up"])
    return {"l1": l1.detach(), "ssim": ssim.detach(), "d_img": s["img"].grad}


def _prepare_adam(c, seed):
    from gs_optim import FusedAdam
    r = _Draws(seed)
    shapes = {"xyz": ((3,), 1.6e-4), "f": ((16, 3), 2.5e-3), "opacity": ((1,), 5e-2), "scaling": ((3,), 5e-3),
              "rotation": ((4,), 1e-3)}
    groups = []
    for name, (shape, lr) in shapes.items():
        p = torch.nn.Parameter(r.n(c["P"], *shape))
        p.grad = r.n(c["P"], *shape) * 1e-3
        groups.append({"params": [p], "lr": lr, "name": name})
    return {"opt": FusedAdam(groups, lr=0.0, eps=1e-15)}


def _run_adam(s):
    opt = s["opt"]
    opt.step()
    params = [g["params"][0] for g in opt.param_groups]
    return [[p.detach(), opt.state[p]["exp_avg"], opt.state[p]["exp_avg_sq"]] for p in params]


def _prepare_stats(c, seed):
    # two fifths of the anchors visible, three fifths of their candidates selected, nine tenths of those kept
    r = _Draws(seed)
    A, k = c["A"], c["k"]
    vis = r.u(A) < 0.4
    sel = r.u(int(vis.sum()) * k) < 0.6
    flt = r.u(int(sel.sum())) < 0.9
    return {"k": k, "vis": vis, "sel": sel, "flt": flt, "grad": r.n(flt.numel(), 3) * 1e-3, "op": r.n(sel.numel(), 1),
            "acc": [torch.zeros(n, 1, device=DEV) for n in (A, A, A * k, A * k)]}


def _run_stats(s):
    from gs_densify import training_statis
    training_statis(*s["acc"], s["k"], s["grad"], s["op"], s["flt"], s["sel"], s["vis"])
    return s["acc"]


def _prepare_knn(c, seed):
    # an SfM cloud: most points on surfaces (ground and facades) and in clusters, some anywhere
    r = _Draws(seed)
    P = c["P"]
    u = r.u(P, 3)
    which = r.u(P)
    ground = torch.stack([u[:, 0] * 200, u[:, 1] * 200, r.n(P) * 0.05], 1)
    facade = torch.stack([torch.floor(u[:, 0] * 20) * 10 + r.n(P) * 0.05, u[:, 1] * 200, u[:, 2] * 30], 1)
    centres = r.u(512, 3) * torch.tensor([200.0, 200.0, 30.0], device=DEV)
    near = centres[(u[:, 0] * 512).long().clamp(max=511)] + r.n(P, 3) * 0.5
    anywhere = u * torch.tensor([200.0, 200.0, 60.0], device=DEV)
    w = which[:, None]
    pts = torch.where(w < 0.4, ground, torch.where(w < 0.7, facade, torch.where(w < 0.9, near, anywhere)))
    return {"pts": pts.contiguous()}


def _run_knn(s):
    from simple_knn._C import distCUDA2
    return distCUDA2(s["pts"])


# ------------------------------------------------------------------- entry points --

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "render"):
        s = _prepare_view(case, seed, kind == "train")
    else:
        s = {"neural": _prepare_neural, "loss": _prepare_loss, "adam": _prepare_adam, "stats": _prepare_stats,
             "knn": _prepare_knn}[kind](case, seed)
    s["run"] = {"train": _run_view, "render": _run_view, "neural": _run_neural, "loss": _run_loss, "adam": _run_adam,
                "stats": _run_stats, "knn": _run_knn}[kind]
    return s


def run(state):
    return state["run"](state)


def work(case):
    """Inputs read once and outputs written once; operations as the formulas have them (a fused multiply-add is two)."""
    kind = case["kind"]
    if kind in ("train", "render"):
        P, HW = case["P"], case["W"] * case["H"]
        per_g = 44 + (192 if case["sh"] else 12)       # parameters
        images = (9 if case["geo"] else 3) * 4 * HW
        blends = LAYOUTS[case["layout"]][4] * HW
        ch = 8 if case["geo"] else 3
        flops = P * (260 + (150 if case["sh"] else 0) + (60 if case["geo"] else 0)) + blends * (25 + 2 * ch)
        nbytes = P * (per_g + 8) + images              # + radii and observation counts
        if kind == "train":
            nbytes += P * (per_g + 12) + images        # gradients out (absolute screen gradients too), upstream in
            flops += P * (520 + (300 if case["sh"] else 0) + (120 if case["geo"] else 0)) + blends * (60 + 6 * ch)
        return {"bytes": nbytes, "flops": flops}
    if kind == "neural":
        # every anchor is tested for visibility; the visible ones (and half of their candidates) are computed
        A, k = case["A"], case["k"]
        v = _visible(case)
        s = v * k // 2
        per_anchor = 12 + 128 + 12 * k + 24
        nbytes = A * (12 + 12 + 16 + 4) + v * (per_anchor + 5 * k) + s * 56 + s * 56 + A * per_anchor
        flops = A * 250 + v * (2 * (3 * 35 * 32 + 32 * 11 * k) * 3)
        return {"bytes": nbytes, "flops": flops}
    if kind == "loss":
        n = 3 * case["W"] * case["H"]
        return {"bytes": n * (8 + 8 + 8 + 4) + n // 3, "flops": n * (5 * 44 + 40 + 3 * 44 + 20)}
    if kind == "adam":
        n = 59 * case["P"]
        return {"bytes": 28 * n, "flops": 12 * n}
    if kind == "stats":
        A, k = case["A"], case["k"]
        vis = 0.4 * A
        sel = 0.6 * vis * k
        kept = 0.9 * sel
        return {"bytes": A + vis * k * 5 + sel * 9 + vis * 16 + kept * 16, "flops": vis * k + 4 * kept}
    P = case["P"]
    return {"bytes": 16 * P, "flops": 8 * P * (8 * math.log2(max(P, 2)))}


def tolerance(case):
    """About four times the largest difference seen against the same computation in float64."""
    kind = case["kind"]
    if kind in ("train", "render"):
        # images within 3e-6 (4e-5 of single values), gradients within 1e-5 (2e-4); with the geometry channels 1.2e-4
        # (1.3e-2), from pixels whose plane is seen nearly edge-on
        return {"rel": 5e-4, "max": 5e-2} if case["geo"] else {"rel": 4e-5, "max": 1e-3}
    return {"neural": {"rel": 1.6e-6, "max": 1e-4},   # 4e-7 (2.3e-5)
            "loss": {"rel": 5.6e-5, "max": 1.2e-3},   # 1.4e-5 (3e-4): variances as differences of two sums
            "adam": {"rel": 4e-7, "max": 1.2e-6},     # 1e-7 (2.9e-7)
            "stats": {"rel": 2e-7, "max": 7e-7},      # 4.3e-8 (1.8e-7)
            "knn": {"rel": 2e-7, "max": 7e-7}}[kind]  # 4.8e-8 (1.6e-7)
