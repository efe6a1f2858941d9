"""Views whose tiles have long lists, which the forward blend gives to four workgroups each: lengths around the one where
that begins and around whole batches, pixels that saturate early, late and never, cut-off tiles, tile masks, channels that
are not finite, packed, caller-written and gathered operands, against the oracle, bit for bit; and the gradients that come
out of the hit words such a tile leaves."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LONG = 3072  # entries from which on a tile is long


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


def scene(n, everywhere, opacity, seed):
    """n Gaussians around a 73 x 43 image (5 x 3 tiles); those up to `everywhere` are entered in every tile's list."""
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.rand(*s, generator=gen)
    W, Hh = 73, 43
    s1 = torch.exp(r(n) * 2.5) * 0.8
    s2 = torch.clamp(s1 * (0.2 + 0.8 * r(n)), min=0.5)
    ang = r(n) * 3.14159
    c, s = torch.cos(ang), torch.sin(ang)
    i1, i2 = 1 / s1 ** 2, 1 / s2 ** 2
    am = torch.randn(n, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0
    am[:, 3] = 1.0
    radii = torch.ceil(3 * s1).int()
    radii[:everywhere] = 200
    return dict(W=W, H=Hh, tan=0.5, means2D=r(n, 2) * torch.tensor([W + 8.0, Hh + 8.0]) - 4.0,
                co=torch.stack([c * c * i1 + s * s * i2, c * s * (i1 - i2), s * s * i1 + c * c * i2,
                                r(n) * opacity + 0.003], 1).float(),
                radii=radii, depths=r(n) * 10 + 1, rgb=r(n, 3), am=am, bg=torch.tensor([0.3, 0.6, 0.1]),
                up=[torch.randn(k, Hh, W, generator=gen) for k in (3, 5, 1)])


def same(a, b):
    return np.array_equal(a, b, equal_nan=a.dtype.kind == "f")


def check(H, orc, v, cl, geo, ahead, records, gradients=True, gathered=False, bound=0):
    from diff_gaussian_rasterization import _C
    n = {k: t.numpy() for k, t in v.items() if isinstance(t, torch.Tensor)}
    W, Hh, tan, P, clf = v["W"], v["H"], v["tan"], v["co"].shape[0], cl.numpy().ravel()
    b = orc.bin_and_sort(n["radii"], n["means2D"], n["depths"], clf, W, Hh)
    f = orc.render_fwd(b["ranges"], b["point_list"], n["means2D"], n["rgb"], n["am"], n["co"], clf, n["bg"], W, Hh, tan,
                       tan, render_geo=geo)
    d = {k: t.to(DEV) for k, t in v.items() if isinstance(t, torch.Tensor)}
    rec = None
    if records:
        rec = torch.cat([d["means2D"], d["co"], d["rgb"], d["am"], d["depths"][:, None], torch.zeros(P, 1, device=DEV)],
                        1).contiguous()
    args = {"stats_collector": {}}
    R = b["point_list"].shape[0]
    assert gathered == (not records and R * 5 <= P * 4)  # (the library packs records itself above that)
    out, info = _C.render_gaussians_ex(d["bg"], Hh, W, d["means2D"], d["depths"], d["radii"], d["co"], d["rgb"],
                                       cl.to(DEV), torch.eye(4, device=DEV), torch.zeros(3, device=DEV), tan, tan, d["am"],
                                       geo, False, args, expected_instances=R + R // 8 if ahead else 0,
                                       expected_longest_list=bound, blend_records=rec)
    assert info["launched_ahead"] == (ahead and (bound == 0 or info["longest_list"] <= bound))
    R, color, n_render, n_consider, n_contrib, obs, oam, opd, geom, binning, img = out
    for k, got, want in (("color", color, f["color"]), ("n_render", n_render, f["n_render"]),
                         ("n_consider", n_consider, f["n_consider"]), ("n_contrib", n_contrib, f["n_contrib_tile"]),
                         ("observe", obs, f["out_observe"])):
        assert same(got.cpu().numpy(), want), k
    if geo:
        assert same(oam.cpu().numpy(), f["out_all_map"])
        assert same(opd.cpu().numpy(), f["out_plane_depth"])
    if not gradients:
        return b
    got = _C.render_gaussians_backward(d["bg"], tan, tan, oam, d["am"], R, geom, binning, img, cl.to(DEV),
                                       *[u.to(DEV) for u in v["up"]], d["means2D"], d["co"], d["rgb"], geo, False, args,
                                       binning_capacity=info["binning_capacity"], blend_records=rec)
    g = orc.render_bwd(b["ranges"], b["point_list"], n["means2D"], n["co"], n["rgb"], n["am"], f["out_all_map"],
                       f["final_T"], f["n_contrib"], clf, n["bg"], *[u.numpy() for u in v["up"]], W, Hh, tan, tan,
                       render_geo=geo)
    # a Gaussian's sum has at most 73 x 43 terms, whose magnitudes add up to some ten times the sum: another order of them
    # moves it by sqrt(3139) * 2^-24 * 10 = 3.3e-5
    for k, a, w in zip(("dL_dmeans2D", "dL_dmeans2D_abs", "dL_dconic_opacity", "dL_dcolors", "dL_dall_map"), got,
                       (g["dL_dmeans2D"][:, :2], g["dL_dmeans2D_abs"], g["dL_dconic_opacity"], g["dL_dcolors"],
                        g["dL_dall_map"])):
        if k != "dL_dall_map" or geo:
            assert H.rel_l2(a.cpu().numpy(), w) <= 1e-4, k
    return b


@pytest.mark.parametrize("n", [LONG - 1, LONG, LONG + 1, 13 * 256 - 1, 13 * 256 + 1])
@pytest.mark.parametrize("opacity", [0.9, 0.05, 0.01])
def test_every_tile_at_a_length(H, orc, n, opacity):
    # 15 tiles: of long ones eight are split, the other seven are not
    v = scene(n, n, opacity, seed=n)
    cl = torch.ones(3, 5, dtype=torch.bool)
    for geo, ahead, records in ((True, False, False), (True, True, True), (False, True, False), (False, False, True)):
        b = check(H, orc, v, cl, geo, ahead, records, gradients=opacity != 0.05)
        assert (np.diff(b["ranges"].reshape(-1, 2).astype(np.int64)) == n).all()


@pytest.mark.parametrize("n,bound", [(LONG - 1, LONG - 1), (LONG - 1, LONG), (LONG - 1, 4096), (LONG, LONG - 1), (LONG, LONG)])
def test_bounds_on_the_longest_list(H, orc, n, bound):
    # launched ahead without the way for long tiles, with it but without such a tile, and without it where one turns up
    v = scene(n, n, 0.05, seed=n)
    cl = torch.ones(3, 5, dtype=torch.bool)
    for geo in (True, False):
        check(H, orc, v, cl, geo, True, True, bound=bound)


@pytest.mark.parametrize("n", [LONG - 1, LONG, 13 * 256 + 1])
def test_operands_that_are_gathered(H, orc, n):
    # (fewer instances than Gaussians: nobody packs records, and no tile is split)
    v = scene(20 * n, n, 0.05, seed=n)
    v["radii"][n:] = 0
    cl = torch.ones(3, 5, dtype=torch.bool)
    for geo, ahead in ((True, False), (True, True), (False, True)):
        check(H, orc, v, cl, geo, ahead, records=False, gathered=True)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("geo", [False, True])
def test_few_long_tiles(H, orc, masked, geo):
    # the groups of eight are filled up with tiles below the limit, empty and masked ones among them
    v = scene(9000, 0, 0.3, seed=5)
    near = torch.rand(9000, generator=torch.Generator().manual_seed(1)) < 0.7
    v["means2D"][near] = v["means2D"][near] * 0.2 + torch.tensor([2.0, 30.0])
    v["means2D"][~near, 0] *= 0.6  # (the right-most tiles have short lists or none)
    cl = torch.ones(3, 5, dtype=torch.bool)
    if masked:
        cl[1] = False
    b = check(H, orc, v, cl, geo, ahead=False, records=True)
    lengths = np.diff(b["ranges"].reshape(-1, 2).astype(np.int64)).ravel()
    assert 0 < (lengths >= LONG).sum() < 8 and (lengths < LONG).any()


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_channels_that_are_not_finite(H, orc, value):
    v = scene(LONG + 300, LONG + 300, 0.05, seed=9)
    v["rgb"][100:110, 1] = value
    v["am"][700:720, 4] = value
    v["am"][2900:3300:7, 0] = value
    cl = torch.ones(3, 5, dtype=torch.bool)
    for geo, records in ((True, True), (False, True), (True, False)):
        check(H, orc, v, cl, geo, False, records, gradients=False)


def tiles_split(lengths, geo):
    """How many tiles the forward blend splits, from the rule's statement."""
    if 2 * lengths.sum() > 1536 * lengths.max():
        return 0
    for least in (3072, 4096, 6144) if geo else (3072, 4096):
        count = int((lengths >= least).sum())
        if count <= 340:
            break
    return count


# (tiles in x and y, entries of every tile, further entries of the first)
@pytest.mark.parametrize("gx,gy,n,first", [
    (17, 1, 3072, 0),      # three groups of eight, the last one filled up with what there is
    (34, 10, 3072, 0),     # as many as are split at this length
    (31, 11, 3072, 2000),  # one more: the next length
    (31, 11, 4096, 0),     # one more at the next length too: the third, or all of them where there is none
    (31, 11, 6143, 1), (31, 11, 6144, 0),
    (32, 24, 4100, 0),     # two shares of the entries, just
    (769, 1, 4100, 0),     # one tile more, and the longest list is below two shares
    (103, 10, 6144, 2300)  # more tiles to split than are
])
@pytest.mark.parametrize("geo", [True, False])
def test_which_tiles_are_split(H, gx, gy, n, first, geo):
    """The number of tiles to split, which the blend finds behind the word for packed records, and every output against
    the lists built the other way, whose tiles are never split."""
    import ctypes as C
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    W, Hh, P = 16 * gx - 3, 16 * gy - 5, n + first
    gen = torch.Generator().manual_seed(n)
    r = lambda *s: torch.rand(*s, generator=gen)
    means2D = r(P, 2) * torch.tensor([float(W), float(Hh)])
    means2D[n:] = torch.tensor([8.0, 8.0])
    radii = torch.full((P,), 20000, dtype=torch.int32)
    radii[n:] = 1
    size = 1.0 + 12.0 * r(P)
    co = torch.stack([1 / size ** 2, torch.zeros(P), 1 / size ** 2, 0.02 + 0.3 * r(P)], 1)
    am = torch.randn(P, 5, generator=gen)
    am[:, 2] = am[:, 2].abs() + 2.0
    d = [t.to(DEV) for t in (means2D, r(P) * 10 + 1, radii, co, r(P, 3))]
    cl = torch.ones(gy, gx, dtype=torch.bool, device=DEV)
    outs = []
    for limits in ((-1, -1), (0, 0)):
        outs.append(_C.render_gaussians(torch.tensor([0.3, 0.6, 0.1], device=DEV), Hh, W, *d, cl, torch.eye(4, device=DEV),
                                        torch.zeros(3, device=DEV), 0.5, 0.5, am.to(DEV), geo, False,
                                        {"stats_collector": {}, "tile_sort_limits": limits}))
    for a, b in zip(outs[0][1:8], outs[1][1:8]):
        assert torch.equal(a, b)
    lengths = outs[0][2].flatten().cpu().numpy().astype(np.int64)
    assert (np.sort(lengths) == np.sort(np.array([n + first] + [n] * (gx * gy - 1)))).all()
    total = C.c_size_t()
    gn.check(gn.lib.gs_geometry_state_layout(P, None, None, C.byref(total)), "layout")
    geom = outs[0][8]
    at = -geom.data_ptr() % 256 + total.value - 512 + 4  # (the last two words but the alignment's reserve)
    assert int(geom[at:at + 4].view(torch.int32)) == 1 + tiles_split(lengths, geo)
