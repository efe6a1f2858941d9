"""The autograd graph around build_all_map(..., blend_records_of=means2D), on the CPU with torch statements in place of
the kernels: the channels have a node and saved tensors of their own whether or not preprocess_gaussians formed them,
and their gradient goes through the preprocess node exactly where that node runs in the same backward pass."""
import threading

import pytest
import torch
from torch.utils.checkpoint import checkpoint

P = 7


class Kernels:
    """Stand-ins for the operators of `_C` that the two nodes call.  Polynomials: gradients are compared exactly."""

    def __init__(self):
        self.calls = []

    def channels(self, m, s, q):
        return torch.stack([m[:, 0] * q[:, 0], m[:, 1] * q[:, 1], m[:, 2] + q[:, 2], torch.ones_like(m[:, 0]),
                            m[:, 0] * q[:, 3]], 1)

    def channels_gradient(self, m, s, q, g):
        zero = torch.zeros_like(g[:, 0])
        return (torch.stack([g[:, 0] * q[:, 0] + g[:, 4] * q[:, 3], g[:, 1] * q[:, 1], g[:, 2]], 1),
                torch.stack([g[:, 0] * m[:, 0], g[:, 1] * m[:, 1], g[:, 2], g[:, 4] * m[:, 0]], 1) + zero[:, None])

    def preprocess_gaussians_ex(self, m, s, q, sh, o, *rest, blend_records=None, all_map=None, **kw):
        self.calls.append("preprocess")
        m, s, q, o = m.detach(), s.detach(), q.detach(), o.detach()
        if all_map is not None:
            all_map.copy_(self.channels(m, s, q))
        n = m.shape[0]
        return ((0, m[:, :2] * 2, m[:, 2] + 0, torch.ones(n, dtype=torch.int32), None,
                 torch.cat([s * 3, o], 1), torch.zeros(n, 3), torch.zeros(n, 3, dtype=torch.bool)), None)

    def preprocess_gaussians_backward(self, radii, cov, clamped, m, s, q, sh, *rest, dcolor_ddir=None,
                                      dL_dall_map=None):
        self.calls.append("preprocess backward" + (" with channels" if dL_dall_map is not None else ""))
        g2, gco = rest[9], rest[10]
        dm = torch.cat([g2 * 2, torch.zeros(m.shape[0], 1)], 1)
        dq = torch.zeros_like(q)
        if dL_dall_map is not None:
            a, b = self.channels_gradient(m, s, q, dL_dall_map)
            dm, dq = dm + a, dq + b
        return dm, gco[:, :3] * 3, dq, torch.zeros_like(sh), gco[:, 3:]

    def build_all_map(self, m, s, q, vm, cp):
        self.calls.append("channels")
        return self.channels(m.detach(), s.detach(), q.detach())

    def build_all_map_backward(self, m, s, q, vm, cp, g):
        self.calls.append("channels backward")
        return self.channels_gradient(m, s, q, g)


@pytest.fixture
def K(monkeypatch):
    import diff_gaussian_rasterization as dgr
    k = Kernels()
    for name in ("preprocess_gaussians_ex", "preprocess_gaussians_backward", "build_all_map",
                 "build_all_map_backward"):
        monkeypatch.setattr(dgr._C, name, getattr(k, name))
    dgr._linked_all_map_seen[0] = False
    yield k
    dgr._linked_all_map_seen[0] = False


def leaves(seed=0):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randint(-4, 5, s, generator=gen).float().requires_grad_()
    return dict(m=r(P, 3), s=r(P, 3), q=r(P, 4), sh=r(P, 3), o=r(P, 1))


def settings():
    import diff_gaussian_rasterization as dgr
    return dgr.GaussianRasterizationSettings(32, 32, 0.5, 0.5, torch.zeros(3), 1.0, torch.eye(4), torch.eye(4), 3,
                                             torch.zeros(3), False, True, False)


def view(t, rs, linked=True):
    import diff_gaussian_rasterization as dgr
    means2D, rgb, co, radii, depths = dgr.preprocess_gaussians(t["m"], t["s"], t["q"], t["sh"], t["o"], rs, None)
    am = dgr.build_all_map(t["m"], t["s"], t["q"], rs.viewmatrix, rs.campos,
                           blend_records_of=means2D if linked else None)
    return means2D, co, am


def image_loss(means2D, co):
    return (means2D * means2D).sum() + (co * co).sum()


def channel_loss(am):
    return (am * am).sum()


def grads(t):
    return [t[k].grad for k in sorted(t)]


def same(a, b):
    return all((x is None) == (y is None) and (x is None or torch.equal(x, y)) for x, y in zip(a, b))


def reference(parts):
    """The gradients of the chosen losses with the channels as an operator of their own."""
    t = leaves()
    means2D, co, am = view(t, settings(), linked=False)
    loss = 0
    if "image" in parts:
        loss = loss + image_loss(means2D, co)
    if "channels" in parts:
        loss = loss + channel_loss(am)
    loss.backward()
    return grads(t)


def test_one_backward_pass_uses_the_channels_of_the_preprocess_kernel(K):
    want = reference("image channels".split())
    rs = settings()
    for n in range(3):
        t = leaves()
        K.calls.clear()
        means2D, co, am = view(t, rs)
        (image_loss(means2D, co) + channel_loss(am)).backward()
        assert same(grads(t), want), n
        if n > 0:  # (the first view learns that the channels are wanted)
            assert K.calls == ["preprocess", "preprocess backward with channels"]


@pytest.mark.parametrize("order", ["channels first", "image first"])
def test_two_losses_differentiated_one_after_the_other(K, order):
    want = reference("image channels".split())
    rs = settings()
    for n in range(3):
        t = leaves()
        means2D, co, am = view(t, rs)
        losses = [channel_loss(am), image_loss(means2D, co)]
        for loss in losses if order == "channels first" else losses[::-1]:
            loss.backward()
        assert same(grads(t), want), n


@pytest.mark.parametrize("parts", ["image", "channels"])
def test_one_of_the_two_losses(K, parts):
    want = reference([parts])
    rs = settings()
    for n in range(2):
        t = leaves()
        means2D, co, am = view(t, rs)
        (image_loss(means2D, co) if parts == "image" else channel_loss(am)).backward()
        assert same(grads(t), want), n


def test_retained_graph_failed_pass_and_hooks(K):
    rs = settings()
    view(leaves(), rs)
    want = reference("image channels".split())
    t = leaves()
    means2D, co, am = view(t, rs)
    loss = image_loss(means2D, co) + channel_loss(am)
    seen = []
    am.register_hook(lambda g: seen.append(g.clone()))
    loss.backward(retain_graph=True)
    assert same(grads(t), want)
    # a pass that ends between the two nodes leaves nothing behind for the next one
    stop = means2D.register_hook(lambda g: 1 / 0)
    with pytest.raises(ZeroDivisionError):
        loss.backward(retain_graph=True)
    stop.remove()
    for x in t.values():
        x.grad = None
    image_loss(means2D, co).backward(retain_graph=True)
    assert same(grads(t), reference(["image"]))
    for x in t.values():
        x.grad = None
    loss.backward()
    assert same(grads(t), want)
    assert all(torch.equal(g, 2 * am.detach()) for g in seen) and len(seen) >= 2


def test_gradients_of_chosen_inputs(K):
    rs = settings()
    view(leaves(), rs)
    for names in (["m"], ["q"], ["s"], ["o"], ["q", "o"], ["m", "s"]):
        got = {}
        for linked in (False, True):
            t = leaves()
            means2D, co, am = view(t, rs, linked)
            loss = image_loss(means2D, co) + channel_loss(am)
            got[linked] = torch.autograd.grad(loss, [t[k] for k in names] + [am])
        assert same(got[False], got[True]), names
    # an input that has become a leaf of its own between the two calls
    t = leaves()
    base = t["m"]
    t["m"] = base * 1.0
    means2D, rgb, co, radii, depths = __import__("diff_gaussian_rasterization").preprocess_gaussians(
        t["m"], t["s"], t["q"], t["sh"], t["o"], rs, None)
    t["m"].detach_().requires_grad_()
    import diff_gaussian_rasterization as dgr
    am = dgr.build_all_map(t["m"], t["s"], t["q"], rs.viewmatrix, rs.campos, blend_records_of=means2D)
    (image_loss(means2D, co) + channel_loss(am)).backward()
    a, _ = K.channels_gradient(t["m"].detach(), None, t["q"].detach(), 2 * am.detach())
    assert torch.equal(t["m"].grad, a)
    assert torch.equal(base.grad[:, :2], 8 * base.detach()[:, :2])


def test_checkpointed_view(K):
    want = reference("image channels".split())
    rs = settings()
    for n in range(3):
        t = leaves()

        def run(*args):
            means2D, co, am = view(dict(zip(sorted(t), args)), rs)
            return image_loss(means2D, co) + channel_loss(am)

        checkpoint(run, *[t[k] for k in sorted(t)], use_reentrant=False).backward()
        assert same(grads(t), want), n


def test_linked_and_unlinked_views_in_turn(K):
    want = reference("image channels".split())
    rs = settings()
    for n in range(6):
        t = leaves()
        means2D, co, am = view(t, rs, linked=n % 3 != 1)
        saved = len(am.grad_fn.saved_tensors)
        (image_loss(means2D, co) + channel_loss(am)).backward()
        assert saved == 5 and same(grads(t), want), n


def test_another_stream_gets_channels_of_its_own(K, monkeypatch):
    """What the preprocess kernel writes belongs to the stream that kernel runs on."""
    import diff_gaussian_rasterization as dgr
    rs = settings()
    view(leaves(), rs)
    current = [11]
    monkeypatch.setattr(dgr._n, "stream_handle", lambda device: current[0])
    t = leaves()
    means2D, rgb, co, radii, depths = dgr.preprocess_gaussians(t["m"], t["s"], t["q"], t["sh"], t["o"], rs, None)
    current[0] = 12
    K.calls.clear()
    am = dgr.build_all_map(t["m"], t["s"], t["q"], rs.viewmatrix, rs.campos, blend_records_of=means2D)
    assert K.calls == ["channels"]
    (image_loss(means2D, co) + channel_loss(am)).backward()
    assert K.calls[1:] == ["channels backward", "preprocess backward"] or \
        K.calls[1:] == ["preprocess backward", "channels backward"]
    blend = means2D._gs_blend
    blend.records = torch.zeros(P, 16)
    parts = [r() for r in blend.refs]
    assert not blend.usable([means2D] + parts[1:], am, True)
    current[0] = 11
    assert dgr.build_all_map(t["m"], t["s"], t["q"], rs.viewmatrix, rs.campos, blend_records_of=means2D) is not None
    assert K.calls.count("channels") == 1  # (handed out on its own stream)


def test_views_of_several_threads_do_not_meet(K, monkeypatch):
    """What a preprocess call leaves goes to its own outputs, whichever thread runs in between."""
    import diff_gaussian_rasterization as dgr
    rs = settings()
    view(leaves(), rs)
    plain = dgr._PreprocessGaussians.apply
    inside, go = threading.Event(), threading.Event()

    def apply(*args):
        out = plain(*args)
        if threading.current_thread().name == "first":
            inside.set()
            go.wait(10)
        return out

    monkeypatch.setattr(dgr._PreprocessGaussians, "apply", apply)
    monkeypatch.setattr(dgr, "_linked_all_map_seen", [True])
    outs = {}

    def work(name, seed):
        t = leaves(seed)
        outs[name] = t, dgr.preprocess_gaussians(t["m"], t["s"], t["q"], t["sh"], t["o"], rs, None)

    first = threading.Thread(target=work, args=("a", 1), name="first")
    first.start()
    assert inside.wait(10)

    def second_apply(*args):
        out = plain(*args)
        go.set()  # (the first call goes on while the second is between its two halves)
        first.join(10)
        return out

    monkeypatch.setattr(dgr._PreprocessGaussians, "apply", second_apply)
    work("b", 2)
    for name in "ab":
        t, out = outs[name]
        assert out[0]._gs_blend.sources[0]() is t["m"], name


def test_views_in_inference_mode(K):
    """Tensors of inference mode have no version counter to check the link by: such a view is an unlinked one."""
    import diff_gaussian_rasterization as dgr
    rs = settings()
    view(leaves(), rs)
    dgr._expectations[(rs.image_height, rs.image_width, torch.device("cpu"))] = (100, 10)  # (records are worth writing)
    try:
        want = K.channels(*[leaves()[k].detach() for k in "msq"])
        with torch.inference_mode():
            means2D, co, am = view(leaves(), rs)
            cold = {k: v.detach().clone() for k, v in leaves().items()}
        assert torch.equal(am, want) and not hasattr(means2D, "_gs_blend")
        with torch.no_grad():
            assert torch.equal(view(cold, rs)[2], want)
        t = leaves()
        means2D = dgr.preprocess_gaussians(t["m"], t["s"], t["q"], t["sh"], t["o"], rs, None)[0]
        with torch.inference_mode():
            for _ in range(2):  # (handed out, then formed)
                am = dgr.build_all_map(t["m"], t["s"], t["q"], rs.viewmatrix, rs.campos, blend_records_of=means2D)
                assert torch.equal(am, want)
    finally:
        dgr._expectations.clear()


def test_expectations_remembered_by_several_threads():
    """More image sizes than are kept, from four threads: entries come and go under each other's hands."""
    import sys
    import diff_gaussian_rasterization as dgr
    failed = []

    def work(i):
        try:
            for k in range(20000):
                dgr._remember((i, k), 1, 1)
        except Exception as e:
            failed.append(repr(e))

    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        [t.start() for t in threads]
        [t.join() for t in threads]
        assert not failed and len(dgr._expectations) <= dgr._MAX_EXPECTATIONS
    finally:
        sys.setswitchinterval(interval)
        dgr._expectations.clear()


def test_expectations_of_cameras_on_both_sides_of_a_long_list():
    # (instances, longest list) of the views of one size, and the bound on the longest list that the next one is launched
    # with: 0 is any length
    import diff_gaussian_rasterization as dgr
    saved = dict(dgr._expectations)
    dgr._expectations.clear()
    try:
        bounds = []
        for longest in (100, 1638, 1639, 3276, 4500, 3000, 4500, 3276, 1639, 1638, 100, 3000):
            dgr._remember("size", 1000, longest)
            bounds.append(dgr._expectation("size")[1])
        assert bounds == [256, 2048, 4096, 4096, 0, 0, 0, 0, 0, 2048, 256, 0]
        dgr._remember("another size", 1000, 3000)
        assert dgr._expectation("another size") == (int(1000 * dgr._MARGIN) + 65536, 4096)
        dgr._expectations["size"] = (1000, 3000)  # (an entry without the third figure)
        assert dgr._expectation("size")[1] == 4096
    finally:
        dgr._expectations.clear()
        dgr._expectations.update(saved)


def test_bound_that_leaves_no_tile_to_split():
    # a quarter more than the longest list is below 3072: the view is launched without the way for longer lists
    import diff_gaussian_rasterization as dgr
    saved = dict(dgr._expectations)
    dgr._expectations.clear()
    try:
        bounds = []
        for longest in (0, 100, 1638, 1639, 2457, 2458, 3276, 4500, 2457, 1638):
            dgr._remember("size", 1000, longest)
            bounds.append(dgr._launch_bounds("size")[1])
        assert bounds == [0, 256, 2048, 3071, 3071, 4096, 4096, 0, 0, 2048]
        assert dgr._launch_bounds("no such size") == (0, 0)
    finally:
        dgr._expectations.clear()
        dgr._expectations.update(saved)


def test_expected_instances_are_those_of_the_fullest_of_the_last_views():
    import diff_gaussian_rasterization as dgr
    saved = dict(dgr._expectations)
    dgr._expectations.clear()
    try:
        room = lambda n: int(n * dgr._MARGIN) + 65536
        for n, most in ((1000, 1000), (500, 1000), (3000, 3000), *[(700, 3000)] * 7, (700, 700), (0, 700)):
            dgr._remember("size", n, 100)
            assert dgr._expectation("size") == (room(most), 256)
            assert dgr._expectations["size"][:3] == (n, 100, False)
        dgr._expectations["size"] = (2000, 100, False)  # (an entry without the views before)
        assert dgr._expectation("size")[0] == room(2000)
        dgr._remember("size", 900, 100)
        assert dgr._expectation("size")[0] == room(2000)
    finally:
        dgr._expectations.clear()
        dgr._expectations.update(saved)


def test_longest_list_of_the_last_views():
    import diff_gaussian_rasterization as dgr
    saved = dict(dgr._expectations)
    dgr._expectations.clear()
    try:
        assert dgr._recent_longest("size") == 0
        for longest, most in ((100, 100), (5000, 5000), *[(200, 5000)] * 7, (300, 300)):
            dgr._remember("size", 1000, longest)
            assert dgr._recent_longest("size") == most
        dgr._expectations["size"] = (2000, 70, False)  # (an entry without the views before)
        assert dgr._recent_longest("size") == 70
        dgr._remember("size", 900, 50)
        assert dgr._recent_longest("size") == 70 and dgr._expectation("size")[0] == int(2000 * dgr._MARGIN) + 65536
    finally:
        dgr._expectations.clear()
        dgr._expectations.update(saved)
