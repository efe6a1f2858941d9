"""What preprocess_gaussians leaves for build_all_map(..., blend_records_of=means2D) and render_gaussians, on the CPU with
torch statements in place of the kernels."""
import threading

import pytest
import torch

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
