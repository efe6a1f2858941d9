"""The one-pass gather of a view's anchors (gaussian_renderer/__init__.py:794-798) and its gradient against
torch's index_select: the same values bit for bit (no arithmetic is done on them)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _arrays(A, k, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(DEV).requires_grad_()
    return r(A, 3), r(A, 32), r(A, k, 3), r(A, 6)


# a workgroup takes 256 rows, the counting kernel four such chunks, the scan over chunks 4096 chunks per step
@pytest.mark.parametrize("A,k,share", [(1, 10, 1.0), (1, 10, 0.0), (255, 1, 0.5), (256, 4, 1.0), (257, 10, 0.35),
                                       (1023, 7, 0.0), (1025, 16, 0.02), (70_001, 10, 0.35), (4096 * 256 + 3, 1, 0.3)])
def test_rows_and_gradients_equal_index_select(A, k, share):
    from gs_neural import _VisibleRows, _visible_rows
    leaf = _arrays(A, k, A)
    mask = (torch.rand(A, generator=torch.Generator().manual_seed(A + 1)) < share).to(DEV)
    idx = mask.nonzero(as_tuple=True)[0]
    out = _visible_rows(mask, *leaf, True)
    if idx.numel():
        assert type(out[0].grad_fn).__name__ == _VisibleRows.__name__ + "Backward"
    assert torch.equal(out[4], idx)
    ups = [torch.randn_like(o) for o in out[:4]]
    for o, t in zip(out, leaf):
        assert torch.equal(o, t.index_select(0, idx))
    torch.autograd.backward(list(out[:4]), ups)
    for t, u in zip(leaf, ups):
        assert torch.equal(t.grad, torch.zeros_like(t).index_copy_(0, idx, u))


def test_forms_of_inputs_and_gradients():
    from gs_neural import _visible_rows
    A, k = 1000, 5
    leaf = _arrays(A, k, 3)
    mask = torch.rand(A, device=DEV) < 0.4
    idx = mask.nonzero(as_tuple=True)[0]
    dense = lambda g: torch.zeros(A, *g.shape[1:], device=DEV).index_copy_(0, idx, g)
    # an expanded gradient, a feature gradient that starts off 16 bytes, two arrays without a gradient
    anchor, feat, offsets, scaling, none = _visible_rows(mask, leaf[0], leaf[1], leaf[2].detach(), leaf[3], False)
    n = idx.numel()
    g_feat = torch.randn(n * 32 + 1, device=DEV)[1:].view(n, 32)
    g_anchor = torch.randn(n, 1, device=DEV).expand(n, 3)
    got = torch.autograd.grad([anchor, feat], [leaf[0], leaf[1], leaf[3]], [g_anchor, g_feat], allow_unused=True)
    assert none is None and not offsets.requires_grad and got[2] is None
    assert torch.equal(got[0], dense(g_anchor)) and torch.equal(got[1], dense(g_feat))
    # a graph of the backward pass
    w = torch.randn(n, 3, device=DEV, requires_grad=True)
    anchor = _visible_rows(mask, *leaf, False)[0]
    g, = torch.autograd.grad(anchor, leaf[0], w, create_graph=True)
    u = torch.randn(A, 3, device=DEV)
    assert torch.equal(torch.autograd.grad(g, w, u)[0], u[idx])
    # strided and misaligned arrays, uint8 and short masks are gathered all the same
    wide = torch.randn(A, 64, device=DEV)
    off = torch.randn(A * 32 + 1, device=DEV)[1:].view(A, 32)
    for feat in (wide[:, ::2], off):
        out = _visible_rows(mask, leaf[0], feat, leaf[2], leaf[3], False)
        assert torch.equal(out[1], feat[idx]) and torch.equal(out[3], leaf[3][idx])
    assert torch.equal(_visible_rows((mask * 3).to(torch.uint8), *leaf, False)[1], leaf[1][idx])
    assert torch.equal(_visible_rows(mask[:300], *leaf, False)[2], leaf[2][:300][mask[:300]])
