"""Densification statistics (GaussianModel.training_statis, scene/gaussian_model.py:1181-1205) on the GPU:
the fused call against the CPU oracle and against torch's own mask indexing on the device."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _case(A, k, seed, p_vis, p_sel, p_flt):
    gen = torch.Generator().manual_seed(seed)
    vis = torch.rand(A, generator=gen) < p_vis
    V = int(vis.sum())
    sel = torch.rand(V * k, generator=gen) < p_sel
    S = int(sel.sum())
    flt = torch.rand(S, generator=gen) < p_flt
    grad = torch.randn(S, 3, generator=gen)
    opacity = torch.randn(V * k, 1, generator=gen)
    acc = [torch.rand(A, 1, generator=gen), torch.rand(A, 1, generator=gen).round(),
           torch.rand(A * k, 1, generator=gen), torch.rand(A * k, 1, generator=gen).round()]
    return vis, sel, flt, grad, opacity, acc


@pytest.mark.parametrize("A,k,seed,p", [(5000, 10, 0, (0.6, 0.7, 0.8)), (4097, 5, 1, (1.0, 1.0, 1.0)),
                                        (3000, 10, 2, (0.02, 0.3, 0.5)), (2048, 1, 3, (0.5, 0.5, 0.0)),
                                        (1000, 10, 4, (0.0, 0.5, 0.5))])
def test_training_stats_matches_oracle(orc, A, k, seed, p):
    import gs_densify
    vis, sel, flt, grad, opacity, acc = _case(A, k, seed, *p)
    ref = orc.training_stats(acc[0].numpy(), acc[1].numpy(), acc[2].numpy(), acc[3].numpy(), k, grad.numpy(),
                             opacity.numpy(), flt.numpy(), sel.numpy(), vis.numpy())
    d = [t.to(DEV) for t in acc]
    gs_densify.training_statis(d[0], d[1], d[2], d[3], k, grad.to(DEV), opacity.to(DEV), flt.to(DEV), sel.to(DEV),
                               vis.to(DEV))
    for got, want in zip(d, ref):
        # same additions in the same order (one per slot and call): identical up to the last bit of sqrt's input
        assert np.abs(got.cpu().numpy().ravel() - want).max() <= 1e-6 * max(1.0, np.abs(want).max())


def test_training_stats_full_size_against_mask_indexing():
    """1 M anchors x 10 offsets, checked against the torch statements it replaces, run on the device."""
    import gs_densify
    A, k = 1_000_000, 10
    gen = torch.Generator(device=DEV).manual_seed(5)
    vis = torch.rand(A, generator=gen, device=DEV) < 0.4
    V = int(vis.sum())
    sel = torch.rand(V * k, generator=gen, device=DEV) < 0.6
    S = int(sel.sum())
    flt = torch.rand(S, generator=gen, device=DEV) < 0.9
    grad = torch.randn(S, 3, generator=gen, device=DEV)
    opacity = torch.randn(V * k, 1, generator=gen, device=DEV)
    acc = [torch.zeros(A, 1, device=DEV), torch.zeros(A, 1, device=DEV), torch.zeros(A * k, 1, device=DEV),
           torch.zeros(A * k, 1, device=DEV)]
    mine = [t.clone() for t in acc]
    for _ in range(2):  # twice: accumulation, not assignment
        gs_densify.training_statis(mine[0], mine[1], mine[2], mine[3], k, grad, opacity, flt, sel, vis)
        temp = opacity.clone().view(-1)
        temp[temp < 0] = 0
        acc[0][vis] += temp.view(-1, k).sum(dim=1, keepdim=True)
        acc[1][vis] += 1
        vis_rep = vis.unsqueeze(1).repeat(1, k).view(-1)
        combined = torch.zeros(A * k, dtype=torch.bool, device=DEV)
        combined[vis_rep] = sel
        temp_mask = combined.clone()
        combined[temp_mask] = flt
        acc[2][combined] += torch.norm(grad[flt, :2], dim=-1, keepdim=True)
        acc[3][combined] += 1
    assert torch.equal(mine[1], acc[1]) and torch.equal(mine[3], acc[3])
    assert float((mine[0] - acc[0]).abs().max()) <= 1e-5
    assert float((mine[2] - acc[2]).abs().max()) <= 1e-5
    assert int(mine[3].sum()) == 2 * int(flt.sum())


def test_training_stats_rejects_inconsistent_inputs():
    import gs_densify
    z = lambda *s: torch.zeros(*s, device=DEV)
    with pytest.raises(RuntimeError):
        gs_densify.training_statis(z(4, 1), z(4, 1), z(8, 1), z(8, 1), 2, z(3, 3), z(5, 1),
                                   torch.ones(3, dtype=torch.bool, device=DEV),
                                   torch.ones(5, dtype=torch.bool, device=DEV),
                                   torch.ones(4, dtype=torch.bool, device=DEV))
    with pytest.raises(RuntimeError):
        gs_densify.training_statis(torch.zeros(4, 1), torch.zeros(4, 1), torch.zeros(8, 1), torch.zeros(8, 1), 2,
                                   torch.zeros(0, 3), torch.zeros(0, 1), torch.zeros(0, dtype=torch.bool),
                                   torch.zeros(0, dtype=torch.bool), torch.zeros(4, dtype=torch.bool))


def test_update_max_radii_matches_torch_statement():
    import gs_densify
    gen = torch.Generator().manual_seed(3)
    n = 100_003
    m = torch.rand(n, generator=gen) * 40
    radii = torch.randint(0, 80, (n,), generator=gen, dtype=torch.int32)
    vis = torch.rand(n, generator=gen) < 0.4
    want = m.clone()
    want[vis] = torch.max(want[vis], radii[vis].float())
    got = gs_densify.update_max_radii(m.to(DEV), radii.to(DEV), vis.to(DEV)).cpu()
    assert torch.equal(got, want)
    assert torch.equal(got[~vis], m[~vis])


@pytest.mark.parametrize("A,k,p", [(1, 1, (1.0, 1.0, 1.0)), (255, 10, (1.0, 0.5, 0.9)), (257, 256, (0.9, 0.6, 0.9)),
                                   (700, 255, (1.0, 0.97, 0.6)), (300, 257, (0.7, 0.6, 0.9)), (1025, 3, (0.4, 0.0, 1.0)),
                                   (3000, 7, (0.5, 0.6, 0.9))])
@pytest.mark.parametrize("offset", [0, 1])
def test_training_stats_chunk_edges(orc, A, k, p, offset):
    """Anchors, candidates and rounds that end inside and at the edge of a chunk, the offset counts on either side of
    the last one that chunks take, and masks that start at any byte.  Sums of k terms in the oracle's order."""
    import gs_densify
    vis, sel, flt, grad, opacity, acc = _case(A, k, A + k, *p)
    ref = orc.training_stats(acc[0].numpy(), acc[1].numpy(), acc[2].numpy(), acc[3].numpy(), k, grad.numpy(),
                             opacity.numpy(), flt.numpy(), sel.numpy(), vis.numpy())
    shifted = lambda m: torch.cat([torch.ones(offset, dtype=torch.bool), m]).to(DEV)[offset:]
    d = [t.to(DEV) for t in acc]
    gs_densify.training_statis(d[0], d[1], d[2], d[3], k, grad.to(DEV), opacity.to(DEV), shifted(flt), shifted(sel),
                               shifted(vis))
    for got, want in zip(d, ref):
        assert np.abs(got.cpu().numpy().ravel() - want).max() <= 1e-6 * max(1.0, np.abs(want).max())


# spans of 16384 mask entries: on either side of one, of their number that a thread adds up by itself, and beyond
@pytest.mark.parametrize("A,k,p", [(16384, 1, (1.0, 0.5, 0.9)), (16385, 3, (1.0, 1.0, 0.9)), (33_000, 10, (0.99, 0.6, 0.9)),
                                   (512 * 16384, 1, (1.0, 0.6, 0.9)), (512 * 16384 + 1, 1, (0.5, 0.6, 0.9)),
                                   (900_000, 10, (0.95, 0.6, 0.9))])
def test_training_stats_span_edges(orc, A, k, p):
    import gs_densify
    vis, sel, flt, grad, opacity, acc = _case(A, k, A + k, *p)
    ref = orc.training_stats(acc[0].numpy(), acc[1].numpy(), acc[2].numpy(), acc[3].numpy(), k, grad.numpy(),
                             opacity.numpy(), flt.numpy(), sel.numpy(), vis.numpy())
    d = [t.to(DEV) for t in acc]
    gs_densify.training_statis(d[0], d[1], d[2], d[3], k, grad.to(DEV), opacity.to(DEV), flt.to(DEV), sel.to(DEV),
                               vis.to(DEV))
    for got, want in zip(d, ref):
        assert np.abs(got.cpu().numpy().ravel() - want).max() <= 1e-6 * max(1.0, np.abs(want).max())


# whole sectors of 16 slots and what is left of them, accumulators that do not start at a multiple of 16 bytes, every
# number of anchors a workgroup takes; gains of 0, infinite and NaN ones, and slots without a gain, which keep their bits
@pytest.mark.parametrize("A,k", [(1003, 1), (513, 10), (300, 16), (301, 17), (130, 33), (67, 65), (35, 129), (17, 256)])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_training_stats_sectors(orc, A, k, shift):
    import gs_densify
    vis, sel, flt, grad, opacity, acc = _case(A, k, A + k, 0.4, 0.5, 0.7)
    S = grad.shape[0]
    grad[:: 7] = 0.0
    grad[min(3, S - 1)] = float("inf")
    grad[min(5, S - 1)] = float("nan")
    acc[2][::3] = -0.0
    acc[2][1::5] = float("nan")
    ref = orc.training_stats(acc[0].numpy(), acc[1].numpy(), acc[2].numpy(), acc[3].numpy(), k, grad.numpy(),
                             opacity.numpy(), flt.numpy(), sel.numpy(), vis.numpy())
    place = lambda a: torch.cat([torch.full((shift, 1), 7.0), a, torch.full((3, 1), 7.0)]).to(DEV)
    whole = [place(a) for a in acc]
    d = [w[shift:shift + a.shape[0]] for w, a in zip(whole, acc)]
    gs_densify.training_statis(d[0], d[1], d[2], d[3], k, grad.to(DEV), opacity.to(DEV), flt.to(DEV), sel.to(DEV),
                               vis.to(DEV))
    for w, a in zip(whole, acc):
        assert bool((w[:shift] == 7.0).all()) and bool((w[shift + a.shape[0]:] == 7.0).all())
    for got, want in zip(d, ref):
        got, want = got.cpu().numpy().ravel(), want.ravel()
        assert np.array_equal(np.isfinite(got), np.isfinite(want))
        ok = np.isfinite(want)
        assert np.abs(got[ok] - want[ok]).max() <= 1e-6 * max(1.0, np.abs(want[ok]).max())
    hit = torch.zeros(A * k, dtype=torch.bool)
    cand = hit.clone()
    cand[vis.repeat_interleave(k)] = sel
    hit[cand] = flt
    bits = lambda x: x.cpu().contiguous().view(torch.int32).ravel()
    assert torch.equal(bits(d[2])[~hit], bits(acc[2])[~hit]) and torch.equal(bits(d[3])[~hit], bits(acc[3])[~hit])
