"""The counting sort by tile at the numbers of Gaussians where its workgroups' chunks change: one, two and four Gaussians a
thread, the last thread's and the last workgroup's partly filled, more instances in a chunk than the LDS stages.  Lists,
ranges and prefix sums against the oracle, bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    import gpu_harness
    return gpu_harness


# (chunks of 512 Gaussians up to 131 072, then 256 of them: a Gaussian a thread up to 262 144, two up to 524 288, four up
# to 1 048 576, several rounds beyond)
@pytest.mark.parametrize("P", [1, 511, 512, 513, 1023, 131_072, 131_073, 262_144, 262_145, 524_288, 524_289, 1_048_576,
                               1_048_577])
@pytest.mark.parametrize("masked", [False, True])
def test_chunks(orc, H, P, masked):
    lists(orc, H, P, 3, masked)


@pytest.mark.parametrize("P", [600, 300_000])
def test_more_instances_than_are_staged(orc, H, P):
    lists(orc, H, P, 120 if P < 1000 else 60, False)


def lists(orc, H, P, largest, masked):
    import gsrast_native as gn
    from diff_gaussian_rasterization import _C
    W, Hh = 1152, 864
    gx, gy = H.grid(W, Hh)
    rng = np.random.default_rng(P)
    radii = rng.integers(0, largest + 1, P).astype(np.int32)
    means = (rng.random((P, 2)) * [W + 40.0, Hh + 40.0] - 20.0).astype(np.float32)
    depths = (rng.random(P) * 50 + 1).astype(np.float32)
    cl = np.ones((gy, gx), bool)
    if masked:
        cl[rng.random((gy, gx)) < 0.3] = False
    want = orc.bin_and_sort(radii, means, depths, cl.reshape(-1), W, Hh)
    R = int(want["point_list"].shape[0])
    co = torch.zeros(P, 4, device=DEV)  # (opacity 0: nothing is blended)
    co[:, 0] = co[:, 2] = 1.0
    for ahead in (False, True):
        out, info = _C.render_gaussians_ex(
            torch.zeros(3, device=DEV), Hh, W, torch.from_numpy(means).to(DEV), torch.from_numpy(depths).to(DEV),
            torch.from_numpy(radii).to(DEV), co, torch.zeros(P, 3, device=DEV), torch.from_numpy(cl).to(DEV),
            torch.eye(4, device=DEV), torch.zeros(3, device=DEV), 0.5, 0.5, None, False, False, {"stats_collector": {}},
            expected_instances=R + 100 if ahead else 0)
        assert out[0] == R and info["launched_ahead"] == ahead
        geom, binning, img = out[8:11]

        def part(buf, offset, words):
            base = -buf.data_ptr() % 256 + offset
            return buf[base: base + 4 * words].view(torch.int32).cpu().numpy().view(np.uint32)

        off = [C.c_size_t() for _ in range(5)]
        gn.check(gn.lib.gs_binning_state_layout(info["binning_capacity"], W, Hh, *[C.byref(x) for x in off]), "layout")
        assert np.array_equal(part(binning, off[0].value, R), want["point_list"])
        assert np.array_equal(part(binning, off[1].value, 2 * R).view(np.uint64), want["keys"])
        gn.check(gn.lib.gs_image_state_layout(W, Hh, *[C.byref(x) for x in off]), "layout")
        assert np.array_equal(part(img, off[3].value, 2 * gx * gy), want["ranges"].reshape(-1))
        goff = [C.c_size_t() for _ in range(3)]
        gn.check(gn.lib.gs_geometry_state_layout(P, *[C.byref(x) for x in goff]), "layout")
        assert np.array_equal(part(geom, goff[1].value, P), want["point_offsets"])
