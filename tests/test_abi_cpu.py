"""CPU-only checks of the C ABI: the library loads, exports every symbol the
public header declares, and its host-only helpers agree with the oracle.  No
kernel is launched here."""
import ctypes as C
import os
import re

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "gsrast.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gs_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    import gsrast_native as gn
    names = _declared()
    assert len(names) >= 26
    for n in names:
        assert hasattr(gn.lib, n), f"{n} is declared in include/gsrast.h but not exported by libgsrast.so"
    assert set(names) == set(gn.EXPORTED_SYMBOLS), set(names) ^ set(gn.EXPORTED_SYMBOLS)


def test_host_helpers(orc):
    import gsrast_native as gn
    for n in [0, 1, 2, 3, 1200, 3888, 8160, 65535, 65536, 2 ** 31]:
        assert gn.lib.gs_higher_msb(n) == orc.higher_msb(n)
    bx, by, od = C.c_int(), C.c_int(), C.c_int()
    assert gn.lib.gs_get_block_xy(C.byref(bx), C.byref(by), C.byref(od)) == 0
    assert (bx.value, by.value, od.value) == (16, 16, 256)
    assert gn.lib.gs_get_block_xy(None, None, None) != 0 and "null" in gn.last_error()


def test_state_layouts_are_aligned_and_disjoint():
    import gsrast_native as gn
    sz = [C.c_size_t() for _ in range(5)]
    assert gn.lib.gs_image_state_layout(1152, 864, *[C.byref(s) for s in sz]) == 0
    a, nc, n2, rg, tot = [s.value for s in sz]
    N = 1152 * 864
    assert a % 256 == nc % 256 == n2 % 256 == rg % 256 == 0
    assert nc >= a + 4 * N and n2 >= nc + 4 * N and rg >= n2 + 4 * N and tot >= rg + 8 * 72 * 54
    assert gn.lib.gs_binning_state_layout(1_771_093, 1152, 864, *[C.byref(s) for s in sz]) == 0
    pl, k, plu, ku, tot = [s.value for s in sz]
    R = 1_771_093
    offs = sorted([(pl, 4 * R), (k, 8 * R), (plu, 4 * R), (ku, 8 * R)])
    for (o1, l1), (o2, _) in zip(offs, offs[1:]):
        assert o1 + l1 <= o2 and o1 % 256 == 0
    assert tot > offs[-1][0] + offs[-1][1]
    assert gn.lib.gs_scan_workspace_bytes(10_000_000) >= 4 * (10_000_000 // 2048)
    assert gn.lib.gs_sort_workspace_bytes(R) >= 256 * 4 * (R // 2048)
    assert gn.lib.gs_knn_workspace_bytes(1000) > 1000 * 16


def test_layouts_and_capacities_at_the_instance_limit():
    """A view may hold up to 2^31-2 instances: at that count every array of the binning buffer still starts
    behind the one before it (no offset is formed in 32 bits), the per-instance workspaces are sized in 64 bits,
    and the radix sort over all keys, whose capacity is 2^30-2 pairs, refuses more before launching anything."""
    import gsrast_native as gn
    R = 2 ** 31 - 2
    sz = [C.c_size_t() for _ in range(5)]
    assert gn.lib.gs_binning_state_layout(R, 1920, 1080, *[C.byref(s) for s in sz]) == 0
    pl, k, plu, ku, tot = [s.value for s in sz]
    offs = sorted([(pl, 4 * R), (k, 8 * R), (plu, 4 * R), (ku, 8 * R)])
    for (o1, l1), (o2, _) in zip(offs, offs[1:]):
        assert o1 + l1 <= o2 and o1 % 256 == 0
    # point list, keys, 16-byte records, emission indices, block hits, 24 bytes of per-tile radix sort scratch
    assert tot >= (4 + 8 + 16 + 4 + 2 + 24) * R
    assert gn.lib.gs_render_backward_workspace_bytes(R) == 64 * R + 256
    assert gn.lib.gs_sort_max_pairs() == 2 ** 30 - 2
    assert gn.lib.gs_sort_workspace_bytes(2 ** 30 - 2) > 5 * 512 * 4 * ((2 ** 30 - 2) // 4096)
    one = C.c_void_p(256)  # never dereferenced: the count is refused first
    assert gn.lib.gs_sort_pairs_u64(2 ** 30 - 1, one, one, one, one, 44, one, 1 << 40, None) != 0
    assert "2^30-2" in gn.last_error()
    assert gn.lib.gs_sort_pairs_u32(2 ** 31, one, one, one, one, 32, one, 1 << 40, None) != 0
    assert "2^30-2" in gn.last_error()


def test_argument_validation_without_a_gpu():
    import gsrast_native as gn
    assert gn.lib.gs_preprocess_forward(*([None] * 8), 10, 3, 16, 0, 480, *([None] * 5), 1.0, None, None, None, 0.5, 0.5,
                                        0, 0, None, None, None) != 0
    assert "bad sizes" in gn.last_error()
    assert gn.lib.gs_sort_pairs_u64(5, None, None, None, None, 70, None, 0, None) != 0
    assert "end_bit" in gn.last_error()
    assert gn.lib.gs_mark_visible(0, None, None, None, None, None) == 0  # empty input is a no-op


def test_python_modules_refuse_cpu_tensors():
    import pytest
    import torch
    from diff_gaussian_rasterization import GaussianRasterizationSettings, GaussianRasterizer
    from simple_knn._C import distCUDA2
    rs = GaussianRasterizationSettings(32, 32, 0.5, 0.5, torch.zeros(3), 1.0, torch.eye(4), torch.eye(4), 3,
                                       torch.zeros(3), False, True, False)
    rast = GaussianRasterizer(rs)
    z = torch.zeros
    with pytest.raises(RuntimeError, match="no CPU path"):
        rast.preprocess_gaussians(z(4, 3), z(4, 3), z(4, 4), z(4, 3), z(4, 1), {})
    with pytest.raises(RuntimeError, match="no CPU path"):
        distCUDA2(z(10, 3))


def test_tensors_the_kernels_use_in_place_are_checked():
    """What preprocess and render read or write without a copy of their own is refused unless it has the rows the
    kernels address; looked at before anything else, so the refusal is seen without a GPU."""
    import pytest
    import torch
    import gsrast_native as gn
    P = 6
    z = torch.zeros
    cam = (z(4, 4), z(4, 4))

    def forward(records=None, all_map=None):
        gn.ops.preprocess_forward(z(P, 3), z(P, 3), z(P, 4), None, z(P, 1), 1.0, *cam, z(3), 0.5, 0.5, 32, 32, 0, False,
                                  False, False, False, records, all_map, 0)

    def backward(ddir=None, gmap=None):
        gn.ops.preprocess_backward(z(P, dtype=torch.int32), None, z(P, 3, dtype=torch.bool), z(P, 3), z(P, 3), z(P, 4),
                                   z(P, 16, 3), 1.0, *cam, 0.5, 0.5, 32, 32, 0, z(3), z(P, 2), z(P, 4), None, False, ddir,
                                   gmap, 0)

    def render_backward(records):
        u8 = z(16, dtype=torch.uint8)
        gn.ops.render_backward(z(3), 0.5, 0.5, None, None, 0, u8, u8, u8, z(4, dtype=torch.bool), z(3, 32, 32), None,
                               None, z(P, 2), z(P, 4), z(P, 3), False, False, False, 0, records, 0)

    for call, name, shape in ((lambda t: forward(records=t), "blend_records", (P, 16)),
                              (lambda t: forward(all_map=t), "all_map", (P, 5)),
                              (lambda t: backward(ddir=t), "dcolor_ddir", (P, 3, 3)),
                              (render_backward, "blend_records", (P, 16))):
        short = z(P - 1, *shape[1:])
        strided = z(*shape[:-1], 2 * shape[-1])[..., ::2]
        for bad in (short, strided, z(*shape, dtype=torch.float64), z(*shape, device="meta"), z(P * 16)):
            with pytest.raises(RuntimeError, match=f"{name} must be a contiguous"):
                call(bad)
        with pytest.raises(RuntimeError, match="no CPU path"):
            call(z(*shape))
    for bad in (z(P - 1, 5), z(P, 4), z(P, 5, device="meta")):
        with pytest.raises(RuntimeError, match="dL_dall_map must have shape"):
            backward(gmap=bad)
    with pytest.raises(RuntimeError, match="no CPU path"):
        backward(gmap=z(P, 10)[:, ::2])  # (made contiguous by the call)


def test_the_table_needs_neither_torch_nor_the_torch_extension():
    """gsrast_native is what any caller of the C ABI can use: the library and its table of argument types."""
    import subprocess
    import sys
    code = """
import sys
sys.modules["torch"] = None  # (import torch raises)
sys.path.insert(0, %r)
import gsrast_native as gn
gn.OPS_PATH = "/nowhere/gsrast_ops.so"
assert gn.lib.gs_higher_msb(8160) == 13 and len(gn.EXPORTED_SYMBOLS) > 25
gn.RenderOptions(), gn.RenderResult()
for name in ("ops", "stream_handle"):
    try:
        getattr(gn, name)
    except ImportError:
        continue
    raise SystemExit(name)
assert not hasattr(gn, "nothing_of_that_name")
""" % os.path.join(ROOT, "citygs-x_amd")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.stdout, r.stderr)


def test_adam_steps_of_any_size_fit_their_launches():
    """A launch has fewer than 2^32 threads; 2^34 elements of four arrays fit the card's memory."""
    import gsrast_native as gn
    for sizes in ([], [0, -1], [1], [511, 512, 513, 0, 5], [2 ** 34 + 77], [2 ** 33, 2 ** 33, 0, 3],
                  [2 ** 29], [2 ** 29 + 1, 7], [2 ** 29 - 512, 512, 1], [2 ** 29 - 511, 512], [100] * 70, [2 ** 28] * 40):
        n = len(sizes)
        out = (C.c_longlong * 2000)()
        rows = gn.lib.gs_selftest_adam_plan(n, (C.c_longlong * max(n, 1))(*sizes), out, 400)
        assert rows <= 400
        table = np.array(out[:5 * rows], np.int64).reshape(rows, 5)
        done = [0] * n
        for launch, tensor, first, elements, threads in table:
            assert first == done[tensor] and first % 4 == 0 and elements > 0  # (16-byte accesses stay aligned)
            done[tensor] += int(elements)
            assert 0 < threads < 2 ** 32
        assert done == [max(k, 0) for k in sizes]
        for launch in set(table[:, 0].tolist()):
            mine = table[table[:, 0] == launch]
            # 128 threads per 512 elements of a slice; a launch follows when the one before it is full
            assert (mine[:, 4] == 128 * ((mine[:, 3] + 511) // 512).sum()).all()
        assert (np.diff(table[:, 0]) >= 0).all() and (np.diff(table[:, 0]) <= 1).all()
    one = (C.c_longlong * 1)(7)
    assert gn.lib.gs_selftest_adam_plan(1, None, one, 0) == -1 and gn.lib.gs_selftest_adam_plan(1, one, None, 1) == -1
    assert gn.lib.gs_selftest_adam_plan(1, one, None, 0) == 1
