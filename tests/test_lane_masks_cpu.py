"""The built kernels, as a listing: gfx950 wants two issue slots between a vector instruction that writes a lane mask (VCC
or a pair of scalar registers) and a vector instruction that reads it.  The compiler sees to that in the code it writes
itself, and does not look into inline assembly."""
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "citygs-x_amd", "lib", "libgsrast.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def masks(operand):
    if operand in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc"}
    m = re.match(r"^s\[(\d+):(\d+)\]$", operand) or re.match(r"^s((\d+))$", operand)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


def short_gaps(listing):
    """(kernel, writer, reader, slots between) of every pair that is less than two slots apart, and the number of pairs."""
    kernel, slot, written, pairs, short = None, 0, {}, 0, []
    for line in listing.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.*)>:", line)
        if head:
            kernel, written = head.group(1), {}
            continue
        m = re.match(r"^\s+(\S+)\s*(.*?)\s*//", line)
        if not m:
            continue
        op, operands = m.group(1), [o.split()[0] for o in m.group(2).split(",") if o.split()]
        if op == "s_nop":
            slot += int(operands[0], 0) + 1
            continue
        slot += 1
        if op.startswith(("s_branch", "s_endpgm", "s_setpc")):
            written = {}  # what follows is reached from elsewhere
        if not op.startswith("v_"):
            continue
        results = 2 if re.search(r"_co_u32|div_scale|mad_[ui]64", op) else 1
        read = set().union(*[masks(o) for o in operands[results:]])
        if op == "v_cndmask_b32_e32" or op.startswith("v_div_fmas"):
            read.add("vcc")
        for r in read & set(written):
            pairs += 1
            if slot - written[r][0] - 1 < 2:
                short.append((kernel, written[r][1], op, slot - written[r][0] - 1))
        for o in operands[:results]:
            for r in masks(o):
                written[r] = (slot, op)
    return short, pairs


def test_the_reader_of_the_listing():
    line = lambda text: "\t" + text + "    // 000000000000: 00000000\n"
    head = "0000000000001000 <kernel>:\n"
    pair = line("v_cmp_ngt_f32_e32 vcc, v1, v2"), line("v_addc_co_u32_e32 v0, vcc, v0, v0, vcc")
    assert short_gaps(head + "".join(pair)) == ([("kernel", "v_cmp_ngt_f32_e32", "v_addc_co_u32_e32", 0)], 1)
    assert len(short_gaps(head + pair[0] + line("s_nop 0") + pair[1])[0]) == 1
    assert short_gaps(head + pair[0] + line("s_nop 1") + pair[1]) == ([], 1)
    far = line("v_cmp_lt_f32_e64 s[4:5], v1, v2"), line("v_cndmask_b32_e64 v0, v1, v2, s[4:5]")
    assert len(short_gaps(head + far[0] + line("v_mov_b32_e32 v9, v8") + far[1])[0]) == 2  # (both halves of the pair)
    assert short_gaps(head + far[0] + 2 * line("v_mov_b32_e32 v9, v8") + far[1]) == ([], 2)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_lane_masks_are_read_two_slots_after_they_are_written(tmp_path):
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(p for p in tmp_path.iterdir() if p.name.endswith("gfx950"))
    assert objects
    pairs = 0
    for p in objects:
        short, n = short_gaps(subprocess.run([OBJDUMP, "-d", str(p)], check=True, capture_output=True, text=True).stdout)
        assert not short, short[:10]
        pairs += n
    assert pairs > 1000  # (the listing was understood)
