"""The built code of the kernels that read LDS by asm: what the compiler may not do while such a read is on its way."""
import os
import re
import subprocess

import pytest

from microllm_rocm_amd.ops import library

READ = re.compile(r"ds_read_b128 v\[(\d+):(\d+)\]")
BRANCH = re.compile(r"s_(c?branch|setpc|call|endpgm)")


def registers(text):
    out = set()
    for first, last in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        out.update(range(int(first), int(last) + 1))
    return out | {int(number) for number in re.findall(r"\bv(\d+)\b", text)}


def faults(lines):
    """Reads by asm seen, and the lines of one kernel that stand between such a read and the wait for it and may not: a branch, a place that is
    branched to, or an instruction of the compiler's that names a register the read writes."""
    on_their_way, in_asm, reads, found = set(), False, 0, []
    for line in lines:
        text = line.split("//")[0].strip()
        if text.startswith(";"):
            in_asm = "ASMSTART" in text or (in_asm and "ASMEND" not in text)
            continue
        text = text.split(";")[0].strip()
        if not text:
            continue
        read = READ.match(text) if in_asm else None
        if read:
            if registers(read.group(0)) & on_their_way:
                found.append(text)
            on_their_way.update(range(int(read.group(1)), int(read.group(2)) + 1))
            reads += 1
        elif text.startswith("s_waitcnt") and "lgkmcnt(0)" in text:
            on_their_way = set()
        elif on_their_way and (text.endswith(":") or BRANCH.match(text) or (not text.startswith(".") and registers(text) & on_their_way)):
            found.append(text)
    return reads, found


def test_what_is_found():
    read, wait = [";;#ASMSTART", "ds_read_b128 v[4:7], v1 offset:16", ";;#ASMEND"], ["s_waitcnt vmcnt(4) lgkmcnt(0)"]
    product = ["v_mfma_f32_16x16x32_bf16 v[20:23], v[8:11], v[12:15], v[20:23]"]
    assert faults(read + product + wait + ["v_mov_b32 v4, v5", "s_cbranch_scc1 .LBB0_2"]) == (1, [])
    assert faults(read + ["v_mov_b32_e32 v9, v6"] + wait)[1] and faults(read + ["s_cbranch_vccnz .LBB0_3"] + wait)[1] and faults(read + [".LBB0_3:"] + wait)[1]
    assert faults(read + ["s_waitcnt vmcnt(0)"] + read + wait)[1]
    assert faults(["ds_read_b128 v[4:7], v1", "s_branch .LBB0_1"]) == (0, [])      # the compiler's own reads are its own to wait for


@pytest.mark.parametrize("source,kernel", [("gemm_tiled", "gemm_tiled_kernel"), ("moe_tiled", "moe_tiled_kernel")])
def test_no_branch_and_no_copy_while_operands_are_on_their_way(source, kernel, tmp_path):
    try:
        hipcc = library._hipcc()
    except library.KernelLibraryError:
        pytest.skip("no hipcc here")
    target = tmp_path / f"{source}.s"
    subprocess.run([hipcc, *library.HIPCC_FLAGS, "-S", "--cuda-device-only", os.path.join(library.CSRC, f"{source}.hip"), "-o", str(target)],
                   check=True, capture_output=True)
    bodies = re.findall(r"^(_Z\w*" + kernel + r"\w*):[^\n]*\n(.*?)^\.Lfunc_end", target.read_text(), re.S | re.M)
    assert bodies
    for name, body in bodies:
        reads, found = faults(body.split("\n"))
        assert reads > 0 and not found, (name, found[:5])
