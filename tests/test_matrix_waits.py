"""Distances around the matrix instructions of the large products, which are written as asm: the compiler keeps none for those.  Read off the
built libraries' own code: a vector instruction that writes what a matrix instruction reads stands at least 2 wait states before it, one
that reads what it wrote at least 18 behind it (a product of 8 passes)."""
import glob
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BEFORE, BEHIND = 2, 18


def registers(operand):
    m = re.fullmatch(r"([av])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if m is None:
        return set()
    first = int(m[2] or m[3])
    return {(m[1], i) for i in range(first, int(m[4] or first) + 1)}


def faults(lines):
    """{kernel: (matrix instructions, what stands too near)} of a listing's lines."""
    out, near, name = {}, [], None
    for line in lines:
        head = re.match(r"[0-9a-f]+ <(\S+)>:$", line)
        if head:
            name, near = head[1], []
            out[name] = [0, []]
        text = line.split("//")[0].strip()
        if name is None or head or not text:
            continue
        op, _, rest = text.partition(" ")
        operands = [registers(o.strip().split(" ")[0]) for o in rest.split(",")]
        if op == "s_nop":
            near = (near + [(op, set(), int(rest, 0) + 1)])[-40:]
            continue
        writes = operands[0] if op.startswith("v_") else set()
        reads = set().union(*operands[1 if op.startswith("v_") else 0:])
        matrix = op.startswith("v_mfma")
        out[name][0] += matrix
        states = 0
        for other, wrote, took in reversed(near):
            if states >= (BEFORE if matrix else BEHIND):
                break
            if other.startswith("v_") and other.startswith("v_mfma") != matrix and wrote & (reads | (set() if matrix else writes)):
                out[name][1].append(f"{other} .. {states} .. {text}")
                break
            states += took
        near = (near + [(op, writes, 1)])[-40:]
    return out


def test_the_reading_of_a_listing():
    code = ["0000 <k>:", "\tv_accvgpr_write_b32 a1, 0 // 00", "\tv_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[4:7]",
            "\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]", "\ts_nop 15", "\tv_accvgpr_read_b32 v9, a2"]
    assert faults(code) == {"k": [2, ["v_accvgpr_write_b32 .. 1 .. v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]",
                                      "v_mfma_f32_16x16x32_bf16 .. 16 .. v_accvgpr_read_b32 v9, a2"]]}
    code[1:2] += ["\ts_nop 7"]
    code[5:5] = ["\ts_nop 15"]
    assert faults(code) == {"k": [2, []]}


@pytest.mark.parametrize("module,kernels", [("product", 30), ("moe", 3)])
def test_large_products_keep_their_distances(tmp_path, module, kernels):
    from cpmcu_amd.csrc import build
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    if not build.is_built(module):
        build.build(module)
    lib = shutil.copy(build.lib_path(module), tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, cwd=tmp_path, stdout=subprocess.DEVNULL)
    lines = []
    for code in glob.glob(f"{lib}.*gfx950"):
        lines += subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout.splitlines()
    found = {k: v for k, v in faults(lines).items() if re.match(r"_Z\d+(moe_)?product_kernel", k)}
    assert len(found) >= kernels and all(n > 0 for n, _ in found.values())
    assert {k: bad[:3] for k, (_, bad) in found.items() if bad} == {}
