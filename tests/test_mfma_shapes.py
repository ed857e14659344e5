"""No accumulator of the built kernels passes between MFMAs of two shapes.

An MFMA that takes the result of one of another shape as its accumulator (SrcC)
reads half of it before it is complete unless enough instructions lie between,
and the compiler puts no wait there: back to back v_mfma_f32_16x16x32_f16 and
v_mfma_f32_16x16x16_f16 gave wrong values in two of the four registers on an
MI355X.  Whether a kernel is hit then hangs on its schedule alone, so parity tests
of one build say nothing about the next.  This test reads the instructions of the
objects that the build leaves in _build/ (CPU only).
"""
import glob
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = "/opt/rocm/llvm/bin"
OBJECTS = [os.path.join(ROOT, "_build", f"nx_{n}.o") for n in ("mfd", "mfv", "gemm", "logits")]


def registers(operand):
    m = re.match(r"([va])\[(\d+):(\d+)\]", operand)
    return frozenset(f"{m[1]}{i}" for i in range(int(m[2]), int(m[3]) + 1)) if m else frozenset()


def mixed_chains(lines):
    """(function, instruction) of each MFMA whose accumulator an MFMA of another
    shape wrote last, in the order of the listing."""
    found, function, wrote, count = [], None, {}, 0
    for line in lines:
        m = re.match(r"[0-9a-f]* ?<(\S+)>:|^(_Z\w+):", line)
        if m:
            function, wrote = m[1] or m[2], {}
            continue
        text = line.split("//")[0].split(";")[0].strip()
        op, _, rest = text.partition(" ")
        operands = [o.strip() for o in re.split(r",(?![^\[]*\])", rest)]
        if op.startswith("v_mfma"):
            count += 1
            last = {wrote[r] for r in registers(operands[3]) if r in wrote}
            if last - {op}:
                found.append((function, text))
            wrote.update({r: op for r in registers(operands[0])})
        elif op.startswith(("v_", "ds_read", "buffer_load", "global_load")) and operands:
            single = re.match(r"[va]\d+$", operands[0])
            for r in registers(operands[0]) | ({single[0]} if single else set()):
                wrote.pop(r, None)
    return found, count


def disassembly(obj, tmp_path):
    fat, elf = tmp_path / "fat", tmp_path / "elf"
    for cmd in ([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", obj, str(tmp_path / "copy.o")],
                [f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={elf}",
                 "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"]):
        subprocess.run(cmd, check=True, capture_output=True)
    return subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", str(elf)], check=True,
                          capture_output=True, text=True).stdout.splitlines()


@pytest.mark.skipif(not all(map(os.path.exists, OBJECTS + [f"{LLVM}/clang-offload-bundler"])),
                    reason="no built objects (run nexus_amd.build() first) or no ROCm LLVM tools")
@pytest.mark.parametrize("obj", OBJECTS, ids=os.path.basename)
def test_one_shape_per_accumulator(obj, tmp_path):
    found, count = mixed_chains(disassembly(obj, tmp_path))
    assert count > 0
    assert not found, found[:4]


def test_finds_a_mixed_chain():
    same = ["<f>:", "v_mfma_f32_16x16x32_f16 v[0:3], v[8:11], v[12:15], 0",
            "v_mfma_f32_16x16x32_f16 v[0:3], v[8:11], v[12:15], v[0:3]"]
    mixed = "v_mfma_f32_16x16x16_f16 v[0:3], v[8:9], v[12:13], v[0:3]"
    assert mixed_chains(same) == ([], 2)
    assert mixed_chains(same + ["v_add_f32_e32 v5, v6, v7", mixed]) == ([("f", mixed)], 3)
    assert mixed_chains(same + [f"v_mov_b32_e32 v{i}, 0" for i in range(4)] + [mixed])[0] == []
    assert mixed_chains(same + ["<g>:", mixed])[0] == []
