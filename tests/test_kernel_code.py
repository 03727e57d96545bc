"""What the built kernels' code shows and no result does."""
import collections
import os
import re
import shutil
import subprocess

import pytest

from easyllm_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """mangled kernel name -> number of instructions"""
    if not os.path.exists(OBJDUMP) or not os.path.exists(_lib.LIB_PATH):
        pytest.skip("needs the built library and the ROCm disassembler")
    where = tmp_path_factory.mktemp("code")
    subprocess.run([OBJDUMP, "--offloading", shutil.copy(_lib.LIB_PATH, where)], cwd=where, check=True, capture_output=True)
    counts, kernel = collections.Counter(), None
    for f in os.listdir(where):
        if "gfx950" not in f:
            continue
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", f], cwd=where, check=True, capture_output=True, text=True)
        for line in out.stdout.splitlines():
            label = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if label:
                kernel = label.group(1)
            elif line.startswith("\t"):
                counts[kernel] += 1
    return counts


def test_a_k_tail_costs_the_8_wave_product_few_instructions(instructions):
    """A lane's k row is a sum of a part of its wave's and one of its own: 69 - 103 instructions more than without a tail.  Found by dividing the number
    of its chunk it was 129 - 168 with a k-major operand, and ragged weight gradients took a tenth longer."""
    pairs = 0
    for name, n in instructions.items():
        tail = re.match(r"(.*gemm_d2l_kernelILb[01]ELb[01]E(?:DF16b|f)Lb[01]E)Lb1E(.*)", name)
        if tail:
            assert n - instructions[tail.group(1) + "Lb0E" + tail.group(2)] <= 115, name
            pairs += 1
    assert pairs >= 9
