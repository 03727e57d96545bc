"""The built kernels leave a wait state between a 12- or 16-byte store and the next write of its data registers.

The compiler inserts it except where a buffer store takes its offset from a scalar register, and there the hardware needs it too
(a GEMM epilogue that overwrote the registers right behind such a store lost the last lanes of a row group)."""
import os
import re
import shutil
import subprocess

import pytest

from easyllm_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
STORE = re.compile(r"\s*(buffer|global|flat)_store_dwordx[34]\s+([^/]*)")
WRITE = re.compile(r"\s*v_(?!cmp)\S+\s+([va])(?:\[(\d+):(\d+)\]|(\d+))")
REGS = re.compile(r"([va])\[(\d+):(\d+)\]")


def overwritten_at_once(lines):
    hits = []
    for here, after in zip(lines, lines[1:]):
        m = STORE.match(here)
        if not m:
            continue
        operands = [o.strip() for o in m.group(2).split(",")]
        data = REGS.match(operands[0] if m.group(1) == "buffer" else operands[1])
        w = WRITE.match(after)
        if data and w and w.group(1) == data.group(1):
            first, last = int(w.group(2) or w.group(4)), int(w.group(3) or w.group(4))
            if first <= int(data.group(3)) and last >= int(data.group(2)):
                hits.append((here.strip(), after.strip()))
    return hits


def test_the_scan_finds_what_it_looks_for():
    assert overwritten_at_once(["\tbuffer_store_dwordx4 v[4:7], v0, s[0:3], s9 offen // x", "\tv_mov_b32_e32 v5, v1"])
    assert not overwritten_at_once(["\tbuffer_store_dwordx4 v[4:7], v0, s[0:3], s9 offen", "\tv_mov_b32_e32 v8, v5"])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs the ROCm disassembler")
def test_no_store_data_is_overwritten_in_the_next_instruction(tmp_path):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("the library has not been built")
    lib = shutil.copy(_lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    objects = [f for f in os.listdir(tmp_path) if "gfx950" in f]
    assert objects
    stores = 0
    for f in objects:
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", f], cwd=tmp_path, check=True, capture_output=True, text=True)
        lines = [x for x in out.stdout.splitlines() if x.startswith("\t")]
        stores += sum(1 for x in lines if STORE.match(x))
        hits = overwritten_at_once(lines)
        assert not hits, (len(hits), hits[:3])
    assert stores > 100
