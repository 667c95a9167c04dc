"""Hazards in the built library's own device code that the compiler cannot see inside inline asm."""
import os
import re
import shutil
import subprocess

import pytest

from shardcompute_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def device_code(tmp_path_factory):
    """One list of instructions (text, in address order) per code object of the library."""
    if not os.path.exists(build.LIB_PATH):
        build.build()
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("device_code")
    lib = shutil.copy(build.LIB_PATH, d)             # the bundles are extracted beside it
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=d)
    out = []
    for f in sorted(d.iterdir()):
        if f.name.endswith("gfx950"):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True,
                                  text=True).stdout
            out.append([line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")])
    assert out
    return out


def test_lds_dma_keeps_its_wait_state_after_m0(device_code):
    """An LDS-DMA takes its LDS base from M0 and needs one wait state after a scalar write of
    it (gfx9): with the two back to back it may still read the previous base and land in
    another slot."""
    writes, dmas, bad = 0, 0, []
    for code in device_code:
        for first, second in zip(code, code[1:]):
            dma = re.match(r"global_load_lds_|buffer_load_\w+ .*\blds$", second) is not None
            m0 = re.match(r"s_\w+ m0,", first) is not None
            writes, dmas = writes + m0, dmas + dma
            if m0 and dma:
                bad.append((first, second))
    assert writes > 100 and dmas > 100, (writes, dmas)
    assert not bad, (len(bad), bad[0])
