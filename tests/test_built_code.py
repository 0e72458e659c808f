"""Properties of the built gfx950 code that its sources can only ask for: read from a disassembly of the library."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from acache_amd import _lib

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and Path(p).exists()), None)


def instructions(library, folder):
    """(kernel, instruction) of every code object of the library, in order."""
    shutil.copy(library, folder / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    for part in sorted(folder.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", part.name], cwd=folder, check=True, capture_output=True, text=True)
        kernel = None
        for line in text.stdout.splitlines():
            head = re.match(r"[0-9a-f]+ <(\w+)>:", line)
            if head:
                kernel = head.group(1)
            elif line.startswith("\t"):
                yield kernel, line.split("//")[0].strip()


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_scalar_bases_of_copies_come_from_the_instruction_in_front(tmp_path):
    """A vector memory instruction must not read a scalar register in the five wait states after a vector instruction wrote it
    (a reload of a spilled one is such a write).  The compiler does not look into inline assembly, so every copy that has a
    scalar base moves it itself, right in front: what a scalar instruction writes needs no wait."""
    before, found = "", 0
    for kernel, text in instructions(_lib.LIB_PATH, tmp_path):
        copy = re.match(r"global_load_lds_dword\w* v\d+, (s\[\d+:\d+\])", text)
        if copy:
            found += 1
            assert before.startswith(f"s_mov_b64 {copy.group(1)}, "), (kernel, before, text)
        before = text
    assert found > 100
