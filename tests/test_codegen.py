"""Counts in the built device code that a kernel's hand-written waits rely on.

A wait with a non-zero count is right only while the compiler keeps at least
that many memory operations between it and the copies it is for, so those are
counted in the disassembly of the library that the tests run.  CPU only.
"""
import re
import subprocess
from pathlib import Path

import pytest

from mosaic_amd import _lib, build

LLVM = Path("/opt/rocm/llvm/bin")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    objdump = LLVM / "llvm-objdump"
    if not objdump.exists():
        pytest.skip("llvm-objdump is not installed")
    if not _lib.LIB_PATH.exists():
        build.build()
    work = tmp_path_factory.mktemp("offload")
    lib = work / "lib.so"
    lib.symlink_to(_lib.LIB_PATH)
    subprocess.run([objdump, "--offloading", lib], cwd=work, check=True, capture_output=True)
    return sorted(work.glob("*gfx950"))


def _kernels(code_objects, name: str) -> dict:
    """symbol -> its instructions ("mnemonic operands"), over every instance of a kernel template"""
    found = {}
    for obj in code_objects:
        syms = subprocess.run([LLVM / "llvm-objdump", "-t", obj], check=True, capture_output=True, text=True).stdout
        for sym in re.findall(rf" F \.text\t.* (\S*{name}\S*)$", syms, re.M):
            asm = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", f"--disassemble-symbols={sym}",
                                  obj], check=True, capture_output=True, text=True).stdout
            found[sym] = [ln.split("//")[0].strip() for ln in asm.splitlines() if ln.startswith("\t")]
    return found


def test_mla_whole_split_q_wait(code_objects):
    """Between q's last copy into LDS and the wait for it lie, without a branch, at least as many vector
    loads as the wait leaves in flight."""
    kernels = _kernels(code_objects, "mla_decode_chunk_kernel")
    assert len(kernels) == 2  # bf16 and fp32 partials
    for sym, ins in kernels.items():
        last = max(i for i, x in enumerate(ins) if x.startswith("global_load_lds"))
        wait = next(i for i in range(last, len(ins)) if ins[i + 1].startswith("s_barrier"))
        left = int(re.fullmatch(r"s_waitcnt vmcnt\((\d+)\)", ins[wait]).group(1))
        between = ins[last + 1:wait]
        assert not any(x.startswith(("s_cbranch", "s_branch")) for x in between), sym
        assert sum(x.startswith("global_load") for x in between) >= left > 0, sym
