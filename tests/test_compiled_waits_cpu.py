"""Waits and registers of the compiled kernels, read from the built library's gfx950 code (no GPU).

The write-through stores are inline assembly, which the compiler does not count as memory
operations in flight: it drops the wait of a fence that follows nothing else.  So every fence of
the one-launch normalised GAE (finish_normalized in csrc/rlk_engine.hpp), whose raw advantages
other workgroups read, has to carry a wait of its own."""
import os
import re
import shutil
import subprocess

import pytest

from rl_triton import _native

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READOBJ = "/opt/rocm/llvm/bin/llvm-readobj"


def _code_objects(tmp_path):
    lib = shutil.copy(_native.library_path(), tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], check=True, stdout=subprocess.DEVNULL)
    return sorted(tmp_path.glob("lib.so.*gfx950"))


def _device_code(tmp_path):
    """(kernel, its instructions) of every kernel in the library."""
    for part in _code_objects(tmp_path):
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(part)], check=True, capture_output=True,
                             text=True).stdout
        for m in re.finditer(r"^[0-9a-f]+ <(_ZN\S+)>:\n((?:(?!^[0-9a-f]+ <_ZN).*\n)*)", out, re.M):
            yield m[1], [line.split("//")[0].strip() for line in m[2].splitlines()]


def _unwaited_fences(code):
    """Release fences (a write-back that no atomic operation follows at once) from which an
    s_barrier is reached without a wait for all vector memory operations."""
    bad = []
    for i, op in enumerate(code):
        if not op.startswith("buffer_wbl2"):
            continue
        for nxt in code[i + 1:i + 40]:
            if re.match(r"s_waitcnt.*vmcnt\(0\)", nxt) or "_atomic_" in nxt:
                break
            if nxt.startswith(("s_barrier", "s_endpgm")):
                bad.append(i)
                break
    return bad


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_one_launch_fences_wait_for_the_stores_before_them(tmp_path):
    fences, bad = 0, []
    for kernel, code in _device_code(tmp_path):
        if "OneLaunchOp" in kernel:
            fences += sum(op.startswith("buffer_wbl2") for op in code)
            bad += [kernel] * bool(_unwaited_fences(code))
    assert fences > 0
    assert not bad, bad


@pytest.mark.skipif(not os.path.exists(READOBJ), reason="no llvm-readobj")
def test_lookback_publish_address_stays_in_registers(tmp_path):
    """Aligned float32 V-trace tiles of 8192 steps have registers to spare; with the publish address
    formed under each branch of tile_carry they spilled it, and reloaded it ahead of every publish
    (2% of a [16,131072] call)."""
    spills = {}
    for part in _code_objects(tmp_path):
        notes = subprocess.run([READOBJ, "--notes", str(part)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split(".agpr_count")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)[1]
            spills[name] = int(re.search(r"\.sgpr_spill_count:\s+(\d+)", kernel)[1])
    tiles = {k: n for k, n in spills.items() if "chain_kernelINS_8VtraceOpILb0EfEELi1024ELi2ELi1E" in k}
    assert tiles and not any(tiles.values()), tiles
