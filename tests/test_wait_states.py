"""Wait states that inline asm has to keep by itself, in the built GPU code.

gfx9-family GPUs need one wait state between a scalar write of M0 and a load
with LDS destination, which takes its LDS base from M0.  The compiler inserts
it for its own instructions and does not look inside inline asm, where the
delay-and-sum kernels issue their copies."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from us_lab4a_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
INSTRUCTION = re.compile(r"^\s+([a-z]\w+)\s*([^/]*)//")


def early_loads(listing):
    """(kernel, load) of every LDS load that directly follows a write of M0, and
    the number of LDS loads."""
    kernel, after_m0, loads, early = "", False, 0, []
    for line in listing:
        if line.endswith(">:\n"):
            kernel, after_m0 = line.split("<")[1][:-3], False
        m = INSTRUCTION.match(line)
        if not m:
            continue
        op, args = m.groups()
        if "load_lds_" in op or (op.startswith("buffer_load") and re.search(r"\blds\b", args)):
            loads += 1
            if after_m0:
                early.append((kernel, op))
        after_m0 = op.startswith("s_") and args.split(",")[0].strip() == "m0"
    return early, loads


def test_an_early_load_is_found():
    bad = ["0000 <k>:\n", "\ts_mov_b32 m0, s4    // 0: 00\n", "\tglobal_load_lds_dwordx4 v1, s[2:3]    // 4: 00\n"]
    good = bad[:2] + ["\ts_nop 0    // 4: 00\n", bad[2]]
    assert early_loads(bad) == ([("k", "global_load_lds_dwordx4")], 1)
    assert early_loads(good) == ([], 1)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_m0_is_written_a_wait_state_before_lds_loads(tmp_path):
    lib = shutil.copy(build.LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=tmp_path, check=True, capture_output=True)
    total = 0
    for obj in glob.glob(str(tmp_path / f"*{build.ARCH}")):
        dis = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
        early, loads = early_loads(dis.splitlines(keepends=True))
        assert not early, early[:4]
        total += loads
    assert total > 0, "no LDS loads found in the library"
