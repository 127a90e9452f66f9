"""CPU checks of the gfx950 code in the built library, by disassembling it."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from yirage_amd import _lib

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """Instruction lines of each code object of the library."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = str(tmp_path_factory.mktemp("code"))
    shutil.copy(_lib.LIB_PATH, os.path.join(d, "lib.so"))
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    objs = sorted(glob.glob(os.path.join(d, "*gfx950*")))
    assert objs
    out = []
    for o in objs:
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", o], capture_output=True, text=True, check=True)
        out.append([ln.split("//")[0].strip() for ln in r.stdout.splitlines()])
    return out


def test_lds_loads_wait_for_m0(code):
    """A load into LDS takes its LDS address from M0: on gfx9 at least one wait
    state lies between a scalar write of M0 and the load.  Inside inline
    assembly the compiler adds none."""
    loads, bad = 0, []
    for lines in code:
        for i, ln in enumerate(lines):
            if not (re.match(r"buffer_load_\S+ .*\blds$", ln) or ln.startswith("global_load_lds_")):
                continue
            loads += 1
            if re.match(r"s_\w+ m0\b", lines[i - 1]):
                bad.append((lines[i - 1], ln))
    assert loads > 1000
    assert not bad, f"{len(bad)} of {loads}, e.g. {bad[0]}"
