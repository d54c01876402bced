"""The built library's device code, read back as assembly on the CPU."""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from litevllm import _hip

OBJDUMP = Path(shutil.which("hipcc") or "/opt/rocm/bin/hipcc").resolve().parent.parent \
    / "llvm" / "bin" / "llvm-objdump"
LOAD_TO_LDS = re.compile(r"(global|buffer|scratch)_load\S*_lds_|buffer_load.*\blds\b")
WRITES_M0 = re.compile(r"s_\w+ m0\b")


@pytest.fixture(scope="module")
def device_code(tmp_path_factory):
    """{code object: its instructions in order}"""
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    if not _hip.LIB_PATH.exists():
        pytest.skip("the library is not built")
    work = tmp_path_factory.mktemp("code")
    lib = work / _hip.LIB_PATH.name
    shutil.copy(_hip.LIB_PATH, lib)
    subprocess.run([str(OBJDUMP), "--offloading", lib.name], cwd=work, check=True,
                   capture_output=True)
    out = {}
    for obj in sorted(work.glob("*gfx950")):
        text = subprocess.run([str(OBJDUMP), "-d", "--no-show-raw-insn", str(obj)], check=True,
                              capture_output=True, text=True).stdout
        out[obj.name] = [line.split("//")[0].strip() for line in text.splitlines()
                         if line.startswith("\t")]
    assert out
    return out


def test_wait_state_between_m0_and_loads_into_lds(device_code):
    """One instruction at least between a scalar write of M0 and a load into
    LDS, which takes its address from M0: the hardware needs a wait state there,
    and the compiler puts none into inline assembly."""
    loads, bad = 0, []
    for name, code in device_code.items():
        for prev, insn in zip(code, code[1:]):
            if LOAD_TO_LDS.search(insn):
                loads += 1
                if WRITES_M0.match(prev):
                    bad.append((name, prev, insn))
    assert loads > 0
    assert not bad, (len(bad), bad[:4])
