"""Kernels that pass a barrier with loads under way wait with bare instructions and not with a fence, so the compiler
does not see to it that what a wave has read of LDS is in its registers when another wave writes over it.  The
instructions of those kernels say whether it is: no access to LDS may be under way at a barrier."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from kappai_amd.kernels import lib

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


def accesses_under_way(listing):
    """For each kernel the number of LDS accesses that may be under way at each barrier, in the order of the text."""
    kernels, name, under_way = {}, None, 0
    for line in listing:
        label = re.match(r"[0-9a-f]+ <(\w+)>:", line)
        op = line.split("//")[0].strip()
        wait = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", op)
        if label:
            name, under_way = label.group(1), 0
            kernels[name] = []
        elif op.startswith("ds_"):
            under_way += 1
        elif wait:
            under_way = min(under_way, int(wait.group(1)))
        elif op == "s_barrier":
            kernels[name].append(under_way)
    return kernels


def built(name, defines):
    return (lib._find_built(lib._built_name(name, defines), lib._source_hash(name, defines))
            or lib.compile_library(name, verbose=False, defines=defines))


@pytest.mark.skipif(not OBJDUMP.exists(), reason="no disassembler")
@pytest.mark.parametrize("name,defines", [("attention_mfma", {"HEAD_DIM": 64}), ("attention_mfma", {"HEAD_DIM": 128}),
                                          ("attention_mfma", {"HEAD_DIM": 256}), ("gemm", None), ("mingru", None)])
def test_no_access_to_lds_is_under_way_at_a_barrier(tmp_path, name, defines):
    shutil.copy(built(name, defines), tmp_path / "kernels.so")
    subprocess.run([OBJDUMP, "--offloading", "kernels.so"], cwd=tmp_path, check=True, capture_output=True)
    code, = tmp_path.glob("kernels.so*gfx950")
    text = subprocess.run([OBJDUMP, "-d", code], check=True, capture_output=True, text=True).stdout
    kernels = accesses_under_way(text.splitlines())
    assert any(kernels.values())
    assert {k: v for k, v in kernels.items() if any(v)} == {}
