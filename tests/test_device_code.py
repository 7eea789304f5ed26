"""What the compiled device code of libprt_hip.so (built here from csrc/) may not
hold."""
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def code_objects(prt, tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("llvm-objdump not available")
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(prt.LIB_PATH, where)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=where, timeout=60)
    return sorted(str(f) for f in where.iterdir() if "gfx950" in f.name)


def kernels(code_objects, pattern):
    """Assembly of the kernels whose mangled name matches."""
    out = {}
    for path in code_objects:
        table = subprocess.run([OBJDUMP, "-t", path], check=True, capture_output=True, text=True, timeout=60).stdout
        names = [ln.split()[-1] for ln in table.splitlines() if re.search(pattern, ln) and not ln.endswith(".kd")]
        if names:
            text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(names), path], check=True,
                                  capture_output=True, text=True, timeout=120).stdout
            for part in re.split(r"\n(?=[0-9a-f]+ <)", text)[1:]:
                out[part.split("<")[1].split(">")[0]] = part
    return out


def test_queries_raise_their_flag_by_a_store(code_objects):
    """The error flag of a small host query is in pinned host memory, where an
    atomic OR need not take effect."""
    found = kernels(code_objects, r"k_traceILb[01]ELi[07]E")    # closest and any hit, timed and instrumented
    assert len(found) == 4
    for name, text in found.items():
        assert "s_endpgm" in text and "atomic_or" not in text, name
