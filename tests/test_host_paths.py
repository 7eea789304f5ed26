"""Host control flow of the library on the CPU: the entry points and the host
copies compiled against a stand-in for the HIP runtime (tests/native), which
can be a smaller device, run out of memory and show each copy."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("native") / "host_paths")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-pthread", "-I", NATIVE,
                    os.path.join(NATIVE, "host_paths.cpp"), "-o", out], check=True, timeout=300)
    return out


@pytest.mark.parametrize("name", [
    "small_query_on_small_devices",
    "small_query_memory",
    "bad_ray_counts",
    "no_pinned_memory",
    "host_copies",
    "pinned_caller",
    "copy_threads",
    "work_deal",
    "no_room_for_the_lookahead",
    "no_room_for_the_hit_record",
    "half_a_frame",
    "replaced_buffers",
    "kept_memory",
])
def test_host_path(exe, name):
    r = subprocess.run([exe, name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
