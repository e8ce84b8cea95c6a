"""The rules by which the runtime keeps freed device blocks
(kokkos_amd/csrc/block_cache.hpp), on the CPU against a model of the HIP calls
(tests/cpp/block_cache.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CXX = shutil.which("g++") or shutil.which("c++")


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    if not CXX:
        pytest.skip("no host compiler")
    exe = tmp_path_factory.mktemp("block_cache") / "block_cache"
    cmd = [CXX, "-std=c++17", "-O1", "-Wall", "-I", str(ROOT / "kokkos_amd" / "csrc"),
           str(ROOT / "tests" / "cpp" / "block_cache.cpp"), "-o", str(exe), "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


@pytest.mark.parametrize("name", ["huge_requests", "devices", "recording", "freed_in_stream_order", "freed_twice", "no_memory", "rules"])
def test_block_cache(checks, name):
    r = subprocess.run([str(checks), name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
