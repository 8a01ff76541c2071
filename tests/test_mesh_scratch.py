"""The store of the mesh calls' working memory (surface-remesher_amd/csrc/
mesh_scratch.cpp), compiled for the host over a runtime of the test's own
(tests/c/scratch_store.cpp): what a reset of the device or a growing mesh
does to the blocks that lie in it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    hipcc = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")
    gxx = shutil.which("g++")
    if not hipcc or not gxx:
        pytest.skip("hipcc or g++ not found")
    d = tmp_path_factory.mktemp("scratch")
    objs = []
    for src in (ROOT / "tests" / "c" / "scratch_store.cpp",
                ROOT / "surface-remesher_amd" / "csrc" / "mesh_scratch.cpp"):
        objs.append(str(d / (src.stem + ".o")))
        subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-c",
                        str(src), "-o", objs[-1]], check=True, capture_output=True, timeout=300)
    subprocess.run([gxx, *objs, "-pthread", "-o", str(d / "h")], check=True, capture_output=True,
                   timeout=100)
    return d / "h"


@pytest.mark.parametrize("case", ["reuse", "reset", "reset-release", "reset-evict", "growth", "count"])
def test_store(harness, case):
    r = subprocess.run([str(harness), case], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "ok\n"), r.stderr
