"""A Parareal without memory for the bricks' work field: where the fields themselves fit, it is
created and gives the same bits (tests/memory/limited_memory.cpp bounds the library's hipMalloc
from the host)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EULER, RK4 = 0, 1
FUSED, STAGED = 0, 1


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    lib = os.path.join(ROOT, "stencilparareal_amd")
    exe = str(tmp_path_factory.mktemp("memory") / "limited_memory")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", os.path.join(ROOT, "tests", "memory", "limited_memory.cpp"),
                        "-I", os.path.join(ROOT, "include"), "-L", lib, "-lsp_hip", "-ldl", f"-Wl,-rpath,{lib}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


def test_program_builds(program):
    assert os.path.getsize(program) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,slices,kind,path", [(64, 8, EULER, FUSED), (64, 8, RK4, FUSED), (45, 4, RK4, FUSED),
                                                (64, 8, RK4, STAGED)])
def test_parareal_without_work_field(program, n, slices, kind, path):
    r = subprocess.run([program, str(n), str(slices), str(kind), str(path)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("equal"), (r.returncode, r.stdout, r.stderr[-2000:])
