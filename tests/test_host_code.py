"""Host code of api.hip run on the CPU against a stand-in HIP runtime.

The programs under tests/host link the library's own api.o, scene_io.o and
image_io.o with hip_stub.cpp, where device memory is poisoned host memory, a
kernel launcher marks what its kernel would write, and any call can be made to
fail. Skips without the built objects or the HIP headers.
"""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
BUILD = ROOT / "helios_amd" / "_build"
OBJECTS = [BUILD / f"{n}.o" for n in ("api", "scene_io", "image_io")]
HEADERS = Path("/opt/rocm/include")


def run(program, tmp_path):
    cxx = shutil.which("g++")
    if cxx is None or not (HEADERS / "hip" / "hip_runtime.h").exists() or not all(o.exists() for o in OBJECTS):
        pytest.skip("needs helios_amd/_build/*.o, g++ and the HIP headers")
    exe = tmp_path / program
    src = ROOT / "tests" / "host"
    subprocess.run([cxx, "-O1", "-g", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{HEADERS}", f"-I{ROOT / 'include'}",
                    str(src / f"{program}.cpp"), str(src / "hip_stub.cpp"), *map(str, OBJECTS), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all", "-lz", "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-2000:]
    return r.stdout


def test_a_commit_after_a_failed_one_is_complete(tmp_path):
    out = run("commit_retry", tmp_path)
    assert int(out.split()[0]) > 100, out   # every call of twelve kinds of commit was made to fail


def test_captured_sequences_are_bounded_and_outlive_commits(tmp_path):
    run("sequences", tmp_path)
