"""Host programs over the library's C++ sources, built with the ROCm clang
under AddressSanitizer and UndefinedBehaviorSanitizer and run on the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANGXX = "/opt/rocm/lib/llvm/bin/clang++"
SAN = ["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-fno-omit-frame-pointer", "-g", "-O1"]
FLAGS = ["-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-pthread"]

pytestmark = pytest.mark.skipif(not os.path.exists(CLANGXX), reason="no ROCm clang")


def run(tmp_path, name, sources=(), args=()):
    exe = str(tmp_path / name)
    src = [os.path.join(ROOT, "tests", "native", name + ".cpp")]
    src += [os.path.join(ROOT, "kaust-hierarchical-matrices_amd", "csrc", s) for s in sources]
    b = subprocess.run([CLANGXX, *SAN, *FLAGS, *src, "-o", exe], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    # leak check off: what the program holds while it ends is the subject of one check
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    assert "Sanitizer" not in r.stderr and "runtime error" not in r.stderr
    return r.stdout


def test_a_failed_growth_is_not_recorded(tmp_path):
    assert "buffer check ok" in run(tmp_path, "buffer_check")


@pytest.mark.parametrize("what", ["hold", "share", "wait", "capture", "exit"])
def test_held_device_memory(tmp_path, what):
    assert f"pool check {what} ok" in run(tmp_path, "pool_check", ["pool.cpp"], [what])
