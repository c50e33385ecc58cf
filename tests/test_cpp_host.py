"""The C++ host mirror (include/deltanet.hpp) through its own test binary,
tests/cpp/test_host.cpp: argument checks on the CPU, values against the
oracle on the GPU; and the library's launches, recorded on the CPU in place of
the HIP runtime (tests/cpp/test_launches.cpp). The binaries are built by
__graft_entry__.build() (make -C tests/cpp)."""

import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
BUILD = ROOT / "tests" / "cpp" / "_build"


def run_binary(name, *mode, timeout):
    if not (BUILD / name).exists():
        # Host code only, seconds: build it against the built libraries.
        subprocess.run(["make", "-C", str(ROOT / "tests" / "cpp")], check=True,
                       capture_output=True, timeout=300)
    r = subprocess.run([str(BUILD / name), *mode], capture_output=True, text=True, timeout=timeout)
    print(r.stdout)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    assert "all passed" in r.stdout


def test_cpp_host_argument_checks():
    run_binary("test_host", "--host-only", timeout=60)


def test_library_launches():
    run_binary("test_launches", timeout=60)


@pytest.mark.gpu
def test_cpp_host_values_on_gpu():
    run_binary("test_host", "--gpu", timeout=120)
