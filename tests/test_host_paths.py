"""AddressSanitizer and UndefinedBehaviorSanitizer builds of the host code that production programs
go through, from a caller's program to what the kernels read (tests/cpp/host_paths.cpp)."""
import os
import subprocess

import pytest

import helpers as H

CSRC = os.path.join(H.ROOT, "quantr_amd", "csrc")
SOURCES = ["lower.cpp", "planner.cpp", "plan_image.cpp"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_paths") / "host_paths")
    subprocess.run(["g++", "-O0", "-g", "-std=c++17", "-fsanitize=address,undefined", "-D__HIP_PLATFORM_AMD__",
                    "-include", "algorithm", "-I" + os.path.join(H.ROOT, "include"), "-I" + CSRC, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", "host_paths.cpp")] + [os.path.join(CSRC, s) for s in SOURCES] +
                   ["-o", out, "-lpthread"], check=True)
    return out


@pytest.mark.parametrize("check", ["wide_customs", "plan_images", "expectation_records"])
def test_host_paths(exe, check):
    r = subprocess.run([exe, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
