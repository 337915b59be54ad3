"""The pinned and device blocks kept between calls (quantr_amd/csrc/workspace.cpp) and the samplers'
use of them, over a HIP runtime of stubs that counts allocations (tests/cpp/hip_stubs.hpp) and
kernels written for the host; no GPU is used."""
import os
import subprocess

import pytest

import helpers as H

CSRC = os.path.join(H.ROOT, "quantr_amd", "csrc")


def compiled(tmp_path_factory, name, sources):
    out = str(tmp_path_factory.mktemp(name) / name)
    subprocess.run(["g++", "-O0", "-g", "-std=c++17", "-fsanitize=address,undefined", "-D__HIP_PLATFORM_AMD__",
                    "-include", "algorithm", "-I" + os.path.join(H.ROOT, "include"), "-I" + CSRC, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", name + ".cpp")] + [os.path.join(CSRC, s) for s in sources] +
                   ["-o", out, "-lpthread"], check=True)
    return out


def run(exe, check):
    r = subprocess.run([exe, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


@pytest.fixture(scope="module")
def workspace(tmp_path_factory):
    return compiled(tmp_path_factory, "workspace_check", ["workspace.cpp"])


@pytest.fixture(scope="module")
def sampler(tmp_path_factory):
    return compiled(tmp_path_factory, "sampler_check",
                    ["workspace.cpp", "sampler.cpp", "shots.cpp", "lower.cpp", "planner.cpp"])


@pytest.mark.parametrize("check", ["state_per_circuit", "call_without_a_state", "short_of_device_memory",
                                   "large_uploads"])
def test_kept_blocks(workspace, check):
    run(workspace, check)


@pytest.mark.parametrize("check", ["many_draws", "many_draws_of_programs", "halfway_blocks"])
def test_sampler(sampler, check):
    run(sampler, check)


def test_refused_threads(tmp_path):
    """parallel_for with fewer threads than it asks for (tests/cpp/threads_check.cpp)."""
    exe = str(tmp_path / "threads_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-include", "algorithm",
                    "-I" + os.path.join(H.ROOT, "include"), "-I" + CSRC, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", "threads_check.cpp"), "-o", exe, "-ldl", "-lpthread"], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
