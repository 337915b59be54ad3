"""The pinned and device blocks kept between calls (quantr_amd/csrc/workspace.cpp), over a HIP
runtime of stubs that counts allocations (tests/cpp/workspace_check.cpp); no GPU is used."""
import os
import subprocess

import pytest

import helpers as H


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    csrc = os.path.join(H.ROOT, "quantr_amd", "csrc")
    out = str(tmp_path_factory.mktemp("workspace") / "workspace_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(H.ROOT, "include"), "-I" + csrc, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", "workspace_check.cpp"), os.path.join(csrc, "workspace.cpp"),
                    "-o", out], check=True)
    return out


@pytest.mark.parametrize("check", ["state_per_circuit", "call_without_a_state", "short_of_device_memory"])
def test_kept_blocks(exe, check):
    r = subprocess.run([exe, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
