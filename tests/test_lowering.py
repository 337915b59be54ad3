"""The direct lowering of programs against the general one (tests/cpp/lower_compare.cpp)."""
import os
import subprocess

import helpers as H


def test_direct_lowering_equals_the_general_one(tmp_path):
    csrc = os.path.join(H.ROOT, "quantr_amd", "csrc")
    exe = str(tmp_path / "lower_compare")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-include", "algorithm",
                    "-I" + os.path.join(H.ROOT, "include"), "-I" + csrc, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", "lower_compare.cpp"), os.path.join(csrc, "lower.cpp"),
                    os.path.join(csrc, "planner.cpp"), "-o", exe, "-lpthread"], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


def test_tile_rules(tmp_path):
    """The shapes of reverse-sweep tiles over every size, width and device (tests/cpp/plan_rules.cpp)."""
    csrc = os.path.join(H.ROOT, "quantr_amd", "csrc")
    exe = str(tmp_path / "plan_rules")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-include", "algorithm",
                    "-I" + os.path.join(H.ROOT, "include"), "-I" + csrc, "-I/opt/rocm/include",
                    os.path.join(H.ROOT, "tests", "cpp", "plan_rules.cpp"), os.path.join(csrc, "lower.cpp"),
                    os.path.join(csrc, "planner.cpp"), "-o", exe, "-lpthread"], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
