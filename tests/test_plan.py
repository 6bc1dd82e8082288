"""CPU test of the batched form's plan (gbsw_exec.cpp, built with stand-ins for the
kernels): whatever the lengths, every set of pairs of every launch has a geometry that
its kernel holds, and the launches cover every pair once."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_every_set_has_a_geometry(tmp_path):
    exe = str(tmp_path / "plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    os.path.join(HERE, "host", "plan_check.cpp"), "-o", exe, "-L" + os.path.join(ROCM, "lib"),
                    "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-lamdhip64"], check=True)
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "ok"
