"""CPU test of the length classes, sort keys and LDS layouts that the plan of the
batched form relies on (gbsw_kernel_args.hpp), over every accepted length."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_classes_keys_and_layouts(tmp_path):
    exe = str(tmp_path / "classes_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", os.path.join(HERE, "host", "classes_check.cpp"), "-o", exe],
                   check=True)
    assert subprocess.run([exe], capture_output=True, text=True).stdout.strip() == "ok"
