"""The kernel of batches: which calls it takes, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_plan(tmp_path):
    exe = tmp_path / "test_panel_plan"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "cudaintro_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_panel_plan.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and "panel plan OK" in out.stdout, out.stdout
