"""The fp32 tiles on the bf16 matrix instructions: planner on the host, generated code."""
import os
import re
import shutil
import subprocess

import pytest

from test_build_resources import FLAGS, HIPCC, spill_counts

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cudaintro_amd", "csrc")


def test_plan(tmp_path):
    exe = tmp_path / "test_f32_split_plan"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(ROOT, "tests", "cpp", "test_f32_split_plan.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and "f32 split plan OK" in out.stdout, out.stdout


@pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")
@pytest.mark.parametrize("rows", [64, 96, 128])
def test_main_loop_does_not_spill(tmp_path, rows):
    """The running sums fill the accumulator registers: the main loop must neither move them nor go to
    scratch memory."""
    asm = tmp_path / "split.s"
    subprocess.run([HIPCC, *FLAGS, f"-DCIG_SPLIT_ROWS={rows}", os.path.join(CSRC, "f32_split_rows.hip"), "-o", str(asm)],
                   check=True, stderr=subprocess.DEVNULL)
    text = asm.read_text()
    spills = spill_counts(text)
    assert len(spills) == 3 and not any(spills.values()), spills
    loops = [b for b in re.split(r"\n(?=\.LBB)", text) if b.count("v_mfma_f32_32x32x16_bf16") >= rows]
    assert len(loops) == 3
    for body in loops:
        body = body[:body.rindex("v_mfma_f32_32x32x16_bf16")]
        assert not re.search(r"scratch_|v_accvgpr|buffer_", body)
