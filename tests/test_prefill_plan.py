"""The prefill kernel's host plan on the CPU (csrc/prefill_plan.h): whatever number of splits a call runs
with, every (pair, row block, split) that holds keys is served by exactly one workgroup, and the XCDs get
equal shares of a causal prompt. (A plan whose splits were cut after its numbering was chosen sent workgroups
to row block -1; one that dealt row blocks and splits to the XCDs in turn gave some the empty splits only.)"""

import subprocess
from pathlib import Path


def test_every_row_block_and_split_once(tmp_path):
    exe = tmp_path / "prefill_plan_check"
    src = Path(__file__).with_name("prefill_plan_check.cpp")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
