"""csrc/row_slot.hpp on the host: over grids below, at and above one and two workgroups per compute
unit the acceptance kernel's workgroups take every logits row once, and the two workgroups that
share a compute unit take rows of one sequence as far as the sequences' rows form whole pairs."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_rows_taken_once_and_paired(tmp_path):
    exe = str(tmp_path / "row_slot")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "row_slot.cpp")], check=True)
    n, wrong, split = map(int, subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120).stdout.split())
    assert n == 5 * 20 * 150 and wrong == 0 and split == 0, (n, wrong, split)
