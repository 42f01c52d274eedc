"""Registers of the small-row kernel's plain builds, from the compiler's report of the last build: eight waves of two chunks fit four
workgroups to a compute unit only with 64 registers a thread."""
import os
import re

import pytest

from mlx_eagle_spec_decoding_tree_amd import build


def test_eight_waves_of_two_chunks_leave_room_for_four_workgroups():
    path = os.path.join(build.HERE, "build", "smallpass.hip.o.log")
    if not os.path.exists(path):
        pytest.skip("no report of a build here")
    with open(path, errors="replace") as f:
        text = f.read()
    regs = dict(re.findall(r"Function Name: (\S+).*?\bVGPRs: (\d+)", text, re.S))
    for passes in (1, 2):                         # up to 4, up to 8 rows of x
        name = next(n for n in regs if f"qmm_small_kernelILi8ELi2ELi{passes}ELi0ELb0ELb0E" in n)
        assert int(regs[name]) <= 64, (name, regs[name])
