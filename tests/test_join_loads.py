"""The joins' loads of pair outputs (csrc/join_device.cuh), in the emitted instructions: a loop over slots asks for eight of
them together, so that eight slots cost one trip to memory. No GPU."""
import os
import re
import subprocess

import pytest

from anemone_amd import build

CSRC = os.path.join(build.HERE, "csrc")
SLOTS_IN_FLIGHT = 8


def loops_of(body):
    """The instructions between a label and a branch back to it, a list a loop."""
    lines, at = [line.split(";")[0].strip() for line in body.splitlines()], {}
    for index, line in enumerate(lines):
        if re.fullmatch(r"\.\w+:", line):
            at[line[:-1]] = index
        branch = re.fullmatch(r"s_c?branch\w*\s+(\.\w+)", line)
        if branch and branch.group(1) in at:
            yield lines[at[branch.group(1)]:index]


@pytest.mark.parametrize("unit,kernel", [("kernel_hyper_connection.hip", "expert_join"), ("kernel_trunk_linear.hip", "expert_shared_join_1"),
                                         ("kernel_trunk_linear.hip", "expert_shared_join_4")])
def test_a_loop_over_slots_asks_for_eight_together(tmp_path_factory, unit, kernel):
    out = str(tmp_path_factory.getbasetemp() / (unit + ".s"))
    if not os.path.exists(out):
        subprocess.run(["hipcc", *build.HIP_FLAGS, "-I", build.INCLUDE, "-I", CSRC, "--cuda-device-only", "-S", os.path.join(CSRC, unit), "-o", out],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    body = open(out).read().split("\n%s:" % kernel, 1)[1].split("s_endpgm", 1)[0]
    loops = [[line for line in loop if re.match(r"global_load_(?!lds)", line)] for loop in loops_of(body)]
    loops = [loads for loads in loops if loads]  # the product's loop loads into LDS alone
    assert loops and all(len(loads) == SLOTS_IN_FLIGHT for loads in loops), loops
