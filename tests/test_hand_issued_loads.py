"""Loads that csrc/ issues by hand into registers (assembly whose result is a vector register): the compiler takes such a
register for filled where the load is asked for, so one that it saved or copied before the wait would be taken before its
bytes land. The build refuses these kernels where they spill (anemone_amd/build.py), and the emitted instructions of
router_projection_split's LDS reads are read here. No GPU."""
import os
import re
import subprocess

import pytest

from anemone_amd import build

CSRC = os.path.join(build.HERE, "csrc")
ASSEMBLY = re.compile(r'asm volatile\(\s*((?:"[^"]*"\s*)+):\s*((?:"[^"]*"\s*\([^)]*\)\s*,?\s*)*)', re.S)


def source(name):
    return open(os.path.join(CSRC, name)).read()


def issues_register_loads(text):
    return any(re.search(r"\b(global_load|buffer_load|ds_read)(?!_lds)", instructions) and not re.search(r"_lds", instructions) and '"' in results
               for instructions, results in ASSEMBLY.findall(text))


def headers_of(name, seen=None):
    seen = set() if seen is None else seen
    for header in re.findall(r'#include "([^"]+\.cuh)"', source(name)):
        if header not in seen:
            seen.add(header)
            headers_of(header, seen)
    return seen


def test_every_unit_of_such_loads_is_under_the_build_s_guard():
    own = {name for name in os.listdir(CSRC) if name.endswith((".hip", ".cuh")) and issues_register_loads(source(name))}
    assert "native_device.cuh" in own and "kernel_router.hip" in own
    units = {name for name in build.HIP_SOURCES if own & ({name} | headers_of(name))}
    assert units == set(build.NO_SPILL_SOURCES)
    for unit, kernels in build.NO_SPILL_SOURCES.items():
        assert all(re.search(r"\b%s\(" % kernel, source(unit)) for kernel in kernels or [])


def test_the_guard_takes_the_named_kernels_of_a_unit():
    remark = "/x/kernel_router.hip:1:1: remark: %s [-Rpass-analysis=kernel-resource-usage]"

    def output(**spills):
        return "\n".join(remark % line for name, count in spills.items() for line in ("Function Name: " + name, "    VGPRs Spill: %d" % count))
    assert build.refused_spills("kernel_router.hip", output(router_projection_tiles=2, router_projection_split=0)) == []
    assert build.refused_spills("kernel_router.hip", output(router_projection_tiles=2, router_projection_split=1)) == [("router_projection_split", 1)]
    assert build.refused_spills("kernel_native_linear.hip", output(native_expert_down_1=3)) == [("native_expert_down_1", 3)]
    for unit, text in (("kernel_router.hip", output(router_projection_tiles=0)), ("kernel_native_linear.hip", "")):  # no remarks: nothing was checked
        with pytest.raises(RuntimeError):
            build.refused_spills(unit, text)


def test_the_split_projection_s_reads_land_before_anything_else_touches_them(tmp_path):
    """Between a ds_read_u16_d16_hi and the s_waitcnt lgkmcnt(0) behind it no other instruction names its register, and
    control neither leaves nor enters."""
    out = str(tmp_path / "router.s")
    subprocess.run(["hipcc", *build.HIP_FLAGS, "-I", build.INCLUDE, "-I", CSRC, "--cuda-device-only", "-S", os.path.join(CSRC, "kernel_router.hip"), "-o", out],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    body = open(out).read().split("\nrouter_projection_split:", 1)[1].split("s_endpgm", 1)[0]
    pending, reads, waits = set(), 0, 0
    for line in body.splitlines():
        line = line.split(";")[0].strip()
        if not line or line.startswith("."):
            assert not (line.endswith(":") and pending), "a label between the reads and their wait: %s" % line
            continue
        words = line.replace(",", " ").split()
        named = {int(n) for n in re.findall(r"\bv(\d+)\b", line)}
        for first, last in re.findall(r"\bv\[(\d+):(\d+)\]", line):
            named |= set(range(int(first), int(last) + 1))
        if words[0] == "ds_read_u16_d16_hi":
            register = int(words[1][1:])
            assert not (named - {register}) & pending and register not in pending, line
            pending.add(register)
            reads += 1
        elif words[0] == "s_waitcnt" and "lgkmcnt(0)" in line:
            waits += 1 if pending else 0
            pending.clear()
        else:
            assert not words[0].startswith(("s_cbranch", "s_branch", "s_setpc", "s_endpgm")) or not pending, "control leaves: %s" % line
            assert not named & pending, line
    assert not pending and reads >= 24 and waits >= 3, (reads, waits)
