"""Which pairs of launches the backend queues as one (csrc/joined_launches.cpp): the rule over records alone, on the CPU. A pair whose
quantizer touches what the other launch writes, or writes what it reads, stays two launches."""
import ctypes as C
import struct

import pytest

import anemone_amd as amd

ROWS, E, P, H = 40, 64, 6, 256
STEP = 1 << 20  # every range begins on a place of its own, further apart than any range is long


class Joined(C.Structure):
    _fields_ = [("grid", C.c_uint32 * 2), ("block", C.c_uint32), ("numbers", C.c_uint32 * 3)]


def rule(name, first, second, arena=1 << 34, quantize="activation_quantize_entry"):
    lib = amd.library()
    lib.joined_launch_of.restype = C.c_bool
    lib.joined_launch_of.argtypes = [C.c_char_p, C.c_char_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p]
    out = Joined()
    joins = lib.joined_launch_of(name.encode(), quantize.encode(), C.byref(first), C.byref(second), arena, C.byref(out))
    return (list(out.grid), out.block, list(out.numbers)) if joins else None


def launch(grid, block, record):
    one = amd.launches_of(1)[0]
    for d in range(3):
        one.grid[d], one.block[d] = grid[d], (block, 1, 1)[d]
    one.argument_byte_count = len(record)
    C.memmove(one.argument, record, len(record))
    return one


def quantizer(values=STEP, codes=2 * STEP, exponents=3 * STEP, operands=4 * STEP, width=H, rows=ROWS, grid=None):
    return launch(grid or ((width + 1023) // 1024, rows, 1), 256, struct.pack("<4Q2I", values, codes, exponents, operands, width, 0))


# name: (offset of the member in the record, its bytes, written or not)
SELECT = {"step": (0, 16, False), "scores": (1, ROWS * E * 4, False), "bias": (2, E * 4, False), "expert_offsets": (3, E * 24, False),
          "affinities": (4, ROWS * E * 4, True), "jobs": (5, ROWS * P * 96, True)}
TILES, JOBS = (ROWS * P + 63) // 64 + E, min(ROWS * P, (ROWS * P + 7 * E) // 8)
WIDE = {"step": (0, 16, False), "expert_offsets": (3, E * 24, False), "picks": (5, ROWS * P * 8, False), "counts": (6, E * 4, False),
        "pairs": (7, ROWS * P * 8, True), "runs": (8, E * 8, True), "tiles": (9, TILES * 32, True), "jobs": (10, JOBS * 96, True)}


def router(name, pick_count=P, **places):
    wide = name != "router_select_entry"
    members = [(16 + i) * STEP for i in range(14 if wide else 9)]
    for member, place in places.items():
        members[(WIDE if wide else SELECT)[member][0]] = place
    return launch((1, 1, 1), 512, struct.pack("<%dQ5If" % len(members), *members, ROWS, 0, E, pick_count, 0, 1.5))


@pytest.mark.parametrize("name", ["router_select_entry", "router_wide_small", "router_wide_place"])
def test_router_and_quantizer(name):
    assert rule(name, router(name), quantizer()) == ([1 + ROWS // 2, 1], 512, [1, 1, ROWS])
    assert rule(name, router(name), quantizer(width=1280, rows=3)) == ([4, 1], 512, [1, 2, 3])  # two blocks a vector: the last of six alone
    for member, (_, size, written) in (SELECT if name == "router_select_entry" else WIDE).items():
        for at, length, is_written in ((STEP, 2 * ROWS * H, False), (2 * STEP, ROWS * H, True), (3 * STEP, ROWS * H // 32, True), (4 * STEP, 2 * ROWS * H, True)):
            meets = written or is_written
            for place, overlaps in ((at + length, False), (at + length - 1, True), (at - size, False), (at - size + 1, True)):
                joined = rule(name, router(name, **{member: place}), quantizer())
                assert (joined is None) == (overlaps and meets), (name, member, at, place)


def test_launches_that_are_not_whole():
    name = "router_wide_small"
    first = router(name)
    assert rule(name, first, quantizer(width=1028, grid=(1, ROWS, 1))) is None  # four values no thread takes
    assert rule(name, first, quantizer(grid=(1, ROWS, 2))) is None
    assert rule(name, first, quantizer(width=0, grid=(1, ROWS, 1))) is None
    assert rule(name, first, quantizer(), arena=ROWS * H - 1) is None
    wrong = quantizer()
    wrong.block[0] = 128
    assert rule(name, first, wrong) is None
    wrong = router(name)
    wrong.dynamic_shared_byte_count = 16
    assert rule(name, wrong, quantizer()) is None
    many = quantizer(width=64, rows=0xFFFFFFFF)  # more blocks than a grid of 512 threads has
    assert rule(name, first, many, arena=1 << 62) is None


def hidden(gate=8 * STEP, up=9 * STEP, out=STEP, width=H, rows=ROWS):
    return launch(((width + 2047) // 2048, rows, 1), 256, struct.pack("<3QIf", gate, up, out, width, 10.0))


def test_hidden_and_quantizer():
    name = "trunk_hidden_entry"
    assert rule(name, hidden(), quantizer()) == ([1, ROWS], 256, [0, 0, 0])
    assert rule(name, hidden(width=2112), quantizer(width=2112)) == ([3, ROWS], 256, [0, 0, 0])
    assert rule(name, hidden(out=5 * STEP), quantizer()) is None  # other values
    assert rule(name, hidden(rows=ROWS - 1), quantizer()) is None
    assert rule(name, hidden(width=2 * H), quantizer()) is None
    assert rule(name, hidden(width=264), quantizer(width=264)) is None  # no whole blocks of 32
    size = 2 * ROWS * H
    for member in ("gate", "up"):
        assert rule(name, hidden(**{member: STEP}), quantizer()) is None  # in place
        for at, length in ((STEP, size), (2 * STEP, ROWS * H), (3 * STEP, ROWS * H // 32), (4 * STEP, size)):
            for place, overlaps in ((at + length, False), (at + length - 1, True), (at - size, False), (at - size + 1, True)):
                assert (rule(name, hidden(**{member: place}), quantizer()) is None) == overlaps
    for member in ("codes", "exponents", "operands"):
        assert rule(name, hidden(), quantizer(**{member: STEP + size - 1})) is None


def whole_gate_up(jobs=8 * STEP, codes=9 * STEP, exponents=10 * STEP, out=STEP, width=H, inputs=384, pairs=ROWS, picks=4, job_count=30, strip=64, grid_x=None, block=256):
    record = struct.pack("<5Q4IfI", jobs, codes, exponents, 11 * STEP, out, width, inputs, pairs, picks, 10.0, 0)
    return launch((grid_x or (width + strip - 1) // strip, job_count, 1), block, record)


@pytest.mark.parametrize("name,strip", [("expert_gate_up_4", 64), ("expert_gate_up_e4m3_gfx950_4", 32)])
def test_gate_up_and_quantizer(name, strip):
    def gate_up(**changes):
        return whole_gate_up(strip=strip, **changes)
    assert rule(name, gate_up(), quantizer()) == ([H // strip, 31], 256, [30, 0, 0])
    assert rule(name, gate_up(pairs=64), quantizer(rows=64)) is not None
    assert rule(name, gate_up(pairs=65), quantizer(rows=65)) is None  # more pairs than one launch takes
    assert rule(name, gate_up(pairs=ROWS - 1), quantizer()) is None
    assert rule(name, gate_up(out=5 * STEP), quantizer()) is None
    assert rule(name, gate_up(width=2 * H), quantizer()) is None
    assert rule(name, gate_up(width=272), quantizer(width=272)) is None  # no whole blocks of 32
    rows = (ROWS + 3) // 4
    for member, size in (("jobs", 30 * 96), ("codes", rows * 384), ("exponents", rows * 12)):
        for at, length in ((STEP, 2 * ROWS * H), (2 * STEP, ROWS * H), (3 * STEP, ROWS * H // 32), (4 * STEP, 2 * ROWS * H)):
            for place, overlaps in ((at + length, False), (at + length - 1, True), (at - size, False), (at - size + 1, True)):
                assert (rule(name, gate_up(**{member: place}), quantizer()) is None) == overlaps, (member, at, place)
    for member in ("codes", "exponents", "operands"):
        assert rule(name, gate_up(), quantizer(**{member: STEP + 2 * ROWS * H - 1})) is None


@pytest.mark.parametrize("infix,strip", [("", 64), ("gfx950_", 64), ("e4m3_", 32), ("e4m3_gfx950_", 32)])
@pytest.mark.parametrize("slices", [1, 2, 4, 8])
def test_gate_up_of_fewer_blocks_than_strips(infix, strip, slices):
    """The quantizer's launch covers whole vectors, a joined block its own strip alone."""
    name = "expert_gate_up_%s%d" % (infix, slices)
    for width in (64, H, 11 * 64):
        strips = width // strip

        def joins(**changes):
            launch = whole_gate_up(width=width, strip=strip, **{"block": 64 * slices, **changes})
            return rule(name, launch, quantizer(width=width)) is not None
        assert joins()
        assert not any(joins(grid_x=grid) for grid in (1, strips - 1, strips + 1) if grid not in (0, strips))
        assert not any(joins(block=block) for block in (32 * slices, 128 * slices))


@pytest.mark.parametrize("width", [32, 96, 1120, 2080, 264])
def test_widths_the_quantizer_has_no_order_for(width):
    """Its words of codes lie in groups of 64 values (one float32 scale: 128): a vector of another width is written past its
    end, so that the ranges compared are not what is written."""
    whole = (width + 63) // 64 * 64
    for name in ("router_select_entry", "router_wide_small", "router_wide_place"):
        assert rule(name, router(name), quantizer(width=width)) is None
        assert rule(name, router(name), quantizer(width=whole)) is not None
        wide = "activation_quantize_128_entry"
        assert rule(name, router(name), quantizer(width=whole), quantize=wide) is None or whole % 128 == 0
        assert rule(name, router(name), quantizer(width=2 * whole), quantize=wide) is not None
    assert rule("trunk_hidden_entry", hidden(width=width), quantizer(width=width)) is None
    for name, strip in (("expert_gate_up_4", 64), ("expert_gate_up_e4m3_4", 32)):
        assert rule(name, whole_gate_up(width=width, strip=strip), quantizer(width=width)) is None


def test_every_joined_kernel_is_registered():
    """Under the names of two kernels of the library: a pair that is missing, or misnamed, would run as two launches without a word."""
    lib, kernels, joined = amd.library(), set(), []
    f, g, b = C.c_char_p(), C.c_char_p(), C.c_uint32()
    for i in range(lib.backend_hip_kernel_table_count()):
        assert lib.backend_hip_kernel_table_entry(i, C.byref(f), C.byref(g), C.byref(b)) == 0
        kernels.add((f.value.decode(), g.value.decode()))
    files, functions = (C.c_char_p * 2)(), (C.c_char_p * 2)()
    for i in range(lib.backend_hip_joined_table_count()):
        assert lib.backend_hip_joined_table_entry(i, files, functions, C.byref(g)) == 0
        launches = [(files[k].decode(), functions[k].decode()) for k in range(2)]
        assert all(launch in kernels for launch in launches), launches
        joined.append((launches[0][1], launches[1][1], g.value.decode()))
    assert lib.backend_hip_joined_table_entry(len(joined), files, functions, C.byref(g)) != 0
    want = [(name, "activation_quantize%s_entry" % scales, "%s_quantize%s" % (name, scales))
            for name in ("router_select_entry", "router_wide_small", "router_wide_place") for scales in ("", "_128")]
    want += [("trunk_hidden_entry", "activation_quantize_entry", "trunk_hidden_quantize")]
    want += [(name, "activation_quantize_entry", name + "_joined")
             for infix in ("", "e4m3_", "gfx950_", "e4m3_gfx950_") for slices in (1, 2, 4, 8) for name in ["expert_gate_up_%s%d" % (infix, slices)]]
    assert sorted(joined) == sorted(want)


@pytest.mark.parametrize("quantize,picks,most", [("", 1, 40), ("", 8, 40), ("_128", 1, 16), ("_128", 3, 16), ("_128", 4, 24), ("_128", 0, 24)])
def test_router_and_quantizer_of_many_values(quantize, picks, most):
    """Many values: beside the place launch's LDS the quantizer takes longer than by itself and a launch more."""
    def joins(width, rows):
        places = {name: (i + 1) << 33 for i, name in enumerate(("values", "codes", "exponents", "operands"))}
        second = quantizer(width=width, rows=rows, **places)
        return rule(name, router(name, pick_count=picks), second, arena=1 << 40, quantize="activation_quantize%s_entry" % quantize) is not None
    for name in ("router_select_entry", "router_wide_small", "router_wide_place"):
        for width in (1024, 4096):
            rows = (most << 20) // width
            assert joins(width, rows) and not joins(width, rows + 1)


@pytest.mark.parametrize("name,strip,inputs,most", [
    ("expert_gate_up_4", 64, 3968, 1024), ("expert_gate_up_4", 64, 4096, 2048), ("expert_gate_up_gfx950_8", 64, 8192, 2048), ("expert_gate_up_8", 64, 4096, 1024),
    ("expert_gate_up_1", 64, 1024, 2048), ("expert_gate_up_e4m3_4", 32, 3968, 1536), ("expert_gate_up_e4m3_4", 32, 4096, 4096),
    ("expert_gate_up_e4m3_1", 32, 4096, 1536), ("expert_gate_up_e4m3_gfx950_4", 32, 4096, 1536)])
def test_gate_up_of_many_blocks(name, strip, inputs, most):
    """Many short blocks: quantizing behind each costs more than the launch."""
    slices = int(name[-1])
    for pairs in (32, 64):
        for width, joins in ((most // pairs * strip, True), (most // pairs * strip + 64, False)):
            places = dict(out=STEP, width=width, inputs=inputs, pairs=pairs, picks=8, job_count=pairs, strip=strip, block=64 * slices)
            assert (rule(name, whole_gate_up(**places), quantizer(width=width, rows=pairs)) is not None) == joins, (pairs, width)
