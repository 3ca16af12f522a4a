"""Which launches of the shared expert's interleaved product the backend queues in smaller blocks (csrc/trunk_deep.cpp): the rule over the
launch's record alone, on the CPU."""
import ctypes as C
import struct

import pytest

import anemone_amd as amd
from test_joined_launches import launch

LDS = 160 * 1024
NONE = 3


class Deep(C.Structure):
    _fields_ = [("grid", C.c_uint32 * 2), ("shared_bytes", C.c_uint32)]


def rule(one, most_shared_bytes=LDS):
    lib = amd.library()
    lib.trunk_deep_instance.restype = C.c_uint32
    lib.trunk_deep_instance.argtypes = [C.c_void_p, C.c_uint32, C.c_void_p]
    out = Deep()
    instance = lib.trunk_deep_instance(C.byref(one), most_shared_bytes, C.byref(out))
    return NONE if instance == NONE else (16 << instance, list(out.grid), out.shared_bytes)


def product(rows, inputs, *outputs, **changes):
    outputs = (list(outputs) + [0])[:2]
    one = launch((sum((o + 127) // 128 for o in outputs), (rows + 63) // 64, 1), 256, struct.pack("<7Q4I", *range(0, 7 << 20, 1 << 20), *outputs, inputs, rows))
    one.dynamic_shared_byte_count = 51712
    for name, value in changes.items():
        if name == "block" or name == "grid":
            getattr(one, name)[value[0]] = value[1]
        else:
            setattr(one, name, value)
    return one


@pytest.mark.parametrize("rows,of,groups,window", [(9, 16, 1, 54528), (128, 16, 8, 54528), (129, 32, 5, 66816), (256, 32, 8, 66816), (257, 64, 5, 74752),
                                                   (512, 64, 8, 74752)])
def test_blocks_of_the_fewest_rows_that_all_have_a_place(rows, of, groups, window):
    """64 blocks of 64 outputs: at most 512 blocks."""
    assert rule(product(rows, 4096, 2048, 2048)) == (of, [64, groups], window)
    assert rule(product(rows, 4096, 4096)) == (of, [64, groups], window)
    assert rule(product(513, 4096, 4096)) == NONE
    assert rule(product(rows, 4096, 4096), window) == (of, [64, groups], window)
    assert rule(product(rows, 4096, 4096), window - 1) == NONE  # the card grants a block less


@pytest.mark.parametrize("inputs", [4096, 7680, 7808, 8192, 16384])
def test_places_are_those_of_the_window(inputs):
    """A CU's 160 KB hold two windows of 64 rows up to 7680 inputs, above them one: 257 to 512 blocks would be two rounds. Two of 32
    and of 16 rows at any inputs."""
    assert rule(product(512, inputs, 2048)) == (32, [32, 16], 62720 + (inputs + 511) // 512 * 512)
    for rows, blocks in ((513, 32), (1024, 32), (1024, 17)):
        whole = (64, [blocks, (rows + 63) // 64], 66560 + (inputs + 511) // 512 * 1024)
        assert rule(product(rows, inputs, 64 * blocks)) == (whole if inputs <= 7680 else NONE)


def test_ragged_products():
    assert rule(product(9, 128, 160, 32)) == (16, [4, 1], 5 * 10496 + 256)
    assert rule(product(33, 640, 1056)) == (16, [17, 3], 5 * 10496 + 512)
    assert rule(product(9, 16384, 160)) == (16, [3, 1], 5 * 10496 + 32 * 256)
    assert rule(product(9, 16512, 160)) == NONE
    assert rule(product(9, 192, 160)) == NONE and rule(product(9, 0, 160)) == NONE


def test_launches_that_are_not_the_whole_product():
    for change in ({"grid": (0, 31)}, {"grid": (0, 33)}, {"grid": (1, 1)}, {"grid": (1, 3)}, {"grid": (2, 2)}, {"block": (0, 128)}, {"block": (1, 2)},
                   {"dynamic_shared_byte_count": 51711}, {"dynamic_shared_byte_count": 60000}):
        assert rule(product(100, 4096, 4096)) != NONE and rule(product(100, 4096, 4096, **change)) == NONE, change
    wraps = product(0xFFFFFFFF, 128, 0xFFFFFFFF)  # the products of its sizes are formed in 64 bits
    assert rule(wraps) == NONE
