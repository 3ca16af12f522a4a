"""Two launches queued as one (csrc/joined_launches.h) leave the bytes that they leave one after the other, in a queue and in a graph
that is replayed."""
import numpy as np
import pytest

from _oracle import normals, to_bf16
from anemone_amd import workloads
from test_gpu_shared_join import amd, build, card, fresh_arena, say  # noqa: F401

pytestmark = pytest.mark.gpu


def check(amd, card, launches, ranges, first, joined):
    """launches one by one, in one list, where launches[first] and the one behind it are queued as the kernel `joined`, and as a
    graph of three replays, from the same bytes"""
    assert card.queued_as(launches[first:]) == (joined, 2)
    for index, launch in enumerate(launches):
        assert index == first or card.queued_as(launches[index:])[1] == 1
        assert card.queued_as([launch])[1] == 1
    results = []

    def run(work):
        for offset, size in ranges:
            card.upload(offset, np.full(size, 0xEE, dtype=np.uint8))
        work()
        results.append([card.download(offset, size) for offset, size in ranges])
    run(lambda: [card.run([launch]) for launch in launches])
    run(lambda: card.run(launches))
    graph = card.capture(launches)
    for _ in range(3):
        run(lambda: card.run_graph(graph))
    assert any(np.any(got != 0xEE) for got in results[0])
    for other in results[1:]:
        for index, (one, got) in enumerate(zip(results[0], other)):
            assert np.array_equal(one, got), (joined, index)


@pytest.mark.parametrize("rows,hidden,form", [(1, 128, "select"), (8, 1280, "select"), (3, 4096, "select"), (9, 256, "small"), (64, 1152, "small"),
                                              (384, 128, "small"), (1, 1152, "place"), (385, 256, "place"), (1000, 1152, "place")])
@pytest.mark.parametrize("wide_scales", [False, True])
def test_router_and_quantizer(amd, card, rows, hidden, form, wide_scales):  # noqa: F811
    say("joined launches:", form, rows, hidden, wide_scales)
    layer, _, _ = build(amd, card, hidden, 128, rows, 6, rows + hidden)
    layer.set_rows(to_bf16(normals(rows, rows * hidden)).reshape(rows, hidden))
    quantize = layer.quantize_launch()[0]
    if wide_scales:
        quantize.kernel = layer.kernels.activation_quantize_128
    outputs = [layer.ranges[name] for name in ("codes", "exponents", "operands")]
    if form == "select":
        launches, name, first = [layer.projection_launch()[0], layer.select_launch(0)[0]], "router_select_entry", 1
        extra = [(layer.jobs_offset, rows * 6 * 96), (layer.affinities_offset, rows * layer.E * 4)]
    else:
        wide = layer.wide_router()
        routed = list(wide.launches(small=form == "small"))
        launches, name = [layer.projection_launch()[0]] + routed[:2 if form == "small" else 3], "router_wide_" + form
        first = len(launches) - 1
        extra = [(wide.ranges[key].byte_offset, wide.ranges[key].byte_count) for key in ("pairs", "runs", "tiles", "jobs")]
    check(amd, card, launches + [quantize], [(r.byte_offset, r.byte_count) for r in outputs] + extra, first, name + ("_quantize_128" if wide_scales else "_quantize"))


@pytest.mark.parametrize("rows,inner", [(1, 128), (5, 640), (9, 1152), (70, 2176)])
def test_hidden_and_quantizer(amd, card, rows, inner):  # noqa: F811
    say("joined launches: hidden", rows, inner)
    many = {} if rows <= 8 else {"gate_up_slices": 1, "down_slices": 1, "wide_form": amd.LINEAR_INTERLEAVED_CHUNK_BLOCKS}
    layer, shared, _ = build(amd, card, 256, 256, rows, 1, rows, shared_inner=inner, **many)
    layer.set_rows(to_bf16(normals(rows, rows * 256)).reshape(rows, 256))
    card.run(layer.quantize_launch())
    names = [name for name in shared.ranges if name not in ("streams", "post", "comb", "pair_output")]
    check(amd, card, list(shared.launches()), [(shared.ranges[n].byte_offset, shared.ranges[n].byte_count) for n in names], 1, "trunk_hidden_quantize")


SPECIALS = np.array([0x7F80, 0xFF80, 0x7FC0, 0xFFC1, 0x7F7F, 0xFF7F, 0x0000, 0x8000, 0x0001, 0x8001, 0x7F81, 0x0080], dtype=np.uint16)


def with_specials(values, every):
    """bfloat16 words, some of them infinities, NaNs, the largest, zeros and denormals, in vectors of their own and side by side"""
    out = values.copy().reshape(-1)
    out[::every] = np.resize(SPECIALS, out[::every].size)
    out[1:40] = np.resize(SPECIALS, 39)
    return out.reshape(values.shape)


@pytest.mark.parametrize("wide_scales", [False, True])
@pytest.mark.parametrize("every", [7, 1000])
def test_router_and_quantizer_of_specials(amd, card, wide_scales, every):  # noqa: F811
    say("joined launches: specials of the rows", wide_scales, every)
    rows, hidden = 8, 1152
    layer, _, _ = build(amd, card, hidden, 128, rows, 6, 3)
    layer.set_rows(with_specials(to_bf16(normals(4, rows * hidden)).reshape(rows, hidden), every))
    quantize = layer.quantize_launch()[0]
    quantize.kernel = layer.kernels.activation_quantize_128 if wide_scales else quantize.kernel
    names = ("codes", "exponents", "operands")
    check(amd, card, [layer.projection_launch()[0], layer.select_launch(0)[0], quantize],
          [(layer.ranges[n].byte_offset, layer.ranges[n].byte_count) for n in names], 1, "router_select_entry_quantize" + ("_128" if wide_scales else ""))


@pytest.mark.parametrize("every", [7, 1000])
def test_hidden_and_quantizer_of_specials(amd, card, every):  # noqa: F811
    say("joined launches: specials of gate and up", every)
    rows, inner = 5, 1152
    layer, shared, _ = build(amd, card, 256, 256, rows, 1, rows, shared_inner=inner)
    for seed, name in enumerate(("gate_output", "up_output")):
        card.upload(shared.ranges[name].byte_offset, with_specials(to_bf16(normals(seed, rows * inner)), every + 4 * seed))
    names = [name for name in shared.ranges if name.startswith("hidden")]
    check(amd, card, list(shared.launches())[1:3], [(shared.ranges[n].byte_offset, shared.ranges[n].byte_count) for n in names], 0, "trunk_hidden_quantize")


@pytest.mark.parametrize("weights", ["e2m1", "e4m3_gfx950"])
@pytest.mark.parametrize("every", [7, 1000])
def test_gate_up_and_quantizer_of_specials(amd, card, weights, every):  # noqa: F811
    say("joined launches: specials of gate and up's rows", weights, every)
    layer, kernel = gate_up_layer(amd, card, 8, 5, 384, 2, weights)
    layer.set_rows(with_specials(to_bf16(normals(6, 8 * 1024)).reshape(8, 1024), every))
    card.run(layer.quantize_launch())
    names = ("hidden", "hidden_codes", "hidden_exponents", "hidden_operands")
    check(amd, card, list(layer.expert_launches())[:2], [(layer.ranges[n].byte_offset, layer.ranges[n].byte_count) for n in names], 0, kernel + "_joined")


def gate_up_layer(amd, card, rows, live, inner, slices, weights):  # noqa: F811
    """A layer of 8 picks whose job table holds the pairs of `live` of its rows, and the kernel of its gate and up"""
    fmt = {"e2m1": amd.WEIGHT_FORMAT_E2M1_SCALED, "e4m3": amd.WEIGHT_FORMAT_E4M3_SCALED, "e2m1_gfx950": amd.WEIGHT_FORMAT_E2M1_GFX950,
           "e4m3_gfx950": amd.WEIGHT_FORMAT_E4M3_GFX950}[weights]
    hidden, experts, picks = 1024, 64, 8
    matrix = workloads.fp4_matrix if weights.startswith("e2m1") else workloads.fp8_matrix
    trios = [[matrix(3 * e, inner, hidden), matrix(3 * e + 1, inner, hidden), matrix(3 * e + 2, hidden, inner)] for e in range(2)]
    router = to_bf16(normals(5, experts * hidden) * 0.02).reshape(experts, hidden)
    layer = amd.Fp4Layer(card, hidden, inner, experts, picks, rows, [trios[e % 2] for e in range(experts)], router_weights_bf16=router, weight_format=fmt)
    layer.gate_up_slices, layer.down_slices = slices, min(slices, 2)
    layer.set_rows(to_bf16(normals(rows, rows * hidden)).reshape(rows, hidden))
    card.upload(layer.step_offset, amd.step_block(live))
    card.run([layer.projection_launch()[0], layer.select_launch(0)[0], layer.quantize_launch()[0]])
    infix = {"e2m1": "", "e4m3": "e4m3_", "e2m1_gfx950": "gfx950_", "e4m3_gfx950": "e4m3_gfx950_"}[weights]
    return layer, "expert_gate_up_%s%d" % (infix, slices)


@pytest.mark.parametrize("rows,live,inner,slices", [(1, 1, 128, 1), (8, 8, 640, 4), (8, 5, 384, 2), (3, 2, 256, 8)])
@pytest.mark.parametrize("weights", ["e2m1", "e4m3", "e2m1_gfx950", "e4m3_gfx950"])
def test_gate_up_and_quantizer(amd, card, rows, live, inner, slices, weights):  # noqa: F811
    """Every slice instance; pairs that stand in no job, whose hidden values are quantized as they lie."""
    say("joined launches: gate and up", rows, live, inner, slices, weights)
    layer, kernel = gate_up_layer(amd, card, rows, live, inner, slices, weights)
    names = ("hidden", "hidden_codes", "hidden_exponents", "hidden_operands", "pair_output", "row_output")
    check(amd, card, list(layer.expert_launches()), [(layer.ranges[n].byte_offset, layer.ranges[n].byte_count) for n in names], 0, kernel + "_joined")


@pytest.mark.parametrize("pairs", [1, 21, 63])
@pytest.mark.parametrize("weights", ["e2m1", "e4m3_gfx950"])
def test_pairs_of_the_table_past_the_quantizer(amd, card, pairs, weights):  # noqa: F811
    """A table that names 64 pairs, launches of fewer: the quantizer writes the vectors of its grid alone. Every range has
    room for all 64."""
    say("joined launches: gate and up, pairs", pairs, weights)
    layer, kernel = gate_up_layer(amd, card, 8, 8, 384, 2, weights)
    launches = list(layer.expert_launches())[:2]
    launches[0].argument[48:52] = list(pairs.to_bytes(4, "little"))  # expert_gate_up_arguments.pair_count
    launches[1].grid[1] = pairs
    names = ("hidden", "hidden_codes", "hidden_exponents", "hidden_operands")
    check(amd, card, launches, [(layer.ranges[n].byte_offset, layer.ranges[n].byte_count) for n in names], 0, kernel + "_joined")
    assert np.all(layer.card.download(layer.ranges["hidden_codes"].byte_offset, 64 * 384)[pairs * 384:] == 0xEE)
