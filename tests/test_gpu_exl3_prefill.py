"""GPU parity of the prefill form of the EXL3 routed experts (pairs sorted by expert, grouped GEMM with the trellis
decode fused into the weight tile loads) against the CPU oracle's double-precision layer, through the C ABI. The bound
is the fused decode's: 4e-3 of the output's rms (the reference holds its tensor-core forms to 2e-3 rms of its chain,
tests/exl3_tc_card_test.c:40-41, and its probe to 2e-3 of rms against double,
tools/measure/trellis_expert_probe.cu:73)."""
import ctypes as C
import sys

import numpy as np
import pytest

from _oracle import f32p, normals, orc, ptr, splitmix_words, to_bf16, exl3_matrix, u8p, u16p, u32p

pytestmark = pytest.mark.gpu


def say(*words):
    print(*words, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def amd():
    import anemone_amd
    return anemone_amd


@pytest.fixture(scope="module")
def card(amd):
    card = amd.Card(2 << 30)
    yield card
    card.close()


@pytest.fixture(autouse=True)
def fresh_arena(card):
    card.cursor = 256
    yield


def build_layer(amd, card, hidden, inner, experts_n, picks, rows, seed, width_choices):
    draws = splitmix_words(seed, experts_n * 3) % np.uint64(len(width_choices))
    widths = np.array(width_choices, dtype=np.uint32)[draws.astype(np.int64)].reshape(experts_n, 3)
    matrices = [[exl3_matrix(seed * 1000 + 3 * e + 0, hidden, inner, int(widths[e, 0])),
                 exl3_matrix(seed * 1000 + 3 * e + 1, hidden, inner, int(widths[e, 1])),
                 exl3_matrix(seed * 1000 + 3 * e + 2, inner, hidden, int(widths[e, 2]))] for e in range(experts_n)]
    router = to_bf16(normals(seed + 5, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    layer = amd.Exl3Layer(card, hidden, inner, experts_n, picks, rows, matrices, widths, router_weights_bf16=router,
                          affinity_kind=1, limit=10.0)
    return layer, matrices, widths


def oracle_layer(layer, x, experts, weights, matrices, widths, threads=8):
    rows, H, I, P, E = layer.rows, layer.H, layer.I, layer.P, layer.E
    pointers = (C.c_void_p * (E * 3))(*[m.ctypes.data for trio in matrices for m in trio])
    out = np.zeros((rows, H), dtype=np.float32)
    widths8 = np.ascontiguousarray(widths.astype(np.uint8))
    orc.orc_exl3_moe_layer(ptr(x, u16p), rows, H, I, P, ptr(experts, u32p), ptr(weights, f32p), E, pointers, ptr(widths8, u8p),
                           layer.limit, ptr(out, f32p), None, None, threads)
    return out


@pytest.mark.parametrize("hidden,inner,experts_n,picks,rows,width_choices,skew", [
    (512, 256, 64, 4, 300, [2, 3, 4], 1.5),   # a few experts with more than one chunk of pairs, others ragged
    (512, 384, 64, 8, 70, [3], 0.0),          # one width; 384 outputs: a GEMM block whose last wavefronts lie past the matrix
    (256, 128, 64, 2, 9, [40, 4], 0.0),       # K = 2.5 among the widths; chunks of one or two pairs, experts without any
])
def test_prefill_layer_against_oracle(amd, card, hidden, inner, experts_n, picks, rows, width_choices, skew):
    say("prefill", hidden, inner, experts_n, picks, rows, width_choices, skew)
    layer, matrices, widths = build_layer(amd, card, hidden, inner, experts_n, picks, rows, 21, width_choices)
    x = to_bf16(normals(31, rows * hidden)).reshape(rows, hidden)
    layer.set_rows(x, rows)
    bias = (-skew * np.log(1.0 + np.arange(experts_n))).astype(np.float32)
    card.upload(layer.bias_offset, bias)
    card.run(layer.projection_launch())
    wide = layer.wide_router()
    card.run(wide.launches()[0:1])  # the picks of every row
    picks_table = wide.read("picks", np.dtype([("expert", "<u4"), ("route_weight", "<f4")])).reshape(rows, picks)
    experts = np.ascontiguousarray(picks_table["expert"])
    weights = np.ascontiguousarray(picks_table["route_weight"])
    launches = layer.tcp_launches(wide.ranges["picks"].byte_offset)
    assert len(launches) == 7
    # poison the sort's tables and the output: everything read must have been written by the call
    layout = layer.tcp_layout
    card.upload(layer.tcp_workspace_offset, np.full(layout["operands"], 0xA5, dtype=np.uint8))
    card.upload(layer.out_offset, np.full(rows * hidden * 4, 0xFF, dtype=np.uint8))
    card.run(launches)
    # the route: sorted by expert, rows ascending; place_of its inverse; chunks of at most EXL3_TCP_CHUNK_PAIRS of one expert
    pairs = rows * picks
    sorted_pairs = card.download(layer.tcp_workspace_offset + layout["sorted"], pairs * 4, np.uint32)
    place_of = card.download(layer.tcp_workspace_offset + layout["place_of"], pairs * 4, np.uint32)
    want_sorted = np.argsort(experts.reshape(-1), kind="stable").astype(np.uint32)
    assert np.array_equal(sorted_pairs, want_sorted)
    assert np.array_equal(place_of[sorted_pairs], np.arange(pairs, dtype=np.uint32))
    used = int(card.download(layer.tcp_workspace_offset + layout["header"], 4, np.uint32)[0])
    chunks = card.download(layer.tcp_workspace_offset + layout["chunks"], layout["chunk_capacity"] * 16, np.uint32).reshape(-1, 4)
    counts = np.bincount(experts.reshape(-1), minlength=experts_n)
    most = amd.EXL3_TCP_CHUNK_PAIRS
    assert used == int(((counts + most - 1) // most).sum()) and not chunks[used:].any()
    assert int(chunks[:used, 2].sum()) == pairs and chunks[:used, 2].max() <= most
    assert np.array_equal(chunks[:used, 1], np.concatenate([[0], np.cumsum(chunks[:used, 2])[:-1]]))
    say("  chunks %d, the longest run %d pairs" % (used, counts.max()))
    # the operands are bit-defined: fp16(H128(bf16 x, fp16 suh) / sqrt(128)), by place, gate then up. The down pass has
    # taken the first array since; run the route and the operands once more and read both
    card.run(launches[0:3])
    operands = card.download(layer.tcp_workspace_offset + layout["operands"], 2 * pairs * hidden * 2, np.uint16).reshape(2, pairs, hidden)
    for place in sorted(set(list(range(0, pairs, max(1, pairs // 40))) + [pairs - 1])):
        pair = int(sorted_pairs[place])
        e = int(experts.reshape(-1)[pair])
        for proj in range(2):
            cb = int(orc.orc_exl3_code_bytes(hidden, inner, int(widths[e, proj])))
            suh = np.ascontiguousarray(matrices[e][proj][cb:cb + 2 * hidden]).view(np.uint16)
            expect = np.zeros(hidden, dtype=np.uint16)
            orc.orc_exl3_operand(ptr(x[pair // picks], u16p), ptr(suh, u16p), hidden, ptr(expect, u16p))
            assert np.array_equal(operands[proj, place], expect), ("operands are bit-defined", place, proj)
    card.run(launches)
    got = layer.output()
    want = oracle_layer(layer, x, experts, weights, matrices, widths)
    scale = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    error = float(np.max(np.abs(got - want))) / scale
    say("  max error %.2e of the output's rms" % error)
    assert error <= 4e-3


@pytest.mark.parametrize("picks", [1, 3, 5, 6, 7])
def test_prefill_slots_of_a_row(amd, card, picks):
    """The combine takes a row's slots four at a time: counts that leave some of a batch over."""
    test_prefill_layer_against_oracle(amd, card, 512, 256, 64, picks, 70, [2, 3, 4], 0.0)


@pytest.mark.parametrize("hidden,inner,width_choices", [(512, 384, [2, 3, 4]), (128, 128, [40])])
def test_thin_gemm_at_the_edges_of_its_blocks(amd, card, hidden, inner, width_choices):
    """A call of few pairs an expert (exl3_tcp_gemm_thin: blocks of 48 pairs, instances of one to three blocks of sixteen):
    experts of 15, 16, 17, 32, 33, 47, 48, 49 and 161 pairs, others with none; against the oracle (the bound of the layer
    test above), and the same rows in a call of more pairs an expert (exl3_tcp_gemm: the same operands and weights, the
    float32 sums in another order). What the order moves: here and there a down operand's fp16 rounding by a place, 2^-10 of
    a value; one of five times the operands' rms among `inner` of them moves an output by 5 2^-10 / sqrt(inner) of its rms
    (2.5e-4 at 384). Four such in one output are allowed."""
    say("thin prefill", hidden, inner, width_choices)
    experts_n, picks, rows = 64, 2, 256
    first = np.repeat(np.arange(8), [15, 16, 17, 32, 33, 47, 48, 48])
    second = np.repeat([40, 41, 63], [161, 49, 46])
    layer, matrices, widths = build_layer(amd, card, hidden, inner, experts_n, picks, 3 * rows, 23, width_choices)
    x = to_bf16(normals(35, 3 * rows * hidden)).reshape(3 * rows, hidden)
    table = np.zeros((3 * rows, picks), dtype=np.dtype([("expert", "<u4"), ("route_weight", "<f4")]))
    table["expert"] = np.tile(np.stack([first, np.random.default_rng(3).permutation(second)], axis=1), (3, 1))
    table["route_weight"] = np.random.default_rng(4).uniform(0.1, 1.0, (3 * rows, picks)).astype(np.float32)
    picks_at, got = card.place(table.view(np.uint8).reshape(-1)), {}
    for count in (rows, 3 * rows):  # 8 and 24 pairs an expert on average
        layer.rows, layer.tcp_workspace_offset = count, None
        layer.set_rows(x[:count], count)
        card.upload(layer.out_offset, np.full(count * hidden * 4, 0xFF, dtype=np.uint8))
        launches = layer.tcp_launches(picks_at)
        assert launches[3].grid[2] == (8 if count == rows else 2) and launches[5].grid[2] == (4 if count == rows else 1)
        card.run(launches)
        got[count] = layer.output()[:rows].copy()
    layer.rows = rows
    want = oracle_layer(layer, x[:rows], np.ascontiguousarray(table["expert"][:rows]), np.ascontiguousarray(table["route_weight"][:rows]), matrices, widths)
    scale = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    error, apart = (float(np.max(np.abs(got[rows] - other))) / scale for other in (want, got[3 * rows]))
    say("  max error %.2e of the output's rms, the two forms %.2e apart" % (error, apart))
    assert error <= 4e-3 and apart <= 4 * 5 * 2.0 ** -10 / inner ** 0.5


@pytest.mark.parametrize("counts,thin", [((70, 301, 512), True), ((513, 700), False)])
def test_a_rows_bits_do_not_depend_on_the_calls_other_rows(amd, card, counts, thin):
    """The same seventy rows in calls of several sizes on one side of the line between the two GEMM forms (16 pairs an expert on
    average): every output bit."""
    say("prefill rows of other calls", counts)
    hidden, inner, experts_n, picks, kept = 512, 384, 64, 2, 70
    layer, _, _ = build_layer(amd, card, hidden, inner, experts_n, picks, counts[-1], 27, [2, 3, 4])
    x = to_bf16(normals(37, counts[-1] * hidden)).reshape(counts[-1], hidden)
    table = np.zeros((counts[-1], picks), dtype=np.dtype([("expert", "<u4"), ("route_weight", "<f4")]))
    rng = np.random.default_rng(5)
    table["expert"] = np.argsort(rng.random((counts[-1], experts_n)), axis=1)[:, :picks]
    table["route_weight"] = rng.uniform(0.1, 1.0, table.shape).astype(np.float32)
    outputs = []
    for count in counts:
        order = np.concatenate([np.arange(kept, count), np.arange(kept)])  # the kept rows last: other places, other chunks' columns
        picks_at = card.place(np.ascontiguousarray(table[order]).view(np.uint8).reshape(-1))
        layer.rows, layer.tcp_workspace_offset = count, None
        layer.set_rows(np.ascontiguousarray(x[order]), count)
        launches = layer.tcp_launches(picks_at)
        assert launches[5].grid[2] == (4 if thin else 1)
        card.run(launches)
        outputs.append(layer.output()[count - kept:].view(np.uint32).copy())
    assert all(np.array_equal(outputs[0], other) for other in outputs[1:]) and np.any(outputs[0] != 0)


def test_prefill_equals_fused_decode_on_the_same_rows(amd, card):
    """Eight rows through the fused decode and through the prefill form: the same operands, weights and float32 chains
    cut differently along k (the decode's slices against one chain): equal within float32 rounding of the sums."""
    say("prefill against the fused decode")
    hidden, inner, experts_n, picks, rows = 512, 256, 64, 4, 8
    layer, matrices, widths = build_layer(amd, card, hidden, inner, experts_n, picks, rows, 22, [2, 3, 4])
    x = to_bf16(normals(33, rows * hidden)).reshape(rows, hidden)
    layer.set_rows(x, rows)
    card.run(layer.projection_launch())
    card.run(layer.select_launch(0))
    card.run(layer.tc_launches())
    decode = layer.output().copy()
    wide = layer.wide_router()
    card.run(wide.launches()[0:1])
    card.run(layer.tcp_launches(wide.ranges["picks"].byte_offset))
    prefill = layer.output()
    scale = float(np.sqrt(np.mean(decode.astype(np.float64) ** 2)))
    error = float(np.max(np.abs(prefill - decode))) / scale
    say("  max difference %.2e of rms" % error)
    assert error <= 2e-4


@pytest.mark.parametrize("limit", [10.0, 0.0])
def test_activation_of_products_that_are_no_numbers(amd, card, limit):
    """The activation of gate and up products given to it, among them blocks of infinities and not-a-numbers: with a limit a gate
    that is not a number is the limit and such an up product the lower one (fminf(gate, limit), fminf(fmaxf(up, -limit), limit));
    without one they stay what they are. Against the same steps in float64. What float32 moves: a down operand is a sum of 128
    values, each of some ten roundings, then one to fp16: below 2^-10 of the block's largest value or sum of magnitudes / 128."""
    hidden, inner, experts_n, picks, rows = 128, 256, 64, 2, 70
    say("activation", limit)
    layer, matrices, widths = build_layer(amd, card, hidden, inner, experts_n, picks, rows, 43, [2, 4])
    layer.limit = limit
    layer.set_rows(to_bf16(normals(44, rows * hidden)).reshape(rows, hidden), rows)
    card.upload(layer.bias_offset, np.zeros(experts_n, dtype=np.float32))
    card.run(layer.projection_launch())
    wide = layer.wide_router()
    card.run(wide.launches()[0:1])
    experts = wide.read("picks", np.dtype([("expert", "<u4"), ("route_weight", "<f4")])).reshape(-1)["expert"]
    launches = layer.tcp_launches(wide.ranges["picks"].byte_offset)
    card.run(launches[0:3])
    pairs, layout = rows * picks, layer.tcp_layout
    products = (normals(45, 2 * pairs * inner) * 30.0).astype(np.float32).reshape(2, pairs, inner)
    for place, (gate, up) in enumerate([(np.nan, 1.0), (1.0, np.nan), (np.nan, np.nan), (np.inf, 2.0), (-np.inf, 2.0), (3.0, np.inf),
                                        (3.0, -np.inf), (3e38, -3e38), (-0.0, 0.0)]):
        products[0, 7 * place, 128:], products[1, 7 * place, 128:] = gate, up
    card.upload(layer.tcp_workspace_offset + layout["gate_up"], products)
    card.run(launches[4:5])
    got = card.download(layer.tcp_workspace_offset + layout["operands"], pairs * inner * 2, np.float16).reshape(pairs, inner).astype(np.float64)
    sorted_pairs = card.download(layer.tcp_workspace_offset + layout["sorted"], pairs * 4, np.uint32)
    signs = np.array([[(-1.0) ** bin(i & j).count("1") for j in range(128)] for i in range(128)])

    def block_sums(values):  # the butterflies in float32, as an infinity meets its like in them
        values = values.astype(np.float32).reshape(-1, 128).copy()
        for distance in (1, 2, 4, 8, 16, 32, 64):
            pair = values.reshape(-1, 64 // distance, 2, distance)
            values = np.stack([pair[:, :, 0] + pair[:, :, 1], pair[:, :, 0] - pair[:, :, 1]], axis=2).reshape(-1, 128)
        return values.reshape(-1)

    with np.errstate(all="ignore"):
        for place in range(pairs):
            trio = matrices[int(experts[sorted_pairs[place]])]
            e = int(experts[sorted_pairs[place]])
            scales = []
            for matrix, (rows_in, columns_out) in enumerate([(hidden, inner), (hidden, inner), (inner, hidden)]):
                code_bytes = int(orc.orc_exl3_code_bytes(rows_in, columns_out, int(widths[e, matrix])))
                halves = np.ascontiguousarray(trio[matrix][code_bytes:code_bytes + 2 * (rows_in + columns_out)]).view(np.float16).astype(np.float64)
                scales.append(halves[rows_in:] if matrix < 2 else halves[:rows_in])
            gate, up = [block_sums(products[side, place]).astype(np.float64) / np.sqrt(128.0) * scales[side] for side in (0, 1)]
            if limit > 0.0:
                gate, up = np.fmin(gate, limit), np.fmin(np.fmax(up, -limit), limit)
            values = gate / (1.0 + np.exp(-gate)) * up * scales[2]
            want = (values.reshape(-1, 128) @ signs / np.sqrt(128.0)).reshape(-1)
            for block in range(inner // 128):
                here = slice(128 * block, 128 * block + 128)
                if not np.isfinite(values[here]).all() or np.abs(want[here]).max() > 6e4:
                    assert not np.isfinite(got[place, here]).all(), (place, block)
                    continue
                bound = 2.0 ** -10 * max(np.abs(want[here]).max(), np.abs(values[here]).mean())
                assert np.abs(got[place, here] - want[here]).max() <= bound, (place, block)


@pytest.mark.parametrize("rows", [3071, 3072])
def test_operands_about_the_line_of_their_streamed_form(amd, card, rows):
    """The operands of a step are written past the caches from 96 Mi values an array on (3072 rows of 8 picks by 4096): the row
    below the line and the line itself, bit for bit the oracle's, the first and the last place among those looked at."""
    hidden, inner, experts_n, picks = 4096, 128, 64, 8
    say("streamed operands", rows)
    layer, matrices, widths = build_layer(amd, card, hidden, inner, experts_n, picks, rows, 61, [2, 4])
    x = to_bf16(normals(62, rows * hidden)).reshape(rows, hidden)
    layer.set_rows(x, rows)
    card.upload(layer.bias_offset, np.zeros(experts_n, dtype=np.float32))
    card.run(layer.projection_launch())
    wide = layer.wide_router()
    card.run(wide.launches()[0:1])
    experts = wide.read("picks", np.dtype([("expert", "<u4"), ("route_weight", "<f4")])).reshape(-1)["expert"]
    card.run(layer.tcp_launches(wide.ranges["picks"].byte_offset)[0:3])
    pairs, layout = rows * picks, layer.tcp_layout
    sorted_pairs = card.download(layer.tcp_workspace_offset + layout["sorted"], pairs * 4, np.uint32)
    operands = card.download(layer.tcp_workspace_offset + layout["operands"], 2 * pairs * hidden * 2, np.uint16).reshape(2, pairs, hidden)
    for place in [0, 1, pairs - 2, pairs - 1] + list(range(97, pairs, pairs // 29)):
        pair = int(sorted_pairs[place])
        e = int(experts[pair])
        for side in range(2):
            code_bytes = int(orc.orc_exl3_code_bytes(hidden, inner, int(widths[e, side])))
            suh = np.ascontiguousarray(matrices[e][side][code_bytes:code_bytes + 2 * hidden]).view(np.uint16)
            expect = np.zeros(hidden, dtype=np.uint16)
            orc.orc_exl3_operand(ptr(x[pair // picks], u16p), ptr(suh, u16p), hidden, ptr(expect, u16p))
            assert np.array_equal(operands[side, place], expect), (place, side)
