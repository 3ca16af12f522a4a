"""GPU parity of the wide routed experts whose weights lie in gfx950's own lane order (WEIGHT_FORMAT_E2M1_GFX950,
WEIGHT_FORMAT_E4M3_GFX950, WEIGHT_FORMAT_E4M3_BLOCK128_GFX950; the matrices go through the library's load-time re-lay-out, weight_format_gfx950_pack), through
the C ABI: byte for byte the outputs of the same layer in the reference's lay-out (kernel_wide_linear.hip's launches,
which tests/test_gpu_wide_linear.py holds byte for byte to the job-table kernels and those to the oracle), and the
layer's rows against the CPU oracle reading the re-laid-out bytes itself."""
import ctypes as C
import sys

import numpy as np
import pytest

from _oracle import f32p, normals, orc, ptr, to_bf16, u16p, u32p

pytestmark = pytest.mark.gpu

E2M1, E4M3, B128, E2M1_GFX950, E4M3_GFX950, B128_GFX950 = 3, 5, 6, 7, 8, 9
NATIVE_OF = {E2M1: E2M1_GFX950, E4M3: E4M3_GFX950, B128: B128_GFX950}
NAMES = ("hidden_codes", "hidden_exponents", "hidden_operands", "pair_output", "row_output")


def say(*words):
    print(*words, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def amd():
    import anemone_amd
    return anemone_amd


@pytest.fixture(scope="module")
def card(amd):
    card = amd.Card(3 << 30)
    yield card
    card.close()


@pytest.fixture(autouse=True)
def fresh_arena(card):
    card.cursor = 256
    yield


def matrices_of(hidden, inner, experts_n, seed, fmt, distinct=8):
    from anemone_amd import workloads
    matrix = workloads.fp4_matrix if fmt == E2M1 else workloads.fp8_block128_matrix if fmt == B128 else workloads.fp8_matrix
    trios = [[matrix(seed * 1000 + 3 * e + 0, inner, hidden), matrix(seed * 1000 + 3 * e + 1, inner, hidden),
              matrix(seed * 1000 + 3 * e + 2, hidden, inner)] for e in range(distinct)]
    return [trios[e % distinct] for e in range(experts_n)]


def run_wide(card, layer, x, live):
    layer.set_rows(x, live)
    card.run(layer.projection_launch())
    wide = layer.wide_router()
    card.run(wide.launches())
    card.run(layer.quantize_launch())
    for name in NAMES:
        card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
    card.run(layer.wide_expert_launches(wide))
    return [layer.read(name).copy() for name in NAMES], wide


@pytest.mark.parametrize("hidden,inner,experts_n,picks,rows,live,fmt", [
    (512, 256, 64, 4, 300, 300, E2M1),    # whole blocks of four strips
    (640, 384, 64, 4, 200, 177, E2M1),    # the last block of each product holds two live strips; rows beyond the live ones
    (512, 256, 64, 8, 40, 40, E2M1),      # most tiles hold a few pairs
    (512, 256, 64, 4, 300, 300, E4M3),
    (640, 384, 64, 2, 450, 449, E4M3),
    (512, 256, 64, 1, 700, 700, E2M1),    # one pick a row
    (512, 256, 64, 8, 1500, 1500, E2M1),  # runs of three tiles and more
    (640, 384, 64, 8, 1100, 1003, E2M1),
    (512, 256, 64, 8, 1500, 1401, E4M3),  # blocks of two tiles of one expert, a run's odd last tile alone
    (512, 256, 64, 8, 6000, 5999, E4M3),  # runs of a dozen tiles: the places of a run's tiles by the lanes' look back
    (512, 256, 64, 1, 4300, 4300, -E4M3), # one expert takes every row: a run of 68 tiles, the look back goes round again
    (512, 256, 64, 4, 300, 300, B128),    # float32 scales of 128 x 128 blocks: the quantizer between the two products
    (640, 384, 64, 2, 450, 449, B128),
    (512, 256, 64, 8, 1500, 1401, B128),
    (512, 256, 64, 1, 4300, 4300, -B128),
    # 4-bit weights, whose blocks go in the order of runs: one expert takes every row (a run of 68 tiles: cut in pieces of 16
    # and where a window of 64 tiles ends), the same with the other experts' tiles around it, and few rows of many experts
    # (more unused tiles behind the used ones than the first look takes)
    (512, 256, 64, 1, 4300, 4300, -E2M1),
    (640, 384, 64, 3, 4300, 4287, -E2M1),
    (256, 128, 384, 1, 100, 100, -E2M1),
    # chains of one, two and three K steps: fewer steps than sets of weight registers and stages of columns
    (128, 128, 64, 4, 300, 300, E2M1),
    (256, 128, 64, 4, 300, 297, E2M1),
    (384, 256, 64, 2, 500, 500, E2M1),
    (128, 128, 64, 4, 600, 600, E4M3),
    (256, 128, 64, 8, 300, 300, E4M3),
    (384, 256, 64, 2, 500, 499, E4M3),
    (128, 128, 64, 4, 600, 600, B128),
    (256, 128, 64, 8, 300, 299, B128),
    (384, 256, 64, 2, 500, 500, B128),
])
def test_native_equals_the_reference_lay_out_byte_for_byte(amd, card, hidden, inner, experts_n, picks, rows, live, fmt):
    say("native experts", hidden, inner, experts_n, picks, rows, live, fmt)
    one_expert, fmt = fmt < 0, abs(fmt)
    matrices = matrices_of(hidden, inner, experts_n, 21, fmt)
    router = to_bf16(normals(26, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    x = to_bf16(normals(31, rows * hidden)).reshape(rows, hidden)
    bias = np.zeros(experts_n, dtype=np.float32)
    if one_expert:
        bias[5] = 100.0
    reference = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router, weight_format=fmt)
    card.upload(reference.bias_offset, bias)
    want, wide = run_wide(card, reference, x, live)
    counts = np.bincount(wide.read("picks", np.dtype([("expert", "<u4"), ("route_weight", "<f4")]))["expert"][:live * picks], minlength=experts_n)
    say("  pairs of the busiest expert:", int(counts.max()))
    native = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router,
                          weight_format=NATIVE_OF[fmt])
    card.upload(native.bias_offset, bias)
    got, _ = run_wide(card, native, x, live)
    pairs = live * picks
    for name, a, b in zip(NAMES, want, got):
        per = a.size // (rows if name == "row_output" else rows * picks)
        count = (live if name == "row_output" else pairs) * per
        differing = np.flatnonzero(a.reshape(-1)[:count] != b.reshape(-1)[:count])
        say("  %s: %d of %d bytes differ" % (name, differing.size, count))
        assert differing.size == 0, (name, differing[:8], per)
        assert a.reshape(-1)[:count].tobytes() != bytes([0xEE]) * count, "the launches wrote"
    if live < rows:  # nothing is written for the pairs of the rows beyond the live ones
        for name, b in zip(NAMES[:4], got[:4]):
            if fmt == B128 and name in ("hidden_codes", "hidden_exponents"):
                continue  # the quantizer of 128 values a scale is a launch over every pair the step has room for
            per = b.size // (rows * picks)
            assert np.all(b.reshape(-1)[pairs * per:] == 0xEE), name


@pytest.mark.parametrize("hidden,inner,picks,rows,fmt", [
    # the columns' scale words come four K steps at a time: chains that end inside a chunk, with one, at its first step
    (640, 896, 2, 100, E2M1), (1152, 1024, 2, 100, E2M1),
    (640, 896, 2, 100, E4M3), (1152, 1024, 2, 100, E4M3),
    (640, 896, 2, 100, B128), (1152, 1024, 2, 100, B128),
    # a lane holds the weights' scale words of a step: chains of more steps than the lanes that do
    (8320, 128, 2, 70, E4M3), (128, 8320, 2, 70, E4M3),
    (8320, 128, 2, 70, B128), (128, 8320, 2, 70, B128),
    # one expert's pairs: every number of column blocks of a block of two tiles, each with its own share of a wavefront's loads
    *[(512, 256, 1, rows, -fmt) for rows in (9, 30, 41, 64, 70, 96, 100, 128) for fmt in (E4M3, B128)],
    # the same where the expert has a full block before it: weights that two blocks read are not asked for as a stream
    *[(512, 256, 1, 128 + rows, -fmt) for rows in (9, 30, 41, 64, 70, 96, 100, 128) for fmt in (E4M3, B128)],
])
def test_native_chunks_of_scale_words(amd, card, hidden, inner, picks, rows, fmt):
    test_native_equals_the_reference_lay_out_byte_for_byte(amd, card, hidden, inner, 64, picks, rows, rows, fmt)


@pytest.mark.parametrize("fmt", [E2M1, E4M3, B128])
def test_native_layer_against_oracle(amd, card, fmt):
    """The layer in gfx950's lay-out against the CPU oracle reading the SAME re-laid-out bytes (its own reading of the
    format, oracle/orc_linear.c) with the picks the card made."""
    say("native layer against the oracle", fmt)
    from test_gpu_router_wide import oracle_wide
    hidden, inner, experts_n, picks, rows, live = 512, 256, 64, 4, 150, 143
    native_format = NATIVE_OF[fmt]
    matrices = matrices_of(hidden, inner, experts_n, 33, fmt, distinct=64)
    router = to_bf16(normals(5, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    layer = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router, weight_format=native_format)
    x = to_bf16(normals(9, rows * hidden)).reshape(rows, hidden)
    got, _ = run_wide(card, layer, x, live)
    scores = card.download(layer.scores_offset, rows * experts_n * 4, np.float32).reshape(rows, experts_n)
    _, experts, weights, _, _, _, _ = oracle_wide(layer, scores, np.zeros(experts_n, dtype=np.float32), live)
    packed = [[amd.gfx950_pack(native_format, *((inner, hidden) if m < 2 else (hidden, inner)), matrix) for m, matrix in enumerate(trio)] for trio in matrices]
    pointers = (C.c_void_p * (experts_n * 3))(*[m.ctypes.data for trio in packed for m in trio])
    want = np.zeros((live, hidden), dtype=np.float32)
    orc.orc_linear_moe_layer(native_format, ptr(np.ascontiguousarray(x[:live]), u16p), live, hidden, inner, picks,
                             ptr(np.ascontiguousarray(experts[:live]), u32p), ptr(np.ascontiguousarray(weights[:live]), f32p),
                             experts_n, pointers, 10.0, ptr(want, f32p), None, None, 8)
    row_output = got[4].view(np.float32).reshape(rows, hidden)[:live]
    error = np.sqrt(np.mean((row_output - want) ** 2) / np.mean(want.astype(np.float64) ** 2))
    say("  layer rms error vs oracle: %.2e" % error)
    assert error < 2e-2


def special_rows(rows, hidden):
    """Rows of ordinary values; of values whose sums overflow (a gate of minus infinity makes a hidden value that is not a
    number); with infinities (a scale code of 255: every sum is not a number); of 1e30; with a value that is not a number."""
    x = normals(91, rows * hidden).reshape(rows, hidden).astype(np.float64)
    x[1::5] *= 1e38
    x[3::5] *= 1e30
    x = to_bf16(np.clip(x, -3e38, 3e38).astype(np.float32)).reshape(rows, hidden)
    x[2::5, 7] = 0x7F80
    x[4::5, 9] = 0x7FC1
    return x


@pytest.mark.parametrize("fmt", [E2M1, E4M3, B128])
@pytest.mark.parametrize("limit", [10.0, 1e12, 1e30])
def test_finishes_of_values_without_order_and_of_large_scales(amd, card, fmt, limit):
    """The finishes' side paths: hidden values and down sums that are not numbers, scale codes of the hidden values above 146
    (an activation limit of 1e12 and 1e30 lets them through), in column blocks beside ordinary ones: the wide launches byte
    for byte the job-table kernels', the native launches byte for byte theirs."""
    say("finishes of special values", fmt, limit)
    hidden, inner, experts_n, picks, rows = 256, 128, 64, 4, 120
    from anemone_amd import workloads
    # gates and ups of deviation 16 times the rows' values and more: sums of the second kind of row overflow
    matrix, loud = {E2M1: (workloads.fp4_matrix, dict(scale_code=126)), E4M3: (workloads.fp8_matrix, dict(deviation=1.5)),
                    B128: (workloads.fp8_block128_matrix, dict(deviation=1.5))}[fmt]
    trios = [[matrix(9300 + 3 * e, inner, hidden, **loud), matrix(9301 + 3 * e, inner, hidden, **loud), matrix(9302 + 3 * e, hidden, inner)] for e in range(8)]
    matrices = [trios[e % 8] for e in range(experts_n)]
    router = to_bf16(normals(95, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    x = special_rows(rows, hidden)
    made = [amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router, limit=limit,
                         weight_format=weight_format, gate_up_slices=1, down_slices=1) for weight_format in (fmt, NATIVE_OF[fmt])]
    scores = normals(97, rows * experts_n).astype(np.float32)  # the rows' own scores would not be numbers
    outputs = []
    for layer, wide_form in ((made[0], False), (made[0], True), (made[1], True)):
        layer.set_rows(x, rows)
        card.upload(layer.scores_offset, scores)
        wide = layer.wide_router()
        card.run(wide.launches())
        card.run(layer.quantize_launch())
        for name in ("hidden",) + NAMES:
            card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
        card.run(layer.wide_expert_launches(wide) if wide_form else layer.expert_launches(wide))
        outputs.append([layer.read(name).copy() for name in NAMES])
        if not wide_form:
            values, sums = layer.read("hidden", np.uint16), layer.read("pair_output", np.uint16)
            exponents = layer.read("hidden_exponents", np.uint32 if fmt == B128 else np.uint8)
            say("  hidden values that are not numbers %d, down sums %d, largest scale %d" %
                (np.count_nonzero(values == 0x7FC0), np.count_nonzero(sums == 0x7FC0), int(exponents.max())))
            assert np.any(values == 0x7FC0)
            if limit > 10.0:
                assert fmt == B128 or np.any(exponents > 146)
            if limit == 1e30:
                assert np.any(sums == 0x7FC0)
    for name, narrow, wide, native in zip(NAMES, *outputs):
        if fmt == B128 and name == "hidden_operands":
            continue  # the wide launches leave the hidden values there, the job-table kernels nothing
        assert np.array_equal(narrow, wide), name
        assert np.array_equal(narrow, native), name


@pytest.mark.parametrize("fmt,outputs", [(E2M1, 64), (E2M1, 192), (E2M1, 320), (E2M1, 576), (E4M3, 32), (E4M3, 96), (E4M3, 160)])
def test_down_outputs_of_half_a_strip(amd, card, fmt, outputs):
    """Down products of any outputs the formats store (4-bit: 64 k; one byte: 32 k), not of whole strips of 128: a strip that
    begins at the last tiles again, a matrix of fewer tiles than a strip; the reference's lay-out through the wide and the
    job-table kernels, gfx950's through whole and narrow strips."""
    say("down outputs", fmt, outputs)
    from anemone_amd import workloads
    hidden, inner, experts_n, picks, rows = 640, 256, 64, 2, 150

    class Layer(amd.Fp4Layer):
        def experts_description(self, wide=None):
            description = super().experts_description(wide)
            description.down_shape = amd.Shape(outputs, self.I, self.bits, 0)
            return description

        def wide_router(self):
            return amd.WideRouter(self, self.rows, self.weight_format, amd.Shape(self.I, self.H, self.bits, 0), amd.Shape(outputs, self.I, self.bits, 0))
    down = workloads.fp4_matrix if fmt == E2M1 else workloads.fp8_matrix
    trios = [trio[:2] + [down(5100 + e, outputs, inner)] for e, trio in enumerate(matrices_of(hidden, inner, 8, 99, fmt))]
    router = to_bf16(normals(101, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    x = to_bf16(normals(103, rows * hidden)).reshape(rows, hidden)
    packed = [[amd.gfx950_pack(NATIVE_OF[fmt], *((inner, hidden) if m < 2 else (outputs, inner)), matrix) for m, matrix in enumerate(trio)] for trio in trios]
    count, results = rows * picks, {}
    for native, matrices in ((False, trios), (True, packed)):
        layer = Layer(card, hidden, inner, experts_n, picks, rows, [matrices[e % 8] for e in range(experts_n)], router_weights_bf16=router,
                      weight_format=fmt, gate_up_slices=1, down_slices=1)
        if native:  # the matrices are packed already, in shapes of their own
            layer.weight_format, layer.native = NATIVE_OF[fmt], True
        _, wide = run_wide(card, layer, x, rows)
        forms = {"wide": layer.wide_expert_launches(wide)}
        if not native:
            forms["jobs"] = layer.expert_launches(wide)
        elif fmt == E2M1:
            narrow = forms["narrow"] = layer.wide_expert_launches(wide)
            narrow[0].kernel, narrow[1].kernel = layer.native_kernels.native_expert_gate_up_narrow, layer.native_kernels.native_expert_down_narrow
            narrow[0].grid[0], narrow[1].grid[0] = -(-inner // 128), -(-outputs // 256)
            forms["wide"][0].kernel, forms["wide"][1].kernel = layer.native_kernels.native_expert_gate_up, layer.native_kernels.native_expert_down
            forms["wide"][0].grid[0], forms["wide"][1].grid[0] = -(-inner // 256), -(-outputs // 512)
        for form, launches in forms.items():
            for name in NAMES:
                card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
            card.run(launches)
            sums, sums_of_rows = layer.read("pair_output"), layer.read("row_output")
            assert np.all(sums[count * outputs * 2:] == 0xEE) and np.all(sums_of_rows[rows * outputs * 4:] == 0xEE), (native, form)
            results[native, form] = (sums[:count * outputs * 2].copy(), sums_of_rows[:rows * outputs * 4].copy())
    first = results[False, "jobs"]
    assert np.any(first[0] != 0xEE)
    for which, result in results.items():
        assert all(np.array_equal(a, b) for a, b in zip(first, result)), which


def run_jobs(card, layer, x, live):
    layer.set_rows(x, live)
    card.run(layer.projection_launch())
    card.run(layer.select_launch(0))
    card.run(layer.quantize_launch())
    for name in ("hidden",) + NAMES:
        card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
    card.run(layer.expert_launches())
    return [layer.read(name).copy() for name in ("hidden",) + NAMES], layer.jobs().copy()


@pytest.mark.parametrize("hidden,inner,picks,rows,live,fmt,gate_up_slices,down_slices", [
    (512, 256, 4, 8, 8, E2M1, 4, 2),     # the slice counts the card's order takes
    (512, 256, 4, 8, 7, E2M1, 1, 1),     # one chain; a row beyond the live ones
    (1024, 512, 8, 3, 3, E2M1, 8, 4),
    (640, 384, 2, 5, 5, E2M1, 2, 1),     # five K steps over two slices: chains of two and three steps
    (512, 256, 4, 8, 8, E4M3, 4, 2),
    (640, 384, 8, 2, 2, E4M3, 1, 2),     # 40 tiles of the gate product: strips of two
    (1024, 512, 1, 8, 5, E4M3, 8, 4),
    (512, 256, 4, 8, 8, B128, 4, 2),
    (640, 384, 8, 2, 2, B128, 1, 2),
    (1024, 512, 1, 8, 5, B128, 8, 4),
    (640, 384, 2, 5, 5, B128, 2, 1),
    (128, 128, 4, 8, 8, E2M1, 1, 1),     # one K step
    (256, 128, 4, 8, 7, E4M3, 2, 1),     # two K steps over two slices: a step a chain
    (128, 128, 2, 6, 6, B128, 1, 1),
    (384, 256, 8, 4, 4, E2M1, 1, 2),
])
def test_native_job_table_kernels_equal_the_reference_lay_out(amd, card, hidden, inner, picks, rows, live, fmt, gate_up_slices, down_slices):
    """The job-table kernels (a thin step's) of the formats in gfx950's lane order, expert_gate_up_gfx950_<S> and its like:
    byte for byte what the reference-format kernels of the same slice counts write for the same matrices."""
    say("native job-table kernels", hidden, inner, picks, rows, live, fmt, gate_up_slices, down_slices)
    experts_n = 64
    matrices = matrices_of(hidden, inner, experts_n, 41, fmt, distinct=16)
    router = to_bf16(normals(43, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    x = to_bf16(normals(47, rows * hidden)).reshape(rows, hidden)
    reference = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router, weight_format=fmt,
                             gate_up_slices=gate_up_slices, down_slices=down_slices)
    want, want_jobs = run_jobs(card, reference, x, live)
    native = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices, router_weights_bf16=router,
                          weight_format=NATIVE_OF[fmt], gate_up_slices=gate_up_slices, down_slices=down_slices)
    got, got_jobs = run_jobs(card, native, x, live)
    assert np.array_equal(want_jobs["expert"], got_jobs["expert"]) and np.array_equal(want_jobs["pair_index"], got_jobs["pair_index"])
    pairs = live * picks
    for name, a, b in zip(("hidden",) + NAMES, want, got):
        per = a.size // (rows if name == "row_output" else rows * picks)
        count = (live if name == "row_output" else pairs) * per
        differing = np.flatnonzero(a.reshape(-1)[:count] != b.reshape(-1)[:count])
        say("  %s: %d of %d bytes differ" % (name, differing.size, count))
        assert differing.size == 0, (name, differing[:8], per)
        if not (fmt == B128 and name == "hidden_operands"):  # the quantizer of 128 values a scale writes no operands
            assert a.reshape(-1)[:count].tobytes() != bytes([0xEE]) * count, "the launches wrote"


@pytest.mark.parametrize("steps", range(1, 8))
@pytest.mark.parametrize("fmt", [E2M1, E4M3])
def test_native_thin_chains_of_every_length(amd, card, steps, fmt):
    """The job-table kernels' last K steps, an instance for every number of them, and the steady state ahead of them."""
    test_native_job_table_kernels_equal_the_reference_lay_out(amd, card, 128 * steps, 128 * (8 - steps), 2, 5, 5, fmt, 1, 1)


@pytest.mark.parametrize("hidden,inner,rows,live", [(512, 384, 100, 100), (640, 128, 70, 67), (256, 128, 2500, 2497)])
def test_narrow_and_whole_strips_give_the_same_bytes(amd, card, hidden, inner, rows, live):
    """The 4-bit wide launches of strips of half the tiles (native_expert_gate_up_narrow_1, native_expert_down_narrow_1) and
    of whole strips, over the same rows: every output byte. Widths that end inside a block of either; runs of two tiles."""
    say("narrow and whole strips", hidden, inner, rows, live)
    experts_n, picks = 64, 2
    router = to_bf16(normals(81, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    layer = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices_of(hidden, inner, experts_n, 83, E2M1),
                         router_weights_bf16=router, weight_format=E2M1_GFX950)
    x = to_bf16(normals(85, rows * hidden)).reshape(rows, hidden)
    _, wide = run_wide(card, layer, x, live)
    native = amd.LinearNativeKernels()
    amd.check(card.lib.linear_native_kernels_prepare(amd.backend_table(), card.handle, amd.ARITHMETIC_CLASS_GFX950, C.byref(native)), "prepare")
    launches, outputs = layer.wide_expert_launches(wide), []
    for gate_up, down, tiles in ((native.native_expert_gate_up_narrow, native.native_expert_down_narrow, 1),
                                 (native.native_expert_gate_up, native.native_expert_down, 2)):
        launches[0].kernel, launches[1].kernel = gate_up, down
        launches[0].grid[0], launches[1].grid[0] = -(-inner // (128 * tiles)), -(-hidden // (256 * tiles))
        for name in NAMES:
            card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
        card.run(launches)
        outputs.append([layer.read(name).copy() for name in NAMES])
    for name, a, b in zip(NAMES, *outputs):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), name
        assert not np.all(a.view(np.uint8) == 0xEE)


@pytest.mark.parametrize("fmt", [E4M3, B128])
@pytest.mark.parametrize("hidden,inner,experts_n,picks,rows,live,one_expert", [
    (128, 128, 64, 4, 600, 597, False),   # one K step; a strip of a wavefront alone, three past the matrix
    (256, 384, 64, 8, 300, 300, False),   # two K steps; a block's last strips past the matrix
    (512, 256, 64, 8, 1500, 1401, False), # blocks of two tiles of one expert, a run's odd last tile alone
    (640, 384, 64, 3, 4300, 4287, True),  # a run of 68 tiles among the others: pieces of 16, and where a window of 64 tiles ends
    (256, 128, 384, 1, 100, 100, False),  # more unused tiles behind the used ones than the first look takes
])
def test_whole_and_half_strips_of_one_byte_weights_give_the_same_bytes(amd, card, hidden, inner, experts_n, picks, rows, live, one_expert, fmt):
    """The one-byte launches of strips of twice the tiles (native_expert_gate_up_e4m3_whole_1 and its like, whose blocks go in the
    order of runs) and the others, over the same rows: every output byte that a launch writes, and none besides."""
    say("whole and half strips", fmt, hidden, inner, experts_n, picks, rows, live)
    router = to_bf16(normals(87, experts_n * hidden) * 0.02).reshape(experts_n, hidden)
    layer = amd.Fp4Layer(card, hidden, inner, experts_n, picks, rows, matrices_of(hidden, inner, experts_n, 89, fmt),
                         router_weights_bf16=router, weight_format=NATIVE_OF[fmt])
    if one_expert:
        card.upload(layer.bias_offset, np.where(np.arange(experts_n) == 5, 100.0, 0.0).astype(np.float32))
    x = to_bf16(normals(91, rows * hidden)).reshape(rows, hidden)
    _, wide = run_wide(card, layer, x, live)
    native, infix = layer.native_kernels, "b128" if fmt == B128 else "e4m3"
    launches, outputs = layer.wide_expert_launches(wide), []
    first, second = launches[0], launches[2 if fmt == B128 else 1]
    for suffix, tiles, stages in (("", 1, 3), ("_whole", 2, 2)):
        first.kernel, second.kernel = getattr(native, "native_expert_gate_up_" + infix + suffix), getattr(native, "native_expert_down_" + infix + suffix)
        first.grid[0], second.grid[0] = -(-inner // (64 * tiles)), -(-hidden // (128 * tiles))
        first.dynamic_shared_byte_count, second.dynamic_shared_byte_count = 2 * 16384 + 4096, stages * 16384 + 4096
        for name in NAMES:
            card.upload(layer.ranges[name].byte_offset, np.full(layer.ranges[name].byte_count, 0xEE, dtype=np.uint8))
        card.run(launches)
        outputs.append([layer.read(name).copy() for name in NAMES])
    for name, a, b in zip(NAMES, *outputs):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), name
        if not (fmt == B128 and name == "hidden_operands"):
            assert not np.all(a.view(np.uint8) == 0xEE)
