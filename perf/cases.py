"""Performance cases of the routed-expert path: what a serving program has the library do in one step of one layer.

A case is one pass of a prepared step (`run`): the launches that the prepare functions of include/anemone_ops.h filled at
load time, queued with launch_run and not waited for, with the layer's weights, the router and the step's rows resident
in the card's arena. The sizes are the benchmark configurations' (hidden 4096, 256 experts of intermediate 2048, 8 picks
a row) at the row counts that a server meets: one user's token, a batch of users, a short prompt, a long prompt.

The launches of a step of R rows, as INTEGRATION.md's binding takes them:
  EXL3 experts         R <= 8: projection, select, the fused decode's five; to 64: the wide select in one block and the
                       fused decode over its job table; beyond: the picks and the prefill form's seven.
  FP4 / FP8 experts    R <= 8: projection, select, quantizer, the four of the job table; to 64: the same over the wide
                       select's job table; beyond: the wide select's tiles and the wide products.
  FFN site             R <= 8: the fused front, gate/up to down, the shared expert with its down joined; beyond: the mix
                       project and finish ahead of the router, the shared expert's four and the join behind the experts.
  linear               one EXL3 matrix: the chain's input, product and finish."""
import ctypes as C
import math
import weakref

import numpy as np
import torch

import anemone_amd as amd

FORMATS = {  # (format, gfx950's lane order): the stored format's code
    ("exl3", False): amd.WEIGHT_FORMAT_EXL3,
    ("e2m1", False): amd.WEIGHT_FORMAT_E2M1_SCALED, ("e2m1", True): amd.WEIGHT_FORMAT_E2M1_GFX950,
    ("e4m3", False): amd.WEIGHT_FORMAT_E4M3_SCALED, ("e4m3", True): amd.WEIGHT_FORMAT_E4M3_GFX950,
    ("e4m3_block128", False): amd.WEIGHT_FORMAT_E4M3_BLOCK128, ("e4m3_block128", True): amd.WEIGHT_FORMAT_E4M3_BLOCK128_GFX950,
}
WIDTH_CHOICES = {"mixed": ((2, 0.30), (3, 0.50), (4, 0.20)), "2": ((2, 1.0),), "2.5": ((40, 1.0),), "3": ((3, 1.0),), "4": ((4, 1.0),)}
MEAN_BITS = {"mixed": 2.9, "2": 2.0, "2.5": 2.5, "3": 3.0, "4": 4.0}


def layer_case(rows, weights, **other):
    case = {"kind": "layer", "weights": weights, "gfx950_order": False, "rows": rows, "hidden": 4096, "inner": 2048, "experts": 256, "picks": 8,
            "affinity": "sigmoid", "skew": 0.0, "widths": "mixed"}
    case.update(other)
    return case


def listed():
    return [
        # one matrix by one vector: the smallest call, a projection on its own
        {"name": "exl3_linear_b1", "kind": "linear", "rows": 1, "size": 4096, "widths": "4"},
        # decode of EXL3 weights: one user; a small batch (the configuration the repository's metric is quoted on); a
        # ragged batch of many users
        layer_case(1, "exl3", name="exl3_decode_1"),
        layer_case(8, "exl3", name="exl3_decode_8"),
        layer_case(37, "exl3", name="exl3_decode_37"),
        # a short prompt of a ragged length; a long prompt under skewed expert loads
        layer_case(203, "exl3", name="exl3_prefill_203"),
        layer_case(4096, "exl3", name="exl3_prefill_4096_zipf", skew=1.1),
        # FP8 weights of float32 128 x 128 blocks at one user, a batch, a prompt: as a pack stores them and re-laid at load
        layer_case(1, "e4m3_block128", name="fp8_decode_1"),
        layer_case(64, "e4m3_block128", name="fp8_decode_64", gfx950_order=True),
        layer_case(2048, "e4m3_block128", name="fp8_prefill_2048", gfx950_order=True),
        # FP4 weights: a whole FFN site (front, router, experts, shared expert, join) for a few users; a batch; a long prompt
        layer_case(5, "e2m1", name="fp4_site_decode_5", kind="site"),
        layer_case(32, "e2m1", name="fp4_decode_32", gfx950_order=True),
        layer_case(8192, "e2m1", name="fp4_prefill_8192", gfx950_order=True),
    ]


def log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("linear", "layer", "layer", "layer", "layer", "layer", "layer", "site", "site"))
    if kind == "linear":
        return {"kind": "linear", "rows": rng.randint(1, 8), "size": 128 * log_uniform(rng, 8, 64), "widths": rng.choice(("2", "2.5", "3", "4"))}
    weights = rng.choice(("exl3", "e2m1", "e4m3_block128", "e4m3")) if kind == "layer" else rng.choice(("e2m1", "e4m3"))
    # widths and expert counts up to the benchmark layer's bytes
    hidden, experts, picks = rng.choice((2048, 3072, 4096, 5120)), rng.choice((64, 128, 256, 384)), rng.choice((4, 6, 8))
    inner = min(128 * log_uniform(rng, 6, 16), 256 * 4096 * 2048 // (experts * hidden) // 128 * 128)
    # rows over the whole range, their products at most those of the long prompts listed (half as many for a whole site
    # and for one-byte weights)
    most_rows = {"exl3": 4096, "e2m1": 8192, "e4m3": 4096, "e4m3_block128": 4096}[weights] // (2 if kind == "site" else 1)
    rows = min(log_uniform(rng, 1, most_rows), most_rows * 8 * 4096 * 2048 // (picks * hidden * inner))
    return {"kind": kind, "weights": weights, "gfx950_order": weights != "exl3" and rng.random() < 0.5, "rows": rows, "hidden": hidden,
            "inner": inner, "experts": experts, "picks": picks, "affinity": rng.choice(("sigmoid", "sigmoid", "sqrt_softplus")),
            "skew": rng.choice((0.0, 0.0, 1.1)) if kind == "layer" else 0.0,
            "widths": rng.choice(("mixed", "mixed", "2", "2.5", "3", "4")) if weights == "exl3" else "mixed"}


def expert_loads(case):
    """The share of the rows that pick each expert, by rank: even, or Zipf(skew) with no expert above every row."""
    rows, picks, experts = case["rows"], case["picks"], case["experts"]
    pmf = (1.0 + np.arange(experts)) ** -case["skew"]
    load, capped = np.zeros(experts), np.zeros(experts, dtype=bool)
    for _ in range(experts):
        load = np.where(capped, 1.0, (picks - capped.sum()) * pmf / pmf[~capped].sum())
        over = (load > 1.0) & ~capped
        if not over.any():
            break
        capped |= over
    return load


def expert_matrix_bytes(case):
    weights = case["hidden"] * case["inner"]
    scales = 2.0 * (case["hidden"] + case["inner"]) if case["weights"] == "exl3" else \
        weights / 32 if case["weights"] == "e2m1" else weights / 1024 if case["weights"] == "e4m3" else weights / 4096
    return weights * {"exl3": MEAN_BITS[case["widths"]], "e2m1": 4.0}.get(case["weights"], 8.0) / 8 + scales


def work(case):
    rows = case["rows"]
    if case["kind"] == "linear":
        size = case["size"]
        return {"bytes": size * size * MEAN_BITS[case["widths"]] / 8 + 4.0 * size + rows * size * 6.0, "flops": 2.0 * rows * size * size}
    hidden, inner, experts, picks = case["hidden"], case["inner"], case["experts"], case["picks"]
    distinct = float(np.sum(1.0 - (1.0 - expert_loads(case)) ** rows))
    # the routed experts' matrices and the router's, the rows in, the sums and affinities out
    size = 3.0 * distinct * expert_matrix_bytes(case) + 2.0 * experts * hidden + rows * (6.0 * hidden + 4.0 * experts)
    flops = 6.0 * rows * picks * hidden * inner + 2.0 * rows * experts * hidden
    if case["kind"] == "site":
        # the mix project's weights, the four streams in and out, the shared expert
        size += 24.0 * 4 * hidden * 4 + rows * 4 * hidden * 4.0 + 3.0 * hidden * inner
        flops += 2.0 * rows * 24 * 4 * hidden + 6.0 * rows * hidden * inner
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """EXL3: fp16 operands and weights under float32 sums. FP4 / FP8: the hidden values are rounded to bfloat16 and then
    to E4M3, so that another order of the float32 sums moves a few of their codes by a place."""
    return {"rel": 1e-3} if case.get("weights", "exl3") == "exl3" else {"rel": 1e-2}


# ---- the card: one arena for every state, in slots that a state gives back when it is dropped ----

SLOT_BYTES, SLOTS = 9 << 30, 4


class Arena:
    """The process's one open card (a card opens once), its arena cut into slots, and the arena as a torch tensor. The
    library names places in the arena by offsets and hands out no address: it is read from the open card's record, and
    the arena's size beside it shows that it is the address."""

    def __init__(self):
        self.card = amd.Card(SLOTS * SLOT_BYTES)
        head = C.cast(self.card.handle, C.POINTER(C.c_uint64))  # struct device_card: the device, the stream, the arena, its bytes
        assert head[3] == self.card.arena_bytes, "struct device_card begins otherwise than expected"

        class Interface:
            __cuda_array_interface__ = {"shape": (self.card.arena_bytes,), "typestr": "|u1", "data": (head[2], False), "version": 2}
        self.bytes = torch.as_tensor(Interface(), device="cuda")
        self.free = list(range(SLOTS))

    def take(self):
        if not self.free:
            raise MemoryError("out of memory: every slot of the arena is held by a state")
        slot = self.free.pop(0)
        self.card.wait()  # what the slot's last owner queued
        self.card.cursor = slot * SLOT_BYTES + 256
        return slot

    def view(self, offset, dtype, *shape):
        size = torch.empty((), dtype=dtype).element_size()
        return self.bytes[offset:offset + math.prod(shape) * size].view(dtype).view(*shape)


_arena = None


def arena():
    global _arena
    if _arena is None:
        _arena = Arena()
    return _arena


class State:
    """A prepared step: its launches, its outputs as views of the arena, and what they stand on."""

    def __init__(self, launches, outputs, keep):
        self.step = amd.launches_of(len(launches))
        for i, launch in enumerate(launches):
            self.step[i] = launch
        self.outputs, self.keep = outputs, keep


def normals(generator, *shape):
    return torch.randn(*shape, generator=generator, device="cuda")


def exl3_codes(view, generator):
    """Uniformly random trellis codes: every bit pattern is a tile."""
    words = view[:view.numel() // 8 * 8].view(torch.int64)
    torch.randint(-2 ** 63, 2 ** 63 - 1, words.shape, generator=generator, device="cuda", out=words)


def exl3_scales(view, inputs, outputs, generator):
    """suh = +-1, svh = +-U(0.5, 1.5) / 64, fp16, behind a matrix's codes."""
    signs = torch.randint(0, 2, (inputs + outputs,), generator=generator, device="cuda") * 2 - 1
    magnitudes = torch.ones(inputs + outputs, device="cuda")
    magnitudes[inputs:] = (torch.rand(outputs, generator=generator, device="cuda") + 0.5) / 64
    view.copy_((signs * magnitudes).half().view(torch.uint8))


def exl3_bytes(inputs, outputs, stored_width):
    return inputs * outputs // 16 * (5 if stored_width == 40 else 2 * stored_width) + 2 * (inputs + outputs)


def fill_e4m3(view, generator):
    """E4M3 codes of normal weights whose block's largest lies at the top of the range."""
    for part in view.split(1 << 26):
        part.copy_((normals(generator, part.numel()) * 100).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))


def scaled_matrices(view, weights, generator):
    """Rows of `view`: stored FP4 / FP8 matrices of standard deviation about 0.02, codes and then scales (independent
    values, so that any lane order of them is as good as another)."""
    count, per = view.shape
    codes = {"e2m1": per * 16 // 17, "e4m3": per * 1024 // 1025, "e4m3_block128": per * 4096 // 4097}[weights]
    words = view.reshape(-1)
    if weights == "e2m1":
        exl3_codes(words, generator)
        view[:, codes:] = 120 + torch.randint(0, 2, (count, per - codes), generator=generator, device="cuda", dtype=torch.uint8)
        return
    fill_e4m3(words, generator)
    if weights == "e4m3":
        view[:, codes:] = 114 + torch.randint(0, 2, (count, per - codes), generator=generator, device="cuda", dtype=torch.uint8)
    else:
        scales = (0.9 + 0.2 * torch.rand(count, (per - codes) // 4, generator=generator, device="cuda")) * 2e-4
        view[:, codes:] = scales.view(torch.uint8)


class Layer:
    """What both layers below share: the router, its rows and the step's ranges, made on the card."""

    def common(self, case, generator):
        space = arena()
        self.card = card = space.card
        self.H, self.I, self.E, self.P, self.rows = (case[name] for name in ("hidden", "inner", "experts", "picks", "rows"))
        rows, self.pairs, self.limit, self.route_scale = self.rows, self.rows * self.P, 10.0, 1.5
        self.affinity_kind = amd.AFFINITY_SIGMOID if case["affinity"] == "sigmoid" else amd.AFFINITY_SQRT_SOFTPLUS
        self.step_offset = card.place(amd.step_block(rows))
        self.x_offset = card.reserve(rows * self.H * 2)
        self.scores_offset, self.affinities_offset = card.reserve(rows * self.E * 4), card.reserve(rows * self.E * 4)
        self.bias_offset, self.router_offset = card.reserve(self.E * 4), card.reserve(self.E * self.H * 2)
        self.jobs_offset, self.offsets_offset = card.reserve(self.pairs * 96), card.place(self.expert_offsets)
        self.x = space.view(self.x_offset, torch.bfloat16, rows, self.H)
        self.x.copy_(normals(generator, rows, self.H))
        router = space.view(self.router_offset, torch.bfloat16, self.E, self.H)
        router.copy_(normals(generator, self.E, self.H) * 0.02)
        space.view(self.bias_offset, torch.float32, self.E).copy_(self.bias(case, router, generator))
        self.affinities = space.view(self.affinities_offset, torch.float32, rows, self.E)
        self.router_kernels = amd.RouterKernels()
        amd.check(card.lib.router_kernels_prepare(amd.backend_table(), card.handle, C.byref(self.router_kernels)), "router_kernels_prepare")

    def bias(self, case, router, generator):
        """Zero; or the bias under which the rows' picks follow the skewed loads."""
        bias = torch.zeros(self.E, device="cuda")
        if case["skew"] == 0.0:
            return bias
        scores = self.x.float() @ router.float().t()
        affinities = scores.sigmoid() if case["affinity"] == "sigmoid" else torch.nn.functional.softplus(scores).sqrt()
        loads = torch.from_numpy(expert_loads(case)).float().cuda() * self.rows
        wanted = loads[torch.randperm(self.E, generator=generator, device="cuda")]
        bias = 0.05 * torch.log(wanted / wanted.max())
        for _ in range(120):
            picked = torch.topk(affinities + bias, self.P, dim=1).indices.reshape(-1)
            realised = torch.bincount(picked, minlength=self.E).float()
            bias += 0.02 * torch.log(wanted.clamp(min=0.5) / realised.clamp(min=0.5))
        return bias - bias.max()

    def routing(self):
        """(the wide select or None, the launches of the router)."""
        if self.rows <= amd.LINEAR_MAXIMUM_ROWS:
            return None, [self.projection_launch()[0], self.select_launch(0)[0]]
        wide = self.wide_router()
        return wide, [self.projection_launch()[0]] + list(wide.launches(small=self.rows <= 64))

    def outputs(self, wide, rows_out):
        out = {"rows": rows_out, "affinities": self.affinities}
        if wide is not None:
            out["experts"] = arena().view(wide.ranges["picks"].byte_offset, torch.int32, self.rows, self.P, 2)[..., 0]
        return out


class Exl3Experts(Layer, amd.Exl3Layer):
    def __init__(self, case, generator):
        space, card = arena(), arena().card
        experts, hidden, inner = case["experts"], case["hidden"], case["inner"]
        choices = WIDTH_CHOICES[case["widths"]]
        drawn = torch.multinomial(torch.tensor([p for _, p in choices], device="cuda"), experts * 3, replacement=True, generator=generator).cpu().numpy()
        self.widths = np.array([w for w, _ in choices], dtype=np.uint32)[drawn].reshape(experts, 3)
        self.uniform_width = int(self.widths[0, 0]) if len(choices) == 1 else 0
        self.packed_widths = (self.widths[:, 0] | (self.widths[:, 1] << 8) | (self.widths[:, 2] << 16)).astype(np.uint32)
        sizes = np.array([[exl3_bytes(hidden, inner, int(w)) for w in trio] for trio in self.widths], dtype=np.uint64)
        strides = (sizes.reshape(-1) + np.uint64(63)) // np.uint64(64) * np.uint64(64)
        self.weights_bytes = int(strides.sum()) + 64
        self.weights_offset = card.reserve(self.weights_bytes, 256)
        starts = np.uint64(self.weights_offset) + np.concatenate([np.zeros(1, np.uint64), np.cumsum(strides)[:-1]])
        self.expert_offsets = np.ascontiguousarray(starts.reshape(experts, 3))
        exl3_codes(space.bytes[self.weights_offset:self.weights_offset + self.weights_bytes], generator)
        for index, (start, size) in enumerate(zip(starts.tolist(), sizes.reshape(-1).tolist())):
            inputs, outputs = (hidden, inner) if index % 3 < 2 else (inner, hidden)
            exl3_scales(space.bytes[start + size - 2 * (inputs + outputs):start + size], inputs, outputs, generator)
        self.common(case, generator)
        self.kernels = self.router_kernels
        self.widths_offset = card.place(self.packed_widths) if self.uniform_width == 0 else 0
        self.out_offset = card.reserve(self.rows * hidden * 4)
        if self.rows <= 64:
            self.workspace_offset = card.reserve(amd.exl3_tc_workspace_bytes(self.pairs, hidden, inner))
        self.tcp_workspace_offset = None

    def step(self):
        wide, launches = self.routing()
        if self.rows > 64:  # the prefill form sorts the picks itself
            launches = launches[:2] + list(self.tcp_launches(wide.ranges["picks"].byte_offset))
        elif wide is None:
            launches += list(self.tc_launches())
        else:
            record, fused = self.tc_record(), amd.launches_of(amd.EXL3_TC_LAUNCHES)
            record.jobs_offset, record.job_capacity = wide.ranges["jobs"].byte_offset, wide.job_count
            amd.check(self.card.lib.exl3_tc_prepare(C.byref(record), self.card.arena_bytes, amd.backend_table(), self.card.handle, fused), "exl3_tc_prepare")
            launches += list(fused)
        return launches, self.outputs(wide, arena().view(self.out_offset, torch.float32, self.rows, self.H))


class ScaledExperts(Layer, amd.Fp4Layer):
    def __init__(self, case, generator):
        space, card = arena(), arena().card
        experts, hidden, inner, rows = case["experts"], case["hidden"], case["inner"], case["rows"]
        self.weight_format, self.native = FORMATS[case["weights"], case["gfx950_order"]], case["gfx950_order"]
        self.bits, self.block128 = 4 if case["weights"] == "e2m1" else 8, case["weights"] == "e4m3_block128"
        self.gate_up_slices, self.down_slices = 4, 2
        size = int(expert_matrix_bytes(case))
        stride = (size + 63) // 64 * 64
        self.weights_bytes = 3 * experts * stride
        self.weights_offset = card.reserve(self.weights_bytes, 256)
        self.expert_offsets = (np.uint64(self.weights_offset) + np.arange(3 * experts, dtype=np.uint64) * np.uint64(stride)).reshape(experts, 3)
        matrices = space.view(self.weights_offset, torch.uint8, 3 * experts, stride)
        if stride == size:
            scaled_matrices(matrices, case["weights"], generator)
        else:
            dense = torch.empty(3 * experts, size, dtype=torch.uint8, device="cuda")
            scaled_matrices(dense, case["weights"], generator)
            matrices[:, :size] = dense
        self.common(case, generator)
        pairs = self.pairs
        sizes = {"codes": rows * hidden, "exponents": rows * hidden // 32, "operands": rows * hidden * 2, "hidden": pairs * inner * 2,
                 "hidden_codes": pairs * inner, "hidden_exponents": pairs * inner // 32, "hidden_operands": pairs * inner * 2,
                 "pair_output": pairs * hidden * 2, "row_output": rows * hidden * 4}
        self.ranges = {name: amd.Range(card.reserve(bytes_), bytes_) for name, bytes_ in sizes.items()}
        self.kernels = amd.LinearKernels()
        amd.check(card.lib.linear_kernels_prepare(amd.backend_table(), card.handle, amd.ARITHMETIC_CLASS_GFX950, C.byref(self.kernels)), "linear_kernels_prepare")

    def expert_step(self):
        """(the wide select or None, the router's launches, the quantizer's and the experts')."""
        wide, routing = self.routing()
        if self.rows > 64:  # the wide products read tiles and sorted pairs: no job table
            return wide, routing[:4], [self.quantize_launch()[0]], list(self.wide_expert_launches(wide))
        return wide, routing, [self.quantize_launch()[0]], list(self.expert_launches(wide))

    def step(self):
        wide, routing, quantizer, experts = self.expert_step()
        return routing + quantizer + experts, self.outputs(wide, arena().view(self.ranges["row_output"].byte_offset, torch.float32, self.rows, self.H))


def site_step(layer, generator):
    """The layer's FFN site. Its post is close to zero (base -12), so that the streams a pass leaves behind, mixed among
    themselves, are as good an input for the next pass as the first ones."""
    space, rows, hidden, inner = arena(), layer.rows, layer.H, layer.I
    matrices = torch.empty(3, hidden * inner * 1025 // 1024, dtype=torch.uint8, device="cuda")
    scaled_matrices(matrices, "e4m3", generator)
    many = rows > 64
    shared = amd.SharedExpert(layer, list(matrices.cpu().numpy()), gate_up_slices=1 if many else 4, down_slices=1 if many else 2,
                              wide_form=amd.LINEAR_INTERLEAVED_CHUNK_BLOCKS if many else amd.LINEAR_WIDE_GROUP_BLOCKS)
    base = normals(generator, 24).cpu().numpy() * 0.5
    base[4:8] = -12.0
    front = amd.SiteFront(layer.card, rows, hidden, (normals(generator, 24, 4 * hidden) * 0.02).cpu().numpy(), [0.1, 0.1, 0.1], base,
                          np.full(hidden, 0x3F80, dtype=np.uint16), hidden_range=amd.Range(layer.x_offset, rows * hidden * 2))
    for name in ("streams", "post", "comb"):  # the join reads the post and comb the finish writes
        front.ranges[name] = shared.ranges[name]
    streams = space.view(shared.ranges["streams"].byte_offset, torch.bfloat16, rows, 4, hidden)
    streams.copy_(normals(generator, rows, 4, hidden))
    space.view(front.ranges["carried_pre"].byte_offset, torch.float32, rows * 4).fill_(0.25)
    wide, routing, quantizer, experts = layer.expert_step()
    if rows <= amd.LINEAR_MAXIMUM_ROWS:
        front.front_description(layer=layer)  # reserves the front's scratch
        for name in ("codes", "exponents", "operands"):
            front.ranges[name] = layer.ranges[name]
        launches = [front.front_launch(layer=layer)[0]] + experts[:-1] + list(shared.launches())[:3] + [shared.shared_join_launch()[0]]
    else:
        launches = [front.mix_project_launch()[0], front.site_launches()[0]] + routing + quantizer + experts[:-1] + list(shared.launches()) + \
            [shared.join_launch()[0]]
    outputs = layer.outputs(wide, space.view(shared.ranges["row_sums"].byte_offset, torch.float32, rows, hidden))
    outputs.update(streams=streams, post=space.view(shared.ranges["post"].byte_offset, torch.float32, rows, 4),
                   comb=space.view(shared.ranges["comb"].byte_offset, torch.float32, rows, 4, 4), hidden=layer.x)
    return launches, outputs, (shared, front)


def linear_step(case, generator):
    """One EXL3 matrix by `rows` vectors: the chain's input launch for one projection, its down product and its finish."""
    space, card = arena(), arena().card
    size, rows, width = case["size"], case["rows"], WIDTH_CHOICES[case["widths"]][0][0]
    stored = exl3_bytes(size, size, width)
    at = card.reserve(stored, 256)
    exl3_codes(space.bytes[at:at + stored], generator)
    exl3_scales(space.bytes[at + stored - 4 * size:at + stored], size, size, generator)
    jobs = np.zeros(1, dtype=amd.JOB_DTYPE)
    jobs[0]["gate_offset"] = jobs[0]["up_offset"] = jobs[0]["down_offset"] = at
    jobs[0]["row_count"], jobs[0]["pair_index"][:rows], jobs[0]["route_weight"][:rows] = rows, np.arange(rows), 1.0
    record = amd.Exl3ExpertRecord()
    record.jobs_offset = card.place(jobs.view(np.uint8))
    record.input_offset, record.operands_offset, record.hidden_offset = card.reserve(rows * size * 2), card.reserve(rows * size * 4), card.reserve(rows * size * 2)
    record.products_offset = record.output_offset = card.reserve(rows * size * 8)
    record.input_size = record.inner_size = size
    record.pair_count, record.pairs_per_row, record.job_count = rows, 1, 1
    record.bits_per_weight, record.activation_limit = width, 10.0
    space.view(record.input_offset, torch.bfloat16, rows, size).copy_(normals(generator, rows, size))
    chain = amd.launches_of(amd.EXL3_EXPERT_LAUNCHES)
    amd.check(card.lib.exl3_experts_prepare(C.byref(record), card.arena_bytes, amd.backend_table(), card.handle, amd.ARITHMETIC_CLASS_GFX950, chain),
              "exl3_experts_prepare")
    chain[0].grid[2] = 1  # one projection's operands
    return [chain[0], chain[3], chain[4]], {"rows": space.view(record.output_offset, torch.float32, rows, size)}


def prepare(case, seed):
    """The step of `case` laid out in a free slot of the arena; the slot is free again when the state is dropped."""
    space = arena()
    slot = space.take()
    try:
        generator = torch.Generator(device="cuda").manual_seed(seed)
        if case["kind"] == "linear":
            launches, outputs = linear_step(case, generator)
            keep = ()
        else:
            layer = (Exl3Experts if case["weights"] == "exl3" else ScaledExperts)(case, generator)
            launches, outputs, *keep = site_step(layer, generator) if case["kind"] == "site" else layer.step()
        if space.card.cursor > (slot + 1) * SLOT_BYTES:
            raise ValueError("the case does not fit a slot of the arena")
        state = State(launches, outputs, keep)
        torch.cuda.synchronize()  # torch filled the arena on a stream of its own
    except BaseException:
        space.free.append(slot)
        raise
    weakref.finalize(state, space.free.append, slot)
    return state


def run(state):
    arena().card.run(state.step, wait=False)
    return state.outputs
