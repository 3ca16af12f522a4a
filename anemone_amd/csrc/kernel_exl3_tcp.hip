/*
 * kernel_exl3_tcp.hip -- the routed experts of one EXL3 layer for a prefill-sized call on gfx950: the pairs sorted by
 * expert and the expert computation as a grouped GEMM on the matrix cores with the trellis decode fused into the
 * weight tile loads. The counterpart of the reference's prefill form (source/kernel_exl3_tcp.cuh:7-15,
 * include/anemone/exl3_tc_records.h:205-304): same record, same order of the work (route, operands, gate/up GEMM,
 * activation and down operands, down GEMM, combine in route order).
 *
 * Arithmetic: the chain's (kernel_exl3.hip): fp16 operands from a float32 Hadamard transform, exactly decoded fp16
 * weights, float32 MFMA sums over increasing k (one chain an output: the GEMM is not cut along k), SwiGLU in float32,
 * a row's weighted pair outputs added in slot order. A pair's result does not depend on the other pairs of the call; the
 * two forms of the GEMM, which the call's sizes choose between (exl3_tcp_is_thin), add in an order of their own each.
 *
 * The GEMM block: 256 outputs (four wavefronts of four 16 x 16 tiles) by one chunk of at most EXL3_TCP_CHUNK_PAIRS (160)
 * pairs of one expert. A K step is 64 inputs: the chunk's operand columns (160 x 64 fp16, 20 KB) go from memory straight
 * into LDS once a block and serve all four wavefronts; each wavefront's codes go from memory into the registers of the
 * lanes that decode them, a decoded operand of eight weights a lane feeds up to five matrix instructions of 32 x 32
 * outputs, one for every 32 columns. Decoding is the vector unit's work (about 3.7 instructions a weight) and the
 * products the matrix unit's (32 cycles an instruction).
 */
#include <type_traits>

#include "exl3_stream_device.cuh"
#include "kernel_registry.h"
#include "sort_device.cuh"

#define TCP_SORT_THREADS 512u
#define TCP_GEMM_WAVES 4u
#define TCP_GEMM_THREADS (TCP_GEMM_WAVES * WAVE)
#define TCP_WAVE_PAIRS 2u  /* pairs of adjacent output tiles of a wavefront: 64 outputs */
#define TCP_COLUMN_BLOCKS (EXL3_TCP_CHUNK_PAIRS / 16u) /* of sixteen columns: two a block of the matrix instruction's 32 */
#define TCP_STEP_INPUTS 64u
#define TCP_DIES 8u         /* the card's dies (XCDs), each with a level-2 cache of its own: blocks are dealt to them in turn */
#define TCP_BATCH 4u        /* columns, or slots of a row, the element-wise launches take at a time */
/* values of one of the two operand arrays from which on they are written past the caches (nontemporal): two arrays of 192 MiB and
 * more leave the 256 MB behind the dies before the products read them, whichever way they are written. 256 experts, 8 picks, hidden
 * 4096, as before -> nontemporal: 2048 rows 59.0 -> 61.1 us, 2560 73.9 -> 75.4, 3072 (the line) 89.4 -> 88.6, 4096 128.6 -> 112.6,
 * 6144 208 -> 166; the products behind them take the same */
#define TCP_STREAMED_OPERANDS (96ull << 20)
#define TCP_THIN_PLACES 4u  /* places of a block of a thin call's element-wise launches: one a wavefront */
#define TCP_WAVE_BLOCKS 4u  /* blocks of 128 channels a wavefront of an element-wise launch takes: a row of sixteen lanes each */

struct tcp_shape {
    uint32_t hidden, intermediate, picks, pairs, experts;
    struct exl3_tcp_layout layout;
};

__device__ static __forceinline__ tcp_shape tcp_shape_of(const struct exl3_tcp_record &record)
{
    tcp_shape shape;
    shape.hidden = record.hidden;
    shape.intermediate = record.intermediate;
    shape.picks = record.pairs_per_row;
    shape.pairs = record.row_count * record.pairs_per_row;
    shape.experts = record.expert_count;
    shape.layout = exl3_tcp_layout_of(record.row_count, record.pairs_per_row, record.expert_count, record.hidden, record.intermediate);
    return shape;
}

__device__ static __forceinline__ uint32_t tcp_bits_x2(const struct exl3_tcp_record &record, const unsigned char *arena,
                                                       uint32_t expert, uint32_t matrix)
{
    if (record.widths_offset == 0u) {
        return record.bits_x2;
    }
    return exl3_bits_x2(exl3_width_of(((const uint32_t *)(arena + record.widths_offset))[expert], matrix));
}

__device__ static __forceinline__ uint64_t tcp_matrix_of(const struct exl3_tcp_record &record, const unsigned char *arena,
                                                         uint32_t expert, uint32_t matrix)
{
    return ((const uint64_t *)(arena + record.expert_offsets_offset))[(uint64_t)expert * MODEL_EXPERT_MATRICES + matrix];
}

/* launch 0: grid (ceil(row_count / ROUTER_SORT_ROWS)): counts [block][experts] */
extern "C" __global__ void __launch_bounds__(TCP_SORT_THREADS) exl3_tcp_count(struct exl3_tcp_record record, unsigned char *arena)
{
    __shared__ __attribute__((aligned(16))) uint32_t block_experts[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    const tcp_shape shape = tcp_shape_of(record);
    const uint32_t pairs = sort_block_picks((const struct router_pick *)(arena + record.picks_offset), shape.picks, blockIdx.x,
                                            record.row_count, block_experts);
    __syncthreads();
    __shared__ uint32_t histogram[ROUTER_MOST_EXPERTS];
    sort_count_picks(block_experts, pairs, shape.experts, histogram);
    uint32_t *counts = (uint32_t *)(arena + record.workspace_offset + shape.layout.counts) + (uint64_t)blockIdx.x * shape.experts;
    for (uint32_t expert = threadIdx.x; expert < shape.experts; expert += TCP_SORT_THREADS) {
        counts[expert] = histogram[expert];
    }
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_count, exl3_tcp_record);

/* launch 1: the same grid: the block's pairs placed (sorted [place] and place_of [pair]); block 0 also the runs, the
 * chunks and their number */
extern "C" __global__ void __launch_bounds__(TCP_SORT_THREADS) exl3_tcp_place(struct exl3_tcp_record record, unsigned char *arena)
{
    __shared__ __attribute__((aligned(16))) uint32_t block_experts[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    __shared__ uint32_t block_places[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    __shared__ uint32_t totals[ROUTER_MOST_EXPERTS], starts[ROUTER_MOST_EXPERTS], before[ROUTER_MOST_EXPERTS];
    __shared__ uint32_t chunk_starts[ROUTER_MOST_EXPERTS + 1u], scratch[SORT_MOST_WAVES];
    __shared__ uint32_t first_places[ROUTER_MOST_EXPERTS], cursors[SORT_MOST_WAVES * ROUTER_MOST_EXPERTS];
    const tcp_shape shape = tcp_shape_of(record);
    const uint32_t experts = shape.experts;
    const uint32_t blocks = (record.row_count + ROUTER_SORT_ROWS - 1u) / ROUTER_SORT_ROWS;
    unsigned char *workspace = arena + record.workspace_offset;
    const uint32_t pairs = sort_block_picks((const struct router_pick *)(arena + record.picks_offset), shape.picks, blockIdx.x,
                                            record.row_count, block_experts);
    const uint32_t *counts = (const uint32_t *)(workspace + shape.layout.counts);
    for (uint32_t expert = threadIdx.x; expert < experts; expert += TCP_SORT_THREADS) {
        uint32_t total = 0, lower = 0;
#pragma unroll 8
        for (uint32_t block = 0; block < blocks; block++) {
            const uint32_t count = counts[(uint64_t)block * experts + expert];
            total += count;
            lower += block < blockIdx.x ? count : 0u;
        }
        totals[expert] = total;
        starts[expert] = total;
        before[expert] = lower;
        chunk_starts[expert] = (total + EXL3_TCP_CHUNK_PAIRS - 1u) / EXL3_TCP_CHUNK_PAIRS;
    }
    __syncthreads();
    (void)block_exclusive_scan(starts, experts, scratch);
    uint32_t *sorted = (uint32_t *)(workspace + shape.layout.sorted), *place_of = (uint32_t *)(workspace + shape.layout.place_of);
    const uint32_t first_pair = blockIdx.x * ROUTER_SORT_ROWS * shape.picks;
    /* every pick's place into LDS; the two tables are written behind it, a thread a pick */
    for (uint32_t expert = threadIdx.x; expert < experts; expert += TCP_SORT_THREADS) {
        first_places[expert] = starts[expert] + before[expert];
    }
    __syncthreads();
    sort_place_picks(block_experts, pairs, experts, first_places, cursors, block_places);
    for (uint32_t index = threadIdx.x; index < pairs; index += TCP_SORT_THREADS) {
        const uint32_t place = block_places[index];
        sorted[place] = first_pair + index;
        place_of[first_pair + index] = place;
    }
    if (blockIdx.x != 0u) {
        return;
    }
    struct wide_run *runs = (struct wide_run *)(workspace + shape.layout.runs);
    for (uint32_t expert = threadIdx.x; expert < experts; expert += TCP_SORT_THREADS) {
        runs[expert] = (struct wide_run){starts[expert], totals[expert]};
    }
    const uint32_t used = block_exclusive_scan(chunk_starts, experts, scratch);
    if (threadIdx.x == 0u) {
        chunk_starts[experts] = used;
        uint32_t *header = (uint32_t *)(workspace + shape.layout.header);
        header[0] = used;
        header[1] = header[2] = header[3] = 0u;
    }
    __syncthreads();
    struct exl3_tcp_chunk *chunks = (struct exl3_tcp_chunk *)(workspace + shape.layout.chunks);
    for (uint32_t chunk = threadIdx.x; chunk < shape.layout.chunk_capacity; chunk += TCP_SORT_THREADS) {
        struct exl3_tcp_chunk value = {0, 0, 0, 0};
        if (chunk < used) {
            uint32_t low = 0, high = experts; /* the expert whose chunks hold this one */
            while (high - low > 1u) {
                const uint32_t middle = (low + high) / 2u;
                if (chunk_starts[middle] <= chunk) {
                    low = middle;
                } else {
                    high = middle;
                }
            }
            const uint32_t taken = (chunk - chunk_starts[low]) * EXL3_TCP_CHUNK_PAIRS, left = totals[low] - taken;
            value.expert = low;
            value.first_pair = starts[low] + taken;
            value.pair_count = left < EXL3_TCP_CHUNK_PAIRS ? left : EXL3_TCP_CHUNK_PAIRS;
        }
        chunks[chunk] = value;
    }
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_place, exl3_tcp_record);

__device__ static __forceinline__ struct exl3_tcp_chunk tcp_chunk_of(const tcp_shape &shape, const unsigned char *workspace, uint32_t index)
{
    const uint32_t used = ((const uint32_t *)(workspace + shape.layout.header))[0];
    struct exl3_tcp_chunk chunk = {0, 0, 0, 0};
    if (index < used) {
        chunk = ((const struct exl3_tcp_chunk *)(workspace + shape.layout.chunks))[index];
    }
    return chunk;
}

/* The element-wise launches take a block of 128 values in a row of sixteen lanes, eight consecutive values a lane in
 * row_hadamard128's order (one 16-byte load of bfloat16 or fp16, two of float32): a wavefront is four adjacent blocks of one vector, 1 KB of
 * bfloat16 a load. this lane's block of 128 channels and its first channel, or false past the width */
__device__ static __forceinline__ bool tcp_lane_channels(uint32_t width, uint32_t &channel)
{
    const uint32_t lane = threadIdx.x;
    channel = (blockIdx.x * TCP_WAVE_BLOCKS + lane / 16u) * EXL3_TRANSFORM + 8u * row_group_of(lane);
    return channel < width;
}

/* launch 2: grid (ceil(hidden / 512), chunk capacity, EXL3_TCP_COLUMN_PARTS), block 64: the gate and the up operands of
 * a part of a chunk's pairs, by place: fp16(H128(x suh) / sqrt(128)); a row is read once for both */
extern "C" __global__ void exl3_tcp_operands(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    unsigned char *workspace = arena + record.workspace_offset;
    const struct exl3_tcp_chunk chunk = tcp_chunk_of(shape, workspace, blockIdx.y);
    const uint32_t first_column = blockIdx.z * EXL3_TCP_PART_COLUMNS;
    uint32_t channel;
    if (first_column >= chunk.pair_count || !tcp_lane_channels(shape.hidden, channel)) {
        return;
    }
    const uint32_t lane = threadIdx.x;
    const uint32_t last_column = first_column + EXL3_TCP_PART_COLUMNS < chunk.pair_count ? first_column + EXL3_TCP_PART_COLUMNS : chunk.pair_count;
    float scale[2][8];
#pragma unroll
    for (uint32_t projection = 0; projection < 2u; projection++) {
        const uint64_t matrix = tcp_matrix_of(record, arena, chunk.expert, projection);
        const uint16_t *suh = (const uint16_t *)(arena + matrix + exl3_code_bytes(shape.hidden, shape.intermediate,
                                                                                   tcp_bits_x2(record, arena, chunk.expert, projection)));
        unpack_half8(*(const uint4_t *)(suh + channel), scale[projection]);
    }
    const uint16_t *rows = (const uint16_t *)(arena + record.hidden_offset);
    const uint32_t *sorted = (const uint32_t *)(workspace + shape.layout.sorted);
    uint16_t *operands = (uint16_t *)(workspace + shape.layout.operands);
    const auto write = [&](auto streamed) {
        /* TCP_BATCH columns at a time: their loads are asked for together, so that one column's latency hides behind
         * the others' (a column past the part's last repeats it and is not stored) */
        for (uint32_t first = first_column; first < last_column; first += TCP_BATCH) {
            uint4_t loads[TCP_BATCH];
            uint32_t place[TCP_BATCH];
#pragma unroll
            for (uint32_t i = 0; i < TCP_BATCH; i++) {
                const uint32_t column = first + i < last_column ? first + i : last_column - 1u;
                place[i] = chunk.first_pair + column;
                const uint64_t row = sorted[place[i]] / shape.picks;
                loads[i] = *(const uint4_t *)(rows + row * shape.hidden + channel);
            }
#pragma unroll
            for (uint32_t i = 0; i < TCP_BATCH; i++) {
                const bool kept = first + i < last_column;
#pragma unroll
                for (uint32_t projection = 0; projection < 2u; projection++) {
                    const uint4_t operand = row_operand(loads[i], scale[projection], lane);
                    uint4_t *out = (uint4_t *)(operands + ((uint64_t)projection * shape.pairs + place[i]) * shape.hidden + channel);
                    if (kept && streamed.value) {
                        __builtin_nontemporal_store(operand, out);
                    } else if (kept) {
                        *out = operand;
                    }
                }
            }
        }
    };
    if (shape.pairs * (uint64_t)shape.hidden >= TCP_STREAMED_OPERANDS) { /* the same in every block */
        write(std::true_type{});
    } else {
        write(std::false_type{});
    }
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_operands, exl3_tcp_record);

/* The element-wise launches of a thin call (exl3_tcp_is_thin): grid (ceil(width / 512), ceil(pairs / 4)), block 256: a
 * wavefront a place. By chunks, as above, a handful of pairs an expert is a wavefront or two a SIMD that walk their columns
 * one batch behind the other, among ten times as many blocks that find none; by places every pair is a wavefront of its
 * own and reads its expert's scales itself. The same operands. 203 rows of 256 experts,
 * 8 picks, hidden 4096, intermediate 2048: operands 25 -> 14 us, activate 35 -> 17, the call 881 -> 851.
 * false past the pairs or the width */
__device__ static __forceinline__ bool tcp_thin_place(const tcp_shape &shape, const struct exl3_tcp_record &record, const unsigned char *arena,
                                                      uint32_t width, uint32_t &place, uint32_t &pair, uint32_t &expert, uint32_t &channel, uint32_t &lane)
{
    lane = threadIdx.x % WAVE;
    place = blockIdx.y * TCP_THIN_PLACES + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    channel = (blockIdx.x * TCP_WAVE_BLOCKS + lane / 16u) * EXL3_TRANSFORM + 8u * row_group_of(lane);
    if (place >= shape.pairs || channel >= width) {
        return false;
    }
    pair = ((const uint32_t *)(arena + record.workspace_offset + shape.layout.sorted))[place];
    expert = ((const struct router_pick *)(arena + record.picks_offset))[pair].expert;
    return true;
}

extern "C" __global__ void __launch_bounds__(TCP_THIN_PLACES * WAVE) exl3_tcp_operands_thin(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    uint32_t place, pair, expert, channel, lane;
    if (!tcp_thin_place(shape, record, arena, shape.hidden, place, pair, expert, channel, lane)) {
        return;
    }
    const uint4_t load = *(const uint4_t *)((const uint16_t *)(arena + record.hidden_offset) + (uint64_t)(pair / shape.picks) * shape.hidden + channel);
    uint16_t *operands = (uint16_t *)(arena + record.workspace_offset + shape.layout.operands);
    uint4_t scales[2];
#pragma unroll
    for (uint32_t projection = 0; projection < 2u; projection++) {
        scales[projection] = *(const uint4_t *)((const uint16_t *)(arena + tcp_matrix_of(record, arena, expert, projection) +
                                                                   exl3_code_bytes(shape.hidden, shape.intermediate, tcp_bits_x2(record, arena, expert, projection))) + channel);
    }
#pragma unroll
    for (uint32_t projection = 0; projection < 2u; projection++) {
        float scale[8];
        unpack_half8(scales[projection], scale);
        *(uint4_t *)(operands + ((uint64_t)projection * shape.pairs + place) * shape.hidden + channel) = row_operand(load, scale, lane);
    }
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_operands_thin, exl3_tcp_record);

/*
 * The GEMM block: 256 outputs by one chunk of at most EXL3_TCP_CHUNK_PAIRS pairs of one expert, four wavefronts of 64
 * outputs each (two pairs of adjacent output tiles). A K step is 64 inputs (four K tiles).
 *
 * Weights: the codes go from memory straight into the registers of the lanes that decode them, by the stream product's
 * decode (exl3_stream_device.cuh) under the assignment of chunks to lanes that tcp_wave_gemm states; a decoded operand
 * of eight weights a lane (output half h, input half v) feeds one matrix instruction a block of 32 columns.
 * Operands: a stage holds the step's 64 inputs of every column of the chunk, 128 bytes a column, its eight 16-byte pieces
 * at the slots piece ^ ((column / 2) % 8) so that sixteen lanes of one read (sixteen columns, one piece) meet sixteen
 * different bank groups. Each wavefront brings a share of the stage by LDS DMA a step ahead, one barrier a step; the
 * reader of column block j takes piece 4 s + 2 (lane / 32) + v of column 32 j + lane % 32 as the instruction's B operand.
 *
 * What bounds it: the vector unit's decoding and the matrix unit, at the clock the card holds under both (1.8 GHz), and
 * the cycles in which a wavefront has neither to issue. The step's one barrier therefore stands ahead of its last two
 * operands' matrix instructions (all of the step's columns are in registers by then): the next step's first columns are
 * read and its first operand is decoded in their shadow, where both stood bare behind a barrier at the step's end.
 * 4096 rows of 4096 x 2048 x 256 experts, Zipf(1.1) loads, builds in turns on one card: gate/up 1525 -> 1475 us, down
 * 855 -> 815. The addresses are kept as a base common to the wavefront and one offset a lane, which makes the registers
 * for that (24 spilled with an address a lane, 2 now, neither in the loop over the steps). A wavefront's priority at the
 * issue rises through its step: without it the two wavefronts of a SIMD run into the same phases (gate/up 1460 -> 1420 us,
 * down 815 -> 800; 600 rows of even loads 725 -> 672 and 377 -> 356; raised at half the step alone: 1420, 783, 703, 370;
 * falling instead: no shorter).
 */
/* 16 bytes a lane from memory straight into LDS (lane L lands at lds_base + 16 L), no register in between. Written as
 * assembly: the compiler keeps no book on it, so the wait that ends a step (every load of the wavefront, then the block's
 * barrier) is written out below. */
__device__ static __forceinline__ void tcp_load_to_lds(const unsigned char *base, uint32_t lane_offset, uint32_t lds_base)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_offset), "s"(base), "s"(lds_base) : "memory", "m0");
}

#define TCP_STAGE_COLUMN_BYTES (TCP_STEP_INPUTS * 2u)
#define TCP_STAGE_BYTES (EXL3_TCP_CHUNK_PAIRS * TCP_STAGE_COLUMN_BYTES)

/* A wavefront's product of 64 outputs by the chunk's columns on the matrix instruction of 32 x 32 outputs
 * (v_mfma_f32_32x32x16_f16: A lane l row l % 32, k = 8 (l / 32) + e; B lane l column l % 32, the same k; D lane l
 * column l % 32, register r row r % 4 + 8 (r / 4) + 4 (l / 32); measured on the card). Lane 16 g + i decodes chunk i % 8 of output tile i / 8 + 2 (g % 2) of the
 * wavefront's four and of K tile 2 s + g / 2 of the step's four (s = 0, 1: the step's halves), so the 32 rows of an
 * instruction (h, v) are output (i % 8) + 8 h of those four tiles and its sixteen k are inputs 8 v .. + 7 of the two K
 * tiles of half s: what a lane decodes, and how, is the stream product's; a decoded operand feeds LIVE instructions of
 * twice the work each. LIVE: blocks of 32 columns. */
typedef float float16v_t __attribute__((ext_vector_type(16)));

template <uint32_t bits_x2, uint32_t LIVE>
__device__ static __forceinline__ void
tcp_wave_gemm(const uint32_t *__restrict__ codes, uint32_t out_tiles, uint32_t strip_tile, uint32_t inputs,
                const half_t *__restrict__ columns, uint32_t column_count, uint32_t stages, uint32_t wave,
                uint32_t lane, bool strip_is_live, float16v_t (&accumulator)[2][LIVE])
{
    typedef exl3_chunk<bits_x2> C;
    constexpr uint32_t live_groups = 4u * LIVE; /* groups of eight columns that hold a pair */
    constexpr uint32_t wave_groups = (live_groups + TCP_GEMM_WAVES - 1u) / TCP_GEMM_WAVES;
    const uint32_t g = lane / 16u, i = lane % 16u, c = i % 8u, upper = lane / 32u, row = lane % 32u;
    const bool odd = (c & 1u) != 0u;
    uint32_t own, front;
    exl3_chunk_place<bits_x2>(c, own, front);
    const uint64_t step_stride = 16u * (uint64_t)out_tiles * C::tile_words, half_stride = 8u * (uint64_t)out_tiles * C::tile_words; /* bytes */
    /* a strip past the matrix reads the matrix's first strip (its sums are not stored): every wavefront runs the same loop */
    const unsigned char *tile = (const unsigned char *)(codes + (uint64_t)(strip_is_live ? strip_tile : 0u) * C::tile_words);
    const uint32_t lane_tile = ((g / 2u) * out_tiles + i / 8u + 2u * (g % 2u)) * C::tile_words;
    own = (own + lane_tile) * 4u;
    front = (front + lane_tile) * 4u;
    /* the stage's groups this wavefront brings: wave, wave + 4, ...: lane L column 8 G + L / 8, slot L % 8 */
    uint32_t operand_source[wave_groups];
#pragma unroll
    for (uint32_t part = 0; part < wave_groups; part++) {
        const uint32_t group = wave + TCP_GEMM_WAVES * part, column = 8u * group + lane / 8u;
        const uint32_t piece = (lane % 8u) ^ ((column / 2u) % 8u);
        operand_source[part] = (column < column_count ? column : 0u) * inputs * 2u + piece * 16u;
    }
    /* where this lane reads its B operand (half s, inputs v) of column block j: column 32 j + row, piece 4 s + 2 upper + v */
    const uint32_t read_at = stages + row * TCP_STAGE_COLUMN_BYTES + (((2u * upper) ^ ((row / 2u) % 8u)) * 16u);
#pragma unroll
    for (uint32_t h = 0; h < 2u; h++) {
#pragma unroll
        for (uint32_t j = 0; j < LIVE; j++) {
#pragma unroll
            for (uint32_t r = 0; r < 16u; r++) {
                accumulator[h][j][r] = 0.0f;
            }
        }
    }
    const uint32_t steps = inputs / TCP_STEP_INPUTS;
    exl3_chunk_words<bits_x2> held[2][2];
#pragma unroll
    for (uint32_t s = 0; s < 2u; s++) {
        exl3_chunk_load_at<bits_x2>(tile + s * half_stride, own, front, held[0][s]);
    }
#pragma unroll
    for (uint32_t part = 0; part < wave_groups; part++) {
        if (wave + TCP_GEMM_WAVES * part < live_groups) {
            tcp_load_to_lds((const unsigned char *)columns, operand_source[part], stages + (wave + TCP_GEMM_WAVES * part) * 1024u);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    /* A step is eight operands of eight weights a lane: k = 4 s + 2 v + h (the B operands of (s, v) serve both h and are
     * read a pair of operands ahead). An operand's LIVE matrix instructions are issued with the next operand's decoding
     * between them: the decoding runs in the products' shadow, across the steps as inside one. */
    half8_t operand_b[2][LIVE];
    uint32_t a[4], ahead[4]; /* the operand being multiplied, the one being decoded */
    auto read_operands = [&](uint32_t parity, uint32_t k) { /* those of operands k and k + 1 of a step, out of the stage of its parity */
        const uint32_t at = read_at ^ (64u * (k / 4u) + 16u * (k / 2u % 2u)); /* the piece's number lies in bits 4 to 6 */
#pragma unroll
        for (uint32_t j = 0; j < LIVE; j++) {
            operand_b[k / 2u % 2u][j] = __builtin_bit_cast(half8_t, *(const __attribute__((address_space(3))) uint4_t *)(uintptr_t)(at + parity * TCP_STAGE_BYTES + j * (32u * TCP_STAGE_COLUMN_BYTES)));
        }
    };
    auto decode_weight = [&](const exl3_chunk_words<bits_x2> (&now)[2], uint32_t k, uint32_t w, uint32_t (&into)[4]) {
        const uint32_t s = k / 4u, v = k / 2u % 2u, h = k % 2u, t = w / 2u, m = 8u * t + 4u * h + 2u * v + w % 2u;
        uint32_t funnel[C::words];
#pragma unroll
        for (uint32_t word = 0; word < C::words; word++) {
            funnel[word] = __builtin_amdgcn_alignbit(now[s].z[word], now[s].z[word + 1u], 16u);
        }
        const uint32_t product = exl3_chunk_state<bits_x2>(now[s].z, funnel, m) * EXL3_MUL1_MULTIPLIER;
        if (w % 2u == 0u) {
            into[t] = __builtin_amdgcn_sad_u8(product, 0u, (uint32_t)EXL3_MUL1_BASE * 0x10001u);
        } else {
            const uint32_t sums = __builtin_amdgcn_sad_hi_u8(product, 0u, into[t]);
            const half2_t scale = __builtin_bit_cast(half2_t, (uint32_t)EXL3_MUL1_SCALE * 0x10001u);
            const half2_t bias = __builtin_bit_cast(half2_t, (uint32_t)EXL3_MUL1_BIAS * 0x10001u);
            into[t] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2_t, sums), scale, bias));
        }
    };
    auto ask = [&](uint32_t step, exl3_chunk_words<bits_x2> (&next)[2]) { /* the codes and columns of `step` */
        tile += step_stride;
#pragma unroll
        for (uint32_t s = 0; s < 2u; s++) {
            exl3_chunk_load_at<bits_x2>(tile + s * half_stride, own, front, next[s]);
        }
#pragma unroll
        for (uint32_t part = 0; part < wave_groups; part++) {
            if (wave + TCP_GEMM_WAVES * part < live_groups) {
                tcp_load_to_lds((const unsigned char *)columns + (uint64_t)step * TCP_STAGE_COLUMN_BYTES, operand_source[part],
                                stages + (step % 2u) * TCP_STAGE_BYTES + (wave + TCP_GEMM_WAVES * part) * 1024u);
            }
        }
    };
#pragma unroll
    for (uint32_t s = 0; s < 2u; s++) {
        exl3_chunk_align<bits_x2>(held[0][s], odd);
    }
    read_operands(0u, 0u);
#pragma unroll
    for (uint32_t w = 0; w < 8u; w++) {
        decode_weight(held[0], 0u, w, a);
    }
    auto one_step = [&](uint32_t step, uint32_t parity, exl3_chunk_words<bits_x2> (&now)[2], exl3_chunk_words<bits_x2> (&next)[2]) {
        const bool more = step + 1u < steps; /* the same in every lane */
        if (more) {
            ask(step + 1u, next);
        }
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) {
            const uint32_t h = k % 2u;
            if (k % 2u == 0u && k + 2u < 8u) {
                read_operands(parity, k + 2u);
            }
            /* the further a wavefront is into its step, the more its instructions go first: the other block's wavefront on the SIMD
             * falls behind to where its decoding meets this one's products, and this one reaches its barrier */
            if (k == 0u) {
                __builtin_amdgcn_s_setprio(0);
            } else if (k == 2u) {
                __builtin_amdgcn_s_setprio(1);
            } else if (k == 4u) {
                __builtin_amdgcn_s_setprio(2);
            } else if (k == 6u) {
                __builtin_amdgcn_s_setprio(3);
            }
            if (k == 6u) {
                /* every load of this wavefront has landed (the next step's codes and its share of the next stage), and it
                 * has read this step's stage, which the step after the next takes */
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                __syncthreads();
                if (more) {
#pragma unroll
                    for (uint32_t s = 0; s < 2u; s++) {
                        exl3_chunk_align<bits_x2>(next[s], odd);
                    }
                }
                read_operands(1u - parity, 0u); /* operand_b[0]: operands 4 and 5 are done with it */
            }
            const uint4_t packed = {a[0], a[1], a[2], a[3]};
            const half8_t weights = __builtin_bit_cast(half8_t, packed);
#pragma unroll
            for (uint32_t j = 0; j < LIVE; j++) {
                accumulator[h][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(weights, operand_b[k / 2u % 2u][j], accumulator[h][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (uint32_t w = 0; w < 8u; w++) {
                    if (w * LIVE / 8u == j) {
                        if (k + 1u < 8u) {
                            decode_weight(now, k + 1u, w, ahead);
                        } else {
                            decode_weight(next, 0u, w, ahead);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (uint32_t t = 0; t < 4u; t++) {
                a[t] = ahead[t];
            }
        }
    };
    for (uint32_t step = 0; step < steps; step += 2u) {
        one_step(step, 0u, held[0], held[1]);
        if (step + 1u < steps) {
            one_step(step + 1u, 1u, held[1], held[0]);
        }
    }
}

/* launches 3 and 5: grid (ceil(outputs / 256), chunk capacity, projections), block 256.
 * pass EXL3_TCP_GATE_AND_UP: z = 0 gate, 1 up, products [z][place][intermediate]; pass EXL3_TCP_DOWN: down,
 * products [place][hidden]. */
extern "C" __global__ void __launch_bounds__(TCP_GEMM_THREADS, 2) exl3_tcp_gemm(struct exl3_tcp_record record, unsigned char *arena)
{
    __shared__ __attribute__((aligned(128))) unsigned char stages[2u * TCP_STAGE_BYTES];
    const tcp_shape shape = tcp_shape_of(record);
    unsigned char *workspace = arena + record.workspace_offset;
    /* Which (strip of 256 outputs, chunk, projection) this block takes. The card deals blocks to its eight dies in turn by
     * their number x + gx (y + gy z), so die c holds the blocks whose x % 8 is c. Every output strip of a chunk reads the
     * chunk's operand columns: the blocks of eight consecutive rows m = y + gy z of the grid are re-assigned so that those
     * a die holds among them are all the strips of one (chunk, projection), which then come from memory into that die's
     * level-2 cache once (a grid whose x is no multiple of eight, and the rows past the last whole eight, stay as dealt). */
    const bool down = record.pass == EXL3_TCP_DOWN;
    const uint32_t strips = ((down ? shape.hidden : shape.intermediate) + EXL3_TCP_BLOCK_OUTPUTS - 1u) / EXL3_TCP_BLOCK_OUTPUTS; /* the grid's */
    const uint32_t capacity = shape.layout.chunk_capacity, places = capacity * (down ? 1u : 2u);
    uint32_t strip = blockIdx.x, place = blockIdx.y + capacity * blockIdx.z;
    if (strips % TCP_DIES == 0u && place < places / TCP_DIES * TCP_DIES) {
        strip = (place % TCP_DIES) * (strips / TCP_DIES) + blockIdx.x / TCP_DIES;
        place = place / TCP_DIES * TCP_DIES + blockIdx.x % TCP_DIES;
    }
    const struct exl3_tcp_chunk chunk = tcp_chunk_of(shape, workspace, place % capacity);
    if (chunk.pair_count == 0u) {
        return;
    }
    const uint32_t lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t projection = down ? 2u : place / capacity;
    const uint32_t inputs = down ? shape.intermediate : shape.hidden, outputs = down ? shape.hidden : shape.intermediate;
    const uint32_t bits_x2 = tcp_bits_x2(record, arena, chunk.expert, projection);
    const uint32_t *codes = (const uint32_t *)(arena + tcp_matrix_of(record, arena, chunk.expert, projection));
    const half_t *columns = (const half_t *)(workspace + shape.layout.operands) +
                            ((uint64_t)(down ? 0u : projection) * shape.pairs + chunk.first_pair) * inputs;
    float *products = down ? (float *)(workspace + shape.layout.down) + (uint64_t)chunk.first_pair * outputs
                           : (float *)(workspace + shape.layout.gate_up) + ((uint64_t)projection * shape.pairs + chunk.first_pair) * outputs;
    const uint32_t strip_tile = (strip * EXL3_TCP_BLOCK_OUTPUTS) / EXL3_TILE + wave * 2u * TCP_WAVE_PAIRS;
    const bool strip_is_live = strip_tile * EXL3_TILE < outputs;
    const uint32_t stage_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)stages;
    const uint32_t live_blocks = (chunk.pair_count + 15u) / 16u;
    /* one instance a width and a count of live blocks of 32 columns (1 to 5): the pairs' columns and nothing past them */
#define TCP_GEMM_OF(bits, live)                                                                                                   \
    do {                                                                                                                          \
        float16v_t accumulator[2][live];                                                                                          \
        tcp_wave_gemm<bits, live>(codes, outputs / EXL3_TILE, strip_tile, inputs, columns, chunk.pair_count, stage_base, wave, lane, \
                                    strip_is_live, accumulator);                                                                  \
        if (strip_is_live) {                                                                                                      \
            _Pragma("unroll") for (uint32_t j = 0; j < live; j++)                                                                 \
            {                                                                                                                     \
                const uint32_t column = 32u * j + lane % 32u;                                                                     \
                if (column < chunk.pair_count) {                                                                                  \
                    float *out = products + (uint64_t)column * outputs;                                                           \
                    _Pragma("unroll") for (uint32_t h = 0; h < 2u; h++)                                                           \
                    {                                                                                                             \
                        _Pragma("unroll") for (uint32_t q = 0; q < 4u; q++)                                                       \
                        {                                                                                                         \
                            const uint32_t first_row = 8u * q + 4u * (lane / 32u);                                                \
                            const uint32_t output = EXL3_TILE * (strip_tile + first_row % 16u / 8u + 2u * (first_row / 16u)) +    \
                                                    first_row % 8u + 8u * h;                                                      \
                            *(float4_t *)(out + output) = (float4_t){accumulator[h][j][4u * q], accumulator[h][j][4u * q + 1u],   \
                                                                     accumulator[h][j][4u * q + 2u], accumulator[h][j][4u * q + 3u]}; \
                        }                                                                                                         \
                    }                                                                                                             \
                }                                                                                                                 \
            }                                                                                                                     \
        }                                                                                                                         \
    } while (0)
#define TCP_GEMM_WIDTH(bits)                    \
    if (live_blocks <= 2u) {                    \
        TCP_GEMM_OF(bits, 1u);                  \
    } else if (live_blocks <= 4u) {             \
        TCP_GEMM_OF(bits, 2u);                  \
    } else if (live_blocks <= 6u) {             \
        TCP_GEMM_OF(bits, 3u);                  \
    } else if (live_blocks <= 8u) {             \
        TCP_GEMM_OF(bits, 4u);                  \
    } else {                                    \
        TCP_GEMM_OF(bits, TCP_COLUMN_BLOCKS / 2u); \
    }
    switch (bits_x2) {
    case 4u: TCP_GEMM_WIDTH(4u) break;
    case 5u: TCP_GEMM_WIDTH(5u) break;
    case 6u: TCP_GEMM_WIDTH(6u) break;
    case 8u: TCP_GEMM_WIDTH(8u) break;
    default: return; /* no width of the format: the prepare refuses such a record */
    }
#undef TCP_GEMM_WIDTH
#undef TCP_GEMM_OF
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_gemm, exl3_tcp_record);

/*
 * The GEMM of few pairs an expert. The launch above is written for chunks of up to 160 pairs: their sums (160 registers)
 * leave room for two wavefronts a SIMD, and at two the vector unit issues an instruction every 5 to 6 cycles where it
 * issues one every 4.5 at four; with a handful of pairs an expert the launch is nothing but decoding, and the step's
 * barrier and wait are paid for columns that are not there. This form keeps its operands to itself: codes and operand
 * columns go from memory straight into a wavefront's registers, no LDS and no barrier, at four wavefronts a SIMD.
 * Lanes and decode are the stream product's (exl3_stream_device.cuh), and so is the matrix instruction of 16 x 16 outputs:
 * a decoded operand feeds one for every sixteen pairs. (On the 32 x 32 instruction above, with the same bits as above, the
 * half-empty columns cost: 1012 us for the first call below.)
 * What bounds it is the vector unit (3.75 instructions a weight). Whole calls, hidden 4096, intermediate 2048, 256 experts,
 * 8 picks, this form against the one above: 203 rows 947 / 1120 us, 66 rows 838 / 992, 512 rows 1063 / 1197; 203 rows of
 * Zipf(1.1) loads 960 / 1061. Four wavefronts with room for 32, 48 and 64 pairs a block (three wavefronts): 955, 947 and
 * 975 us at 203 rows, 1002, 960 and 984 at the Zipf loads; two pairs of tiles or four a wavefront: the same.
 */

/* A wavefront's product of TCP_WAVE_PAIRS pairs of adjacent output tiles by CB blocks of sixteen columns. The inner half v
 * of the operands' values is outermost in a step, so that one set of registers holds them: a half's values of the next
 * step are asked for behind its last use, half a step ahead. */
template <uint32_t bits_x2, uint32_t CB>
__device__ static __forceinline__ void tcp_thin_item(const uint32_t *__restrict__ codes, uint32_t inputs, uint32_t outputs, uint32_t strip_tile,
                                                     const half_t *__restrict__ columns, uint32_t column_count, float *__restrict__ products, uint32_t lane)
{
    typedef exl3_chunk<bits_x2> C;
    const uint32_t out_tiles = outputs / EXL3_TILE, g = lane / 16u, i = lane % 16u, c = i % 8u;
    const bool odd = (c & 1u) != 0u;
    uint32_t own, front;
    exl3_chunk_place<bits_x2>(c, own, front);
    const uint64_t step_stride = 4u * (uint64_t)out_tiles * C::tile_words; /* words between steps */
    const uint32_t *tile = codes + ((uint64_t)g * out_tiles + strip_tile + i / 8u) * C::tile_words;
    /* the lane's column of each block at its K tile's values, in bytes (EXL3_TCP_THIN_WIDTH keeps 48 columns within 32
     * bits); a column past the pairs names the first: its sums are not stored, and the instruction keeps columns apart */
    const unsigned char *x = (const unsigned char *)columns;
    uint32_t column_at[CB];
#pragma unroll
    for (uint32_t b = 0; b < CB; b++) {
        const uint32_t column = 16u * b + i;
        column_at[b] = ((column < column_count ? column : 0u) * inputs + g * EXL3_TILE) * 2u;
    }
    float4_t accumulator[TCP_WAVE_PAIRS][2][CB];
#pragma unroll
    for (uint32_t p = 0; p < TCP_WAVE_PAIRS; p++) {
#pragma unroll
        for (uint32_t b = 0; b < CB; b++) {
            accumulator[p][0][b] = accumulator[p][1][b] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    exl3_chunk_words<bits_x2> held[2][TCP_WAVE_PAIRS];
    uint4_t operand[2][CB];
    const auto load_codes = [&](exl3_chunk_words<bits_x2> (&into)[TCP_WAVE_PAIRS]) {
#pragma unroll
        for (uint32_t p = 0; p < TCP_WAVE_PAIRS; p++) {
            exl3_chunk_load<bits_x2>(tile + p * 2u * C::tile_words, own, front, into[p]);
        }
    };
    const auto load_operands = [&](uint32_t v) {
#pragma unroll
        for (uint32_t b = 0; b < CB; b++) {
            operand[v][b] = *(const uint4_t *)(x + column_at[b] + 16u * v);
        }
    };
    const uint32_t steps = inputs / TCP_STEP_INPUTS;
    load_codes(held[0]);
    load_operands(0u);
    load_operands(1u);
    const auto one_step = [&](uint32_t step, exl3_chunk_words<bits_x2> (&now)[TCP_WAVE_PAIRS], exl3_chunk_words<bits_x2> (&next)[TCP_WAVE_PAIRS]) {
        const bool more = step + 1u < steps; /* the same in every lane */
        if (more) {
            tile += step_stride;
            load_codes(next);
        }
        x += more ? TCP_STEP_INPUTS * 2u : 0u; /* the last step asks for its own values again: no branch around the loads */
        uint32_t funnel[TCP_WAVE_PAIRS][C::words];
#pragma unroll
        for (uint32_t p = 0; p < TCP_WAVE_PAIRS; p++) {
            exl3_chunk_align<bits_x2>(now[p], odd);
#pragma unroll
            for (uint32_t word = 0; word < C::words; word++) {
                funnel[p][word] = __builtin_amdgcn_alignbit(now[p].z[word], now[p].z[word + 1u], 16u);
            }
        }
#pragma unroll
        for (uint32_t v = 0; v < 2u; v++) {
#pragma unroll
            for (uint32_t p = 0; p < TCP_WAVE_PAIRS; p++) {
#pragma unroll
                for (uint32_t h = 0; h < 2u; h++) {
                    uint32_t a[4];
#pragma unroll
                    for (uint32_t t = 0; t < 4u; t++) {
                        const uint32_t m = 8u * t + 4u * h + 2u * v;
                        a[t] = exl3_decode_pair(exl3_chunk_state<bits_x2>(now[p].z, funnel[p], m), exl3_chunk_state<bits_x2>(now[p].z, funnel[p], m + 1u));
                    }
                    const uint4_t packed = {a[0], a[1], a[2], a[3]};
                    const half8_t weights = __builtin_bit_cast(half8_t, packed);
#pragma unroll
                    for (uint32_t b = 0; b < CB; b++) {
                        accumulator[p][h][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(weights, __builtin_bit_cast(half8_t, operand[v][b]), accumulator[p][h][b], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0); /* the next operand's decoding, hoisted above, spills */
                }
            }
            load_operands(v);
        }
    };
    for (uint32_t step = 0; step < steps; step += 2u) {
        one_step(step, held[0], held[1]);
        if (step + 1u < steps) {
            one_step(step + 1u, held[1], held[0]);
        }
    }
#pragma unroll
    for (uint32_t b = 0; b < CB; b++) {
        const uint32_t column = 16u * b + i;
        if (column < column_count) {
            float *out = products + (uint64_t)column * outputs;
#pragma unroll
            for (uint32_t p = 0; p < TCP_WAVE_PAIRS; p++) {
#pragma unroll
                for (uint32_t h = 0; h < 2u; h++) {
                    *(float4_t *)(out + exl3_stream_output(strip_tile, p, h, lane)) = accumulator[p][h][b];
                }
            }
        }
    }
}

/* launches 3 and 5 of a call of few pairs an expert (exl3_tcp_is_thin): grid (ceil(outputs / 256), chunk capacity,
 * projections x EXL3_TCP_THIN_PARTS), block 256. A block takes EXL3_TCP_THIN_COLUMNS pairs of a chunk, so that a busy
 * expert's chunk is several blocks side by side and not a long one at the launch's end. */
extern "C" __global__ void __launch_bounds__(TCP_GEMM_THREADS, 4) exl3_tcp_gemm_thin(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    unsigned char *workspace = arena + record.workspace_offset;
    const struct exl3_tcp_chunk chunk = tcp_chunk_of(shape, workspace, blockIdx.y);
    const bool down = record.pass == EXL3_TCP_DOWN;
    const uint32_t projection = down ? 2u : blockIdx.z % 2u, first = (down ? blockIdx.z : blockIdx.z / 2u) * EXL3_TCP_THIN_COLUMNS;
    if (first >= chunk.pair_count) {
        return;
    }
    const uint32_t left = chunk.pair_count - first, count = left < EXL3_TCP_THIN_COLUMNS ? left : EXL3_TCP_THIN_COLUMNS;
    const uint32_t lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t inputs = down ? shape.intermediate : shape.hidden, outputs = down ? shape.hidden : shape.intermediate;
    const uint32_t strip_tile = (blockIdx.x * EXL3_TCP_BLOCK_OUTPUTS) / EXL3_TILE + wave * 2u * TCP_WAVE_PAIRS;
    if (strip_tile * EXL3_TILE >= outputs) {
        return;
    }
    const uint32_t bits_x2 = tcp_bits_x2(record, arena, chunk.expert, projection);
    const uint32_t *codes = (const uint32_t *)(arena + tcp_matrix_of(record, arena, chunk.expert, projection));
    const uint64_t place = chunk.first_pair + first;
    const half_t *columns = (const half_t *)(workspace + shape.layout.operands) + ((uint64_t)(down ? 0u : projection) * shape.pairs + place) * inputs;
    float *products = down ? (float *)(workspace + shape.layout.down) + place * outputs
                           : (float *)(workspace + shape.layout.gate_up) + ((uint64_t)projection * shape.pairs + place) * outputs;
    /* one instance a width and a count of blocks of sixteen columns */
#define TCP_THIN_WIDTH(bits)                                                                         \
    if (count <= 16u) {                                                                              \
        tcp_thin_item<bits, 1u>(codes, inputs, outputs, strip_tile, columns, count, products, lane); \
    } else if (count <= 32u) {                                                                       \
        tcp_thin_item<bits, 2u>(codes, inputs, outputs, strip_tile, columns, count, products, lane); \
    } else {                                                                                         \
        tcp_thin_item<bits, EXL3_TCP_THIN_COLUMNS / 16u>(codes, inputs, outputs, strip_tile, columns, count, products, lane); \
    }
    switch (bits_x2) {
    case 4u: TCP_THIN_WIDTH(4u) break;
    case 5u: TCP_THIN_WIDTH(5u) break;
    case 6u: TCP_THIN_WIDTH(6u) break;
    case 8u: TCP_THIN_WIDTH(8u) break;
    default: return; /* no width of the format: the prepare refuses such a record */
    }
#undef TCP_THIN_WIDTH
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_gemm_thin, exl3_tcp_record);

/* a pair's gate and up products (gate's eight, then up's) as its down operand */
__device__ static __forceinline__ uint4_t tcp_activated(const float4_t (&loads)[4], const float (&gs)[8], const float (&us)[8], const float (&ds)[8],
                                                        float limit, uint32_t lane)
{
    float g[8], u[8];
#pragma unroll
    for (uint32_t j = 0; j < 8u; j++) {
        g[j] = loads[j / 4u][j % 4u];
        u[j] = loads[2u + j / 4u][j % 4u];
    }
    return row_activated(g, u, gs, us, ds, limit, lane);
}

/* launch 4: grid (ceil(intermediate / 512), chunk capacity, EXL3_TCP_COLUMN_PARTS), block 64: per pair of a part of the chunk, gate = H128(gate products) /
 * sqrt(128) x svh, up the same, the SwiGLU with its limit, x the down matrix's suh, H128 -> the fp16 down operand */
extern "C" __global__ void exl3_tcp_activate(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    unsigned char *workspace = arena + record.workspace_offset;
    const struct exl3_tcp_chunk chunk = tcp_chunk_of(shape, workspace, blockIdx.y);
    const uint32_t first_column = blockIdx.z * EXL3_TCP_PART_COLUMNS;
    uint32_t channel;
    if (first_column >= chunk.pair_count || !tcp_lane_channels(shape.intermediate, channel)) {
        return;
    }
    const uint32_t lane = threadIdx.x;
    const uint32_t last_column = first_column + EXL3_TCP_PART_COLUMNS < chunk.pair_count ? first_column + EXL3_TCP_PART_COLUMNS : chunk.pair_count;
    const uint32_t H = shape.hidden, I = shape.intermediate, e = chunk.expert;
    const uint16_t *gate_svh = (const uint16_t *)(arena + tcp_matrix_of(record, arena, e, 0u) + exl3_code_bytes(H, I, tcp_bits_x2(record, arena, e, 0u))) + H;
    const uint16_t *up_svh = (const uint16_t *)(arena + tcp_matrix_of(record, arena, e, 1u) + exl3_code_bytes(H, I, tcp_bits_x2(record, arena, e, 1u))) + H;
    const uint16_t *down_suh = (const uint16_t *)(arena + tcp_matrix_of(record, arena, e, 2u) + exl3_code_bytes(I, H, tcp_bits_x2(record, arena, e, 2u)));
    float gs[8], us[8], ds[8];
    unpack_half8(*(const uint4_t *)(gate_svh + channel), gs);
    unpack_half8(*(const uint4_t *)(up_svh + channel), us);
    unpack_half8(*(const uint4_t *)(down_suh + channel), ds);
    const float limit = record.activation_limit;
    const float *gate_products = (const float *)(workspace + shape.layout.gate_up);
    const float *up_products = gate_products + (uint64_t)shape.pairs * I;
    uint16_t *operands = (uint16_t *)(workspace + shape.layout.operands);
    constexpr uint32_t BATCH = 2u; /* two columns' eight loads together */
    for (uint32_t first = first_column; first < last_column; first += BATCH) {
        float4_t loads[BATCH][4];
        uint64_t place[BATCH];
#pragma unroll
        for (uint32_t i = 0; i < BATCH; i++) {
            const uint32_t column = first + i < last_column ? first + i : last_column - 1u;
            place[i] = chunk.first_pair + column;
            const float4_t *gate = (const float4_t *)(gate_products + place[i] * I + channel), *up = (const float4_t *)(up_products + place[i] * I + channel);
            loads[i][0] = gate[0];
            loads[i][1] = gate[1];
            loads[i][2] = up[0];
            loads[i][3] = up[1];
        }
#pragma unroll
        for (uint32_t i = 0; i < BATCH; i++) {
            const uint4_t operand = tcp_activated(loads[i], gs, us, ds, limit, lane);
            if (first + i < last_column) {
                *(uint4_t *)(operands + place[i] * I + channel) = operand;
            }
        }
    }
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_activate, exl3_tcp_record);

extern "C" __global__ void __launch_bounds__(TCP_THIN_PLACES * WAVE) exl3_tcp_activate_thin(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    const uint32_t H = shape.hidden, I = shape.intermediate;
    uint32_t place, pair, expert, channel, lane;
    if (!tcp_thin_place(shape, record, arena, I, place, pair, expert, channel, lane)) {
        return;
    }
    unsigned char *workspace = arena + record.workspace_offset;
    const float *products = (const float *)(workspace + shape.layout.gate_up);
    const float4_t *gate = (const float4_t *)(products + (uint64_t)place * I + channel), *up = (const float4_t *)(products + ((uint64_t)shape.pairs + place) * I + channel);
    const float4_t loads[4] = {gate[0], gate[1], up[0], up[1]};
    const uint4_t scales[3] = {
        *(const uint4_t *)((const uint16_t *)(arena + tcp_matrix_of(record, arena, expert, 0u) + exl3_code_bytes(H, I, tcp_bits_x2(record, arena, expert, 0u))) + H + channel),
        *(const uint4_t *)((const uint16_t *)(arena + tcp_matrix_of(record, arena, expert, 1u) + exl3_code_bytes(H, I, tcp_bits_x2(record, arena, expert, 1u))) + H + channel),
        *(const uint4_t *)((const uint16_t *)(arena + tcp_matrix_of(record, arena, expert, 2u) + exl3_code_bytes(I, H, tcp_bits_x2(record, arena, expert, 2u))) + channel)};
    float gs[8], us[8], ds[8];
    unpack_half8(scales[0], gs);
    unpack_half8(scales[1], us);
    unpack_half8(scales[2], ds);
    *(uint4_t *)((uint16_t *)(workspace + shape.layout.operands) + (uint64_t)place * I + channel) = tcp_activated(loads, gs, us, ds, record.activation_limit, lane);
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_activate_thin, exl3_tcp_record);

/* launch 6: grid (ceil(hidden / 512), row_count), block 64: a row's pairs in slot order */
extern "C" __global__ void exl3_tcp_combine(struct exl3_tcp_record record, unsigned char *arena)
{
    const tcp_shape shape = tcp_shape_of(record);
    const unsigned char *workspace = arena + record.workspace_offset;
    uint32_t channel;
    if (!tcp_lane_channels(shape.hidden, channel)) {
        return;
    }
    const uint32_t lane = threadIdx.x, row = blockIdx.y;
    const uint32_t H = shape.hidden, I = shape.intermediate;
    const struct router_pick *picks = (const struct router_pick *)(arena + record.picks_offset) + (uint64_t)row * shape.picks;
    const uint32_t *place_of = (const uint32_t *)(workspace + shape.layout.place_of);
    const float *down = (const float *)(workspace + shape.layout.down);
    const float normalization = row_normalization(lane);
    float sum[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    /* TCP_BATCH slots at a time: their products, and behind them their scales, are asked for together (a slot past the last
     * repeats it and is not added; one at a time: 203 rows 12.0 us and not 10.7, 4096 rows 120 and not 117; eight: 12.3, 122) */
    for (uint32_t first = 0; first < shape.picks; first += TCP_BATCH) {
        float4_t low[TCP_BATCH], high[TCP_BATCH];
        uint4_t scales[TCP_BATCH];
        float weight[TCP_BATCH];
#pragma unroll
        for (uint32_t i = 0; i < TCP_BATCH; i++) {
            const uint32_t slot = first + i < shape.picks ? first + i : shape.picks - 1u;
            const float4_t *products = (const float4_t *)(down + (uint64_t)place_of[row * shape.picks + slot] * H + channel);
            low[i] = products[0];
            high[i] = products[1];
        }
#pragma unroll
        for (uint32_t i = 0; i < TCP_BATCH; i++) {
            const struct router_pick pick = picks[first + i < shape.picks ? first + i : shape.picks - 1u];
            weight[i] = pick.route_weight;
            scales[i] = *(const uint4_t *)((const uint16_t *)(arena + tcp_matrix_of(record, arena, pick.expert, 2u) +
                                                              exl3_code_bytes(I, H, tcp_bits_x2(record, arena, pick.expert, 2u))) + I + channel);
        }
#pragma unroll
        for (uint32_t i = 0; i < TCP_BATCH; i++) {
            float v[8] = {low[i][0], low[i][1], low[i][2], low[i][3], high[i][0], high[i][1], high[i][2], high[i][3]}, scale[8];
            unpack_half8(scales[i], scale);
            row_hadamard128(v, lane);
            if (first + i < shape.picks) {
#pragma unroll
                for (uint32_t j = 0; j < 8u; j++) {
                    sum[j] = __fadd_rn(sum[j], __fmul_rn(__fmul_rn(row_normalized(v[j], normalization), scale[j]), weight[i]));
                }
            }
        }
    }
    float4_t *out = (float4_t *)((float *)(arena + record.output_offset) + (uint64_t)row * H + channel);
    out[0] = (float4_t){sum[0], sum[1], sum[2], sum[3]};
    out[1] = (float4_t){sum[4], sum[5], sum[6], sum[7]};
}
ANEMONE_KERNEL(EXL3_TCP_KERNEL_FILE, exl3_tcp_combine, exl3_tcp_record);
