/*
 * kernel_exl3.hip -- EXL3 (trellis, codebook mul1) reconstruction and the routed experts' five-launch chain for
 * gfx950. Entry names and records are the reference's (source/kernel_exl3.cu, include/anemone/exl3_records.h);
 * the work mapping is this build's: one wavefront per 128-value transform block, and products by wavefronts whose lanes
 * take their codes from memory and decode them for v_mfma_f32_16x16x32_f16 (exl3_stream_device.cuh).
 *
 * Arithmetic contract (source/kernel_exl3.cu:133-424): operands fp16( H128(bf16 x . fp16 suh) . norm ); products
 * float32 in four contiguous K slices added in slice order from +0; hidden bf16( min(g, L) / (1 + e^-g) . clamp(u) )
 * with g, u = H128(product) . norm . svh; down operand from the unrounded hidden value; pair output
 * H128(down product) . norm . svh . route weight, in place of the down products; row sum in slot order from +0.
 * Inside a slice the MFMA adds 32 products at a time in its own order, which no host reference has bit for bit.
 */
#include "exl3_stream_device.cuh"
#include "kernel_registry.h"

#define PRODUCT_WAVES EXL3_PRODUCT_SLICES
#define PRODUCT_THREADS (PRODUCT_WAVES * WAVE)

extern "C" __global__ void exl3_reconstruct(struct exl3_reconstruct_record record, unsigned char *arena)
{
    const uint64_t element = (uint64_t)blockIdx.x * LINEAR_ELEMENT_THREADS + threadIdx.x;
    if (element >= (uint64_t)record.input_size * record.output_size) {
        return;
    }
    const uint32_t input = (uint32_t)(element / record.output_size), output = (uint32_t)(element % record.output_size);
    const uint32_t bits_x2 = exl3_bits_x2(record.bits_per_weight);
    const uint32_t ring_bits = EXL3_TILE_VALUES * bits_x2 / 2u, tile_words = ring_bits / 32u;
    const uint64_t tile = (uint64_t)(input / EXL3_TILE) * (record.output_size / EXL3_TILE) + output / EXL3_TILE;
    const uint32_t *words = (const uint32_t *)(arena + record.matrix_offset) + tile * tile_words;
    const uint32_t i = input % EXL3_TILE, o = output % EXL3_TILE;
    const uint32_t position = 8u * (4u * (o % 8u) + (i % 8u) / 2u) + (i & 1u) + 2u * (i / 8u) + 4u * (o / 8u);
    const uint32_t begin = (exl3_window_end(position, bits_x2) + ring_bits - 16u) % ring_bits;
    const uint32_t word = begin / 32u, shift = begin % 32u;
    uint32_t window = words[word] << shift;
    if (shift != 0u) {
        window |= words[(word + 1u) % tile_words] >> (32u - shift);
    }
    ((uint16_t *)(arena + record.output_offset))[element] = exl3_decode_one(window >> 16);
}
ANEMONE_KERNEL(EXL3_KERNEL_FILE, exl3_reconstruct, exl3_reconstruct_record);

/* the stored width of matrix m (0 gate, 1 up, 2 down) of a job's expert */
__device__ static __forceinline__ uint32_t chain_width(const struct exl3_expert_record &record,
                                                       const unsigned char *arena, uint32_t expert, uint32_t matrix)
{
    if (record.widths_offset == 0u) {
        return record.bits_per_weight;
    }
    return exl3_width_of(((const uint32_t *)(arena + record.widths_offset))[expert], matrix);
}

/* The element-wise launches (input, activate, finish): a block is 128 channels of one job, a wavefront one of its rows, or more
 * where the job has more rows than the block wavefronts: rows one behind the other in one wavefront are a chain of their
 * transforms (one 4096-wide matrix by eight rows: input 4.7 -> 2.3 us, finish 3.4 -> 2.2). The step to a wavefront's next row is
 * formed behind a row: ahead of the first it stood in the chain of a launch of one row (input 2.22 -> 2.17 us, the matrix's three
 * launches 10.1 -> 10.0). */
__device__ static __forceinline__ uint32_t element_stride(const struct exl3_expert_record &record)
{
    uint32_t jobs = record.job_count;
    asm volatile("" : "+s"(jobs)); /* not known to be the same for every row */
    return exl3_element_rows(record.pair_count, jobs);
}

extern "C" __global__ void __launch_bounds__(EXL3_ELEMENT_MOST_THREADS) exl3_input(struct exl3_expert_record record, unsigned char *arena)
{
    const struct expert_job_record *job = (const struct expert_job_record *)(arena + record.jobs_offset) + blockIdx.y;
    if (job->row_count == 0u) {
        return;
    }
    const uint32_t lane = threadIdx.x % WAVE, projection = blockIdx.z;
    const uint32_t channel = blockIdx.x * EXL3_TRANSFORM + wave_channel<false>(lane), to = blockIdx.x * EXL3_TRANSFORM + wave_channel<true>(lane);
    const float normalization = row_normalization(lane);
    const uint64_t matrix = projection == 0u ? job->gate_offset : job->up_offset;
    const uint32_t bits_x2 = exl3_bits_x2(chain_width(record, arena, job->expert, projection));
    const uint16_t *suh = (const uint16_t *)(arena + matrix + exl3_code_bytes(record.input_size, record.inner_size, bits_x2));
    const float s0 = half_bits_to_float(suh[channel]), s1 = half_bits_to_float(suh[channel + WAVE]);
    const uint16_t *input = (const uint16_t *)(arena + record.input_offset);
    uint16_t *operands = (uint16_t *)(arena + record.operands_offset);
    for (uint32_t column = threadIdx.x / WAVE; column < job->row_count; column += element_stride(record)) {
        const uint32_t pair = job->pair_index[column];
        const uint64_t row = pair / record.pairs_per_row;
        float v0 = __fmul_rn(bf16_to_float(input[row * record.input_size + channel]), s0);
        float v1 = __fmul_rn(bf16_to_float(input[row * record.input_size + channel + WAVE]), s1);
        wave_hadamard128<false>(v0, v1, lane);
        uint16_t *out = operands + ((uint64_t)projection * record.pair_count + pair) * record.input_size;
        out[to] = float_to_half_bits(row_normalized(v0, normalization));
        out[to + WAVE] = float_to_half_bits(row_normalized(v1, normalization));
    }
}
ANEMONE_KERNEL(EXL3_KERNEL_FILE, exl3_input, exl3_expert_record);

/* Products of one job: block = four wavefronts = the four K slices (whole steps of four K tiles) of one strip of
 * STRIP_TILES output tiles: eight (the stream product), or one in the thin instances, which a launch of few jobs takes so
 * that its blocks cover the card (the same slices and the same order of sums, so the same bits).
 * A thin launch of at most a block a CU has a wavefront a SIMD, so its time is the chain of one wavefront, which issues an
 * instruction every six to seven cycles: its codes' loads run eight steps ahead and pass through no LDS, and a step is its decoding
 * and little else (exl3_stream_tile_product: no copies of registers, scalar addresses; 103 -> 72 vector instructions a step). One
 * 4096 x 4096 matrix of K 4 by one vector, launches queued back to back: the product 6.5 -> 5.75 us, the input, product and finish
 * 10.5 -> 9.85 (in the first form, two K tiles a step through an LDS window, 16.5).
 * The thin instances of more blocks (_thin_many) run five steps ahead: 80 to 90 registers, five wavefronts a SIMD, where eight
 * ahead take 110 to 125 and leave three or four. 512 blocks, product alone, us, before | now | seven ahead: 8192 inputs of K 2.5
 * 16.9 | 15.6 | 15.7, of K 4 17.2 | 16.8 | 17.0; 320 blocks of 5120 inputs, K 3 10.2 | 9.15 | 9.35.
 * The eight-tile instances are held to three wavefronts a SIMD: left to itself the compiler keeps the sums in accumulation
 * registers and copies beside them (175 registers, two wavefronts, for K 4): down of 32 jobs at 1536 x 5120 40.5 -> 39.0 us,
 * of 64 at 2048 x 4096 79.7 -> 74.6. */
template <uint32_t bits_x2, bool down, uint32_t STRIP_TILES, uint32_t STEPS_AHEAD>
__device__ static __forceinline__ void chain_product(const struct exl3_expert_record &record, unsigned char *arena,
                                                     const struct expert_job_record *job, float *partial)
{
    const uint32_t projection = blockIdx.z;
    const uint32_t inputs = down ? record.inner_size : record.input_size;
    const uint32_t outputs = down ? record.input_size : record.inner_size;
    const uint32_t lane = threadIdx.x % WAVE, slice = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint64_t matrix = down ? job->down_offset : projection == 0u ? job->gate_offset : job->up_offset;
    const uint32_t column = lane % 16u;
    /* a column that is not live reads the first column's operand: its sums are not stored */
    const uint32_t pair = job->pair_index[column < job->row_count ? column : 0u];
    const unsigned char *operands = arena + record.operands_offset + (uint64_t)projection * record.pair_count * inputs * 2u;
    const uint32_t steps = inputs / (4u * EXL3_TILE), strip_tile = blockIdx.x * STRIP_TILES;
    const uint32_t first_tile = 4u * (steps * slice / PRODUCT_WAVES), last_tile = 4u * (steps * (slice + 1u) / PRODUCT_WAVES);
    const uint32_t *codes = (const uint32_t *)(arena + matrix);
    float4_t sums[STRIP_TILES];
    if constexpr (STRIP_TILES == 1u) {
        exl3_stream_tile_product<bits_x2, STEPS_AHEAD>(codes, outputs / EXL3_TILE, strip_tile, first_tile, last_tile, operands, pair * inputs * 2u, lane, sums[0]);
    } else {
        float4_t accumulator[STRIP_TILES / 2u][2];
        exl3_stream_product<bits_x2, STRIP_TILES / 2u, true>(codes, outputs / EXL3_TILE, strip_tile, first_tile, last_tile, (const half_t *)operands + (uint64_t)pair * inputs, lane, accumulator);
#pragma unroll
        for (uint32_t n = 0; n < STRIP_TILES; n++) {
            sums[n] = accumulator[n / 2u][n % 2u];
        }
    }
    /* partial [slice][n][lane] as float4; slice 0 then adds the four in order from +0 */
    float4_t *mine = (float4_t *)partial + (slice * STRIP_TILES) * WAVE + lane;
#pragma unroll
    for (uint32_t n = 0; n < STRIP_TILES; n++) {
        mine[n * WAVE] = sums[n];
    }
    __syncthreads();
    if (slice == 0u && column < job->row_count) {
        float *products = (float *)(arena + record.products_offset) + ((uint64_t)projection * record.pair_count + pair) * outputs;
#pragma unroll
        for (uint32_t n = 0; n < STRIP_TILES; n++) {
            float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (uint32_t part = 0; part < PRODUCT_WAVES; part++) {
                const float4_t value = ((const float4_t *)partial)[(part * STRIP_TILES + n) * WAVE + lane];
                sum.x = __fadd_rn(sum.x, value.x);
                sum.y = __fadd_rn(sum.y, value.y);
                sum.z = __fadd_rn(sum.z, value.z);
                sum.w = __fadd_rn(sum.w, value.w);
            }
            /* four outputs a lane, from where the product's form keeps them */
            const uint32_t output = STRIP_TILES == 1u ? strip_tile * EXL3_TILE + 4u * (lane / 16u)
                                                      : exl3_stream_output(strip_tile, n / 2u, n % 2u, lane);
            *(float4_t *)(products + output) = sum;
        }
    }
}

template <uint32_t fixed_bits_x2, bool down, uint32_t STRIP_TILES, uint32_t STEPS_AHEAD = 0u>
__device__ static __forceinline__ void chain_product_entry(const struct exl3_expert_record &record,
                                                           unsigned char *arena)
{
    __shared__ __attribute__((aligned(16))) float partial[PRODUCT_WAVES * STRIP_TILES * WAVE * 4u];
    const struct expert_job_record *job = (const struct expert_job_record *)(arena + record.jobs_offset) + blockIdx.y;
    if (job->row_count == 0u) {
        return;
    }
    uint32_t bits_x2 = fixed_bits_x2;
    if (fixed_bits_x2 == 0u) {
        bits_x2 = exl3_bits_x2(chain_width(record, arena, job->expert, down ? 2u : blockIdx.z));
    }
    switch (bits_x2) {
    case 4u: chain_product<4u, down, STRIP_TILES, STEPS_AHEAD>(record, arena, job, partial); break;
    case 5u: chain_product<5u, down, STRIP_TILES, STEPS_AHEAD>(record, arena, job, partial); break;
    case 6u: chain_product<6u, down, STRIP_TILES, STEPS_AHEAD>(record, arena, job, partial); break;
    case 8u: chain_product<8u, down, STRIP_TILES, STEPS_AHEAD>(record, arena, job, partial); break;
    default: break;
    }
}

#define EXL3_PRODUCT_ENTRY(entry, bits_x2, down, wavefronts, ...)                                            \
    extern "C" __global__ void __launch_bounds__(PRODUCT_THREADS, wavefronts)                                \
        entry(struct exl3_expert_record record, unsigned char *arena)                                        \
    {                                                                                                        \
        chain_product_entry<bits_x2, down, __VA_ARGS__>(record, arena);                                      \
    }                                                                                                        \
    ANEMONE_KERNEL(EXL3_KERNEL_FILE, entry, exl3_expert_record)
#define EXL3_PRODUCT_ENTRIES(name, bits_x2)                                                                  \
    EXL3_PRODUCT_ENTRY(exl3_gate_up_##name, bits_x2, false, 3, EXL3_STRIP_TILES);                            \
    EXL3_PRODUCT_ENTRY(exl3_down_##name, bits_x2, true, 3, EXL3_STRIP_TILES);                                \
    EXL3_PRODUCT_ENTRY(exl3_gate_up_##name##_thin, bits_x2, false, 1, EXL3_THIN_STRIP_TILES, 8u);            \
    EXL3_PRODUCT_ENTRY(exl3_down_##name##_thin, bits_x2, true, 1, EXL3_THIN_STRIP_TILES, 8u);                \
    EXL3_PRODUCT_ENTRY(exl3_gate_up_##name##_thin_many, bits_x2, false, 4, EXL3_THIN_STRIP_TILES, 5u);       \
    EXL3_PRODUCT_ENTRY(exl3_down_##name##_thin_many, bits_x2, true, 4, EXL3_THIN_STRIP_TILES, 5u)
EXL3_PRODUCT_ENTRIES(k2, 4u);
EXL3_PRODUCT_ENTRIES(k2_5, 5u);
EXL3_PRODUCT_ENTRIES(k3, 6u);
EXL3_PRODUCT_ENTRIES(k4, 8u);
EXL3_PRODUCT_ENTRIES(mixed, 0u); /* the width of each matrix from the record's widths table */

extern "C" __global__ void __launch_bounds__(EXL3_ELEMENT_MOST_THREADS) exl3_activate(struct exl3_expert_record record, unsigned char *arena)
{
    const struct expert_job_record *job = (const struct expert_job_record *)(arena + record.jobs_offset) + blockIdx.y;
    if (job->row_count == 0u) {
        return;
    }
    /* the products by channel, the hidden values by the channels their transforms leave a lane with, the operand by channel again */
    const uint32_t lane = threadIdx.x % WAVE;
    const uint32_t channel = blockIdx.x * EXL3_TRANSFORM + wave_channel<false>(lane), between = blockIdx.x * EXL3_TRANSFORM + wave_channel<true>(lane);
    const float normalization = row_normalization(lane);
    const uint32_t H = record.input_size, I = record.inner_size;
    const uint16_t *gate_svh = (const uint16_t *)(arena + job->gate_offset +
                                                  exl3_code_bytes(H, I, exl3_bits_x2(chain_width(record, arena, job->expert, 0u)))) + H;
    const uint16_t *up_svh = (const uint16_t *)(arena + job->up_offset +
                                                exl3_code_bytes(H, I, exl3_bits_x2(chain_width(record, arena, job->expert, 1u)))) + H;
    const uint16_t *down_suh = (const uint16_t *)(arena + job->down_offset +
                                                  exl3_code_bytes(I, H, exl3_bits_x2(chain_width(record, arena, job->expert, 2u))));
    const float gs0 = half_bits_to_float(gate_svh[between]), gs1 = half_bits_to_float(gate_svh[between + WAVE]);
    const float us0 = half_bits_to_float(up_svh[between]), us1 = half_bits_to_float(up_svh[between + WAVE]);
    const float ds0 = half_bits_to_float(down_suh[between]), ds1 = half_bits_to_float(down_suh[between + WAVE]);
    const float limit = record.activation_limit;
    const float *products = (const float *)(arena + record.products_offset);
    for (uint32_t column = threadIdx.x / WAVE; column < job->row_count; column += element_stride(record)) {
        const uint32_t pair = job->pair_index[column];
        float g0 = products[(uint64_t)pair * I + channel], g1 = products[(uint64_t)pair * I + channel + WAVE];
        float u0 = products[((uint64_t)record.pair_count + pair) * I + channel];
        float u1 = products[((uint64_t)record.pair_count + pair) * I + channel + WAVE];
        wave_hadamard128<false>(g0, g1, lane);
        wave_hadamard128<false>(u0, u1, lane);
        float hidden[2];
        const float gate[2] = {__fmul_rn(row_normalized(g0, normalization), gs0), __fmul_rn(row_normalized(g1, normalization), gs1)};
        const float up[2] = {__fmul_rn(row_normalized(u0, normalization), us0), __fmul_rn(row_normalized(u1, normalization), us1)};
#pragma unroll
        for (uint32_t i = 0; i < 2u; i++) {
            const float bounded_gate = fminf(gate[i], limit);
            const float bounded_up = fminf(fmaxf(up[i], -limit), limit);
            hidden[i] = __fmul_rn(det_silu(bounded_gate), bounded_up);
        }
        uint16_t *hidden_out = (uint16_t *)(arena + record.hidden_offset) + (uint64_t)pair * I;
        hidden_out[between] = float_to_bf16(hidden[0]);
        hidden_out[between + WAVE] = float_to_bf16(hidden[1]);
        float v0 = __fmul_rn(hidden[0], ds0), v1 = __fmul_rn(hidden[1], ds1);
        wave_hadamard128<true>(v0, v1, lane);
        uint16_t *operand = (uint16_t *)(arena + record.operands_offset) + (uint64_t)pair * I;
        operand[channel] = float_to_half_bits(row_normalized(v0, normalization));
        operand[channel + WAVE] = float_to_half_bits(row_normalized(v1, normalization));
    }
}
ANEMONE_KERNEL(EXL3_KERNEL_FILE, exl3_activate, exl3_expert_record);

extern "C" __global__ void __launch_bounds__(EXL3_ELEMENT_MOST_THREADS) exl3_finish(struct exl3_expert_record record, unsigned char *arena)
{
    const struct expert_job_record *job = (const struct expert_job_record *)(arena + record.jobs_offset) + blockIdx.y;
    if (job->row_count == 0u) {
        return;
    }
    const uint32_t lane = threadIdx.x % WAVE;
    const uint32_t channel = blockIdx.x * EXL3_TRANSFORM + wave_channel<false>(lane), to = blockIdx.x * EXL3_TRANSFORM + wave_channel<true>(lane);
    const float normalization = row_normalization(lane);
    const uint32_t H = record.input_size, I = record.inner_size;
    const uint16_t *svh = (const uint16_t *)(arena + job->down_offset +
                                             exl3_code_bytes(I, H, exl3_bits_x2(chain_width(record, arena, job->expert, 2u)))) + I;
    const float s0 = half_bits_to_float(svh[to]), s1 = half_bits_to_float(svh[to + WAVE]);
    for (uint32_t column = threadIdx.x / WAVE; column < job->row_count; column += element_stride(record)) {
        const uint32_t pair = job->pair_index[column];
        float *values = (float *)(arena + record.products_offset) + (uint64_t)pair * H;
        float v0 = values[channel], v1 = values[channel + WAVE];
        wave_hadamard128<false>(v0, v1, lane); /* the whole block's loads have landed: the output may take the products' place */
        const float weight = job->route_weight[column];
        float *out = (float *)(arena + record.output_offset) + (uint64_t)pair * H;
        out[to] = __fmul_rn(__fmul_rn(row_normalized(v0, normalization), s0), weight);
        out[to + WAVE] = __fmul_rn(__fmul_rn(row_normalized(v1, normalization), s1), weight);
    }
}
ANEMONE_KERNEL(EXL3_KERNEL_FILE, exl3_finish, exl3_expert_record);

extern "C" __global__ void exl3_row_sum(struct expert_row_sum_arguments record, unsigned char *arena)
{
    const uint32_t channel = blockIdx.x * LINEAR_ELEMENT_THREADS + threadIdx.x;
    if (channel >= record.width) {
        return;
    }
    const uint64_t row = blockIdx.y;
    const float *pairs = (const float *)(arena + record.pair_output_offset);
    float sum = 0.0f;
    for (uint32_t slot = 0; slot < record.pairs_per_row; slot++) {
        sum = __fadd_rn(sum, pairs[(row * record.pairs_per_row + slot) * record.width + channel]);
    }
    ((float *)(arena + record.row_output_offset))[row * record.width + channel] = sum;
}
ANEMONE_KERNEL(EXL3_KERNEL_FILE, exl3_row_sum, expert_row_sum_arguments);
