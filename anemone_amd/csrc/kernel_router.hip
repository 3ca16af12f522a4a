/*
 * kernel_router.hip -- the router of one MoE layer on gfx950: score projection, affinity, top-k choice with route
 * weights, and the job table the routed experts read. Entry names and records follow the reference
 * (source/kernel_router.cu, source/kernel_router.cuh, include/anemone/router_records.h); the expert count, the
 * picks a row, the route scale and the affinity are run-time members of the record (a zero means the reference's
 * 384 / 6 / 1.5 / sqrt(softplus)).
 *
 * What a row's choice is (include/anemone/router_records.h:8-31): affinity a of every expert; the P experts of the
 * largest a + bias compared as the reference's top-k compares float32 (a not-a-number above every number, -0 below
 * +0, the lower expert first among equals); slots in ascending expert order; weights a / (t + 1e-20) * scale, each
 * operation one float32 rounding, t the sum of the P affinities from +0 in ascending expert order (or the
 * reference's tree order for six picks). The job table: a job for each chosen expert, ascending; a column for each
 * row that chose it, rows ascending; unused columns and empty jobs zero. No atomic operation; a row's choice
 * depends on that row alone.
 *
 * exp and log1p are fixed sequences of float32 operations (the same the CPU oracle runs), so that affinities, and
 * with them the expert ids, are the same bits on the card and on the host.
 */
#include "router_device.cuh"
#include "kernel_registry.h"
#include "sort_device.cuh"
#include "quantize_device.cuh"

#define PROJECTION_CHAINS 32u
#define PROJECTION_THREADS 128u

/* scores[row][expert] = sum_k w[expert][k] x[row][k]: 32 fma chains, chain c owning the inputs k = c mod 32 in
 * ascending order, then a halving fold 16, 8, 4, 2, 1 (source/kernel_official_router_projection.cu:33-57).
 * A block takes PROJECTION_EXPERTS experts and up to PROJECTION_ROWS rows: it stages the weights and the rows in
 * chunks of PROJECTION_CHUNK inputs through LDS with 16-byte coalesced loads (the next chunk in flight while this
 * one is consumed); a thread owns chains 2 j and 2 j + 1 of one expert for every row, so the fma order of a chain
 * is the definition's whatever the staging. grid (ceil(E / 8), ceil(rows / 4)), block 128. (A thin step takes a row a
 * block, router_projection_thin.) */
#define PROJECTION_ROWS 4u
#define PROJECTION_EXPERTS 8u
#define PROJECTION_CHUNK 1024u
#define PROJECTION_W_LOADS (PROJECTION_EXPERTS * PROJECTION_CHUNK * 2u / 16u / PROJECTION_THREADS)
__device__ static __forceinline__ void router_projection_block(const struct router_projection_arguments &arguments, unsigned char *arena)
{
    constexpr uint32_t PROJECTION_X_LOADS = PROJECTION_ROWS * PROJECTION_CHUNK * 2u / 16u / PROJECTION_THREADS;
    extern __shared__ __attribute__((aligned(1024))) unsigned char projection_window[]; /* PROJECTION_WINDOW_BYTES */
    static_assert((PROJECTION_EXPERTS + PROJECTION_ROWS) * PROJECTION_CHUNK * 2u == PROJECTION_WINDOW_BYTES, "the window the host asks for");
    uint16_t (*const w_tile)[PROJECTION_CHUNK] = (uint16_t (*)[PROJECTION_CHUNK])projection_window;
    uint16_t (*const x_tile)[PROJECTION_CHUNK] = w_tile + PROJECTION_EXPERTS;
    const uint32_t H = arguments.hidden, thread = threadIdx.x;
    const uint32_t first_expert = blockIdx.x * PROJECTION_EXPERTS, first_row = blockIdx.y * PROJECTION_ROWS;
    const uint16_t *weights = (const uint16_t *)(arena + arguments.weights_offset);
    const uint16_t *rows = (const uint16_t *)(arena + arguments.rows_offset);
    uint4_t w_next[PROJECTION_W_LOADS], x_next[PROJECTION_X_LOADS];
    /* piece p of a tile: 8 values of line p / (CHUNK / 8) at column 8 (p % (CHUNK / 8)); out of range reads zero */
    auto fetch = [&](uint32_t chunk) {
#pragma unroll
        for (uint32_t i = 0; i < PROJECTION_W_LOADS; i++) {
            const uint32_t piece = i * PROJECTION_THREADS + thread, line = piece / (PROJECTION_CHUNK / 8u);
            const uint32_t k = chunk + 8u * (piece % (PROJECTION_CHUNK / 8u)), expert = first_expert + line;
            w_next[i] = (uint4_t){0, 0, 0, 0};
            if (expert < arguments.expert_count && k < H) {
                w_next[i] = *(const uint4_t *)(weights + (uint64_t)expert * H + k);
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < PROJECTION_X_LOADS; i++) {
            const uint32_t piece = i * PROJECTION_THREADS + thread, line = piece / (PROJECTION_CHUNK / 8u);
            const uint32_t k = chunk + 8u * (piece % (PROJECTION_CHUNK / 8u)), row = first_row + line;
            x_next[i] = (uint4_t){0, 0, 0, 0};
            if (row < arguments.row_count && k < H) {
                x_next[i] = *(const uint4_t *)(rows + (uint64_t)row * H + k);
            }
        }
    };
    const uint32_t expert_in_block = thread / 16u, pair = thread % 16u; /* chains 2 pair, 2 pair + 1 */
    float chain[PROJECTION_ROWS][2];
#pragma unroll
    for (uint32_t r = 0; r < PROJECTION_ROWS; r++) {
        chain[r][0] = chain[r][1] = 0.0f;
    }
    fetch(0u);
    for (uint32_t chunk = 0; chunk < H; chunk += PROJECTION_CHUNK) {
        __syncthreads(); /* the tile's readers of the chunk before are done */
#pragma unroll
        for (uint32_t i = 0; i < PROJECTION_W_LOADS; i++) {
            ((uint4_t *)&w_tile[0][0])[i * PROJECTION_THREADS + thread] = w_next[i];
        }
#pragma unroll
        for (uint32_t i = 0; i < PROJECTION_X_LOADS; i++) {
            ((uint4_t *)&x_tile[0][0])[i * PROJECTION_THREADS + thread] = x_next[i];
        }
        if (chunk + PROJECTION_CHUNK < H) {
            fetch(chunk + PROJECTION_CHUNK);
        }
        __syncthreads();
#pragma unroll 4
        for (uint32_t k = 0; k < PROJECTION_CHUNK; k += PROJECTION_CHAINS) {
            const uint32_t w = *(const uint32_t *)&w_tile[expert_in_block][k + 2u * pair];
            const float w0 = __uint_as_float(w << 16), w1 = __uint_as_float(w & 0xFFFF0000u);
#pragma unroll
            for (uint32_t r = 0; r < PROJECTION_ROWS; r++) {
                const uint32_t x = *(const uint32_t *)&x_tile[r][k + 2u * pair];
                chain[r][0] = __fmaf_rn(w0, __uint_as_float(x << 16), chain[r][0]);
                chain[r][1] = __fmaf_rn(w1, __uint_as_float(x & 0xFFFF0000u), chain[r][1]);
            }
        }
    }
    const uint32_t expert = first_expert + expert_in_block;
#pragma unroll
    for (uint32_t r = 0; r < PROJECTION_ROWS; r++) {
        float even = __fadd_rn(0.0f, chain[r][0]), odd = __fadd_rn(0.0f, chain[r][1]);
        /* chain c + distance lies distance / 2 threads on, for the distances 16, 8, 4, 2 */
        even = lanes_sum<1u>(lanes_sum<2u>(lanes_sum<4u>(lanes_sum<8u>(even))));
        odd = lanes_sum<1u>(lanes_sum<2u>(lanes_sum<4u>(lanes_sum<8u>(odd))));
        const float sum = __fadd_rn(even, odd); /* distance 1: chain 0 + chain 1 */
        if (pair == 0u && expert < arguments.expert_count && first_row + r < arguments.row_count) {
            ((float *)(arena + arguments.output_offset))[(uint64_t)(first_row + r) * arguments.expert_count + expert] = __fadd_rn(0.0f, sum);
        }
    }
}


typedef __attribute__((address_space(3))) void *lds_bytes;

/* 16 bytes a lane from memory straight into LDS (lane L lands at lds_base + 16 L). Written as assembly: the compiler keeps
 * no book on it, so the waits for it are written out where a stage is needed. */
__device__ static __forceinline__ void projection_load_to_lds(const void *lane_address, uint32_t lds_base)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(lane_address), "s"(lds_base) : "memory", "m0");
}

/* A thin step's form: a row a block, a wavefront two experts, a lane one chain. The inputs pass through LDS, straight from memory,
 * all THIN_CHUNK of them asked for at once, so that the launch waits for memory one time. A chain's inputs lie 64 bytes apart: the
 * LDS's transposing read gives a lane four of them (ds_read_b64_tr_b16: sixteen lanes name four rows of sixteen 16-bit values, and
 * lane i receives value i of each). A wavefront that has a vector unit to itself issues an instruction in six cycles whatever it
 * is and has fifteen LDS reads on their way at most, so both are what counts: by single reads of 16 bits 4.9 us, by these 4.0
 * (one row of 4096 inputs by 256 experts; two chains a lane, through registers and in chunks of 1024: 5.5; eight rows 5.6 -> 4.35,
 * eight of 5120 by 384 experts 7.2 -> 5.7, three of 2048 by 64 3.6 -> 3.0). A wider row is a chunk behind the other, no chunk on its
 * way while one is added, and still the faster: eight rows of 7168 by 256 8.35 -> 6.05, of 8192 9.3 -> 6.6, of 12288 by 384 14.75 -> 9.6,
 * of 16384 by 512 18.95 -> 12.4. A narrower one asks for the same 74 KB of LDS, two blocks a CU: eight of 512 by 256 2.75 -> 2.4, of
 * 1024 by 1024 (four blocks a CU in two rounds) 4.45 -> 4.35. grid (ceil(E / 8), rows), block 256. */
#define THIN_EXPERTS 2u /* of a wavefront */
#define THIN_CHUNK 4096u
#define THIN_ROW_VALUES (THIN_CHUNK + 32u) /* 64 bytes more: the two experts' chains lie on different banks */
#define THIN_LOADS (THIN_CHUNK / 512u) /* of a row's chunk: 64 lanes of eight values */
typedef short thin_values_t __attribute__((ext_vector_type(4)));
#define THIN_BATCH 16u /* groups of 32 inputs whose reads go together */
struct thin_batch {
    uint2_t w[THIN_BATCH / 4u], x[THIN_BATCH / 4u];
};

/* the inputs of THIN_BATCH groups of the lane's chain, of its expert and of the row */
__device__ static __forceinline__ void thin_read(uint32_t w_at, uint32_t x_at, struct thin_batch &into)
{
    typedef __attribute__((address_space(3))) thin_values_t *place;
#pragma unroll
    for (uint32_t k = 0; k < THIN_BATCH / 4u; k++) {
        into.w[k] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((place)(uintptr_t)(w_at + k * (4u * PROJECTION_CHAINS * 2u))));
        into.x[k] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((place)(uintptr_t)(x_at + k * (4u * PROJECTION_CHAINS * 2u))));
    }
}

/* the first `groups` of a batch into the chain */
__device__ static __forceinline__ float thin_add(const struct thin_batch &batch, uint32_t groups, float chain)
{
#pragma unroll
    for (uint32_t k = 0; k < THIN_BATCH; k++) {
        const uint32_t w = batch.w[k / 4u][k / 2u % 2u], x = batch.x[k / 4u][k / 2u % 2u];
        const float sum = k % 2u == 0u ? __fmaf_rn(__uint_as_float(w << 16), __uint_as_float(x << 16), chain)
                                       : __fmaf_rn(__uint_as_float(w & 0xFFFF0000u), __uint_as_float(x & 0xFFFF0000u), chain);
        chain = k < groups ? sum : chain;
    }
    return chain;
}

__device__ static __forceinline__ void router_projection_thin(const struct router_projection_arguments &arguments, unsigned char *arena)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char projection_window[]; /* PROJECTION_THIN_WINDOW_BYTES: the experts' rows, then the row's */
    static_assert((PROJECTION_EXPERTS + 1u) * THIN_ROW_VALUES * 2u == PROJECTION_THIN_WINDOW_BYTES, "the window the host asks for");
    const uint32_t H = arguments.hidden, lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t first_expert = blockIdx.x * PROJECTION_EXPERTS + wave * THIN_EXPERTS, chain_of = lane % PROJECTION_CHAINS, mine = lane / PROJECTION_CHAINS;
    const uint32_t window_address = (uint32_t)(uintptr_t)(lds_bytes)projection_window;
    const uint16_t *row = (const uint16_t *)(arena + arguments.rows_offset) + (uint64_t)blockIdx.y * H + 8u * lane;
    const uint16_t *weights[THIN_EXPERTS]; /* an expert past the last repeats the last: its score is not stored */
#pragma unroll
    for (uint32_t e = 0; e < THIN_EXPERTS; e++) {
        const uint32_t expert = first_expert + e < arguments.expert_count ? first_expert + e : arguments.expert_count - 1u;
        weights[e] = (const uint16_t *)(arena + arguments.weights_offset) + (uint64_t)expert * H + 8u * lane;
    }
    /* row lane % 16 / 4 of the four, sixteen chains of the 32, eight bytes a lane */
    const uint32_t lane_bytes = lane % 16u / 4u * (PROJECTION_CHAINS * 2u) + lane / 16u % 2u * 32u + lane % 4u * 8u;
    const uint32_t w_at = window_address + (wave * THIN_EXPERTS + mine) * (THIN_ROW_VALUES * 2u) + lane_bytes;
    const uint32_t x_at = window_address + PROJECTION_EXPERTS * (THIN_ROW_VALUES * 2u) + lane_bytes;
    float chain = 0.0f;
    for (uint32_t chunk = 0; chunk < H; chunk += THIN_CHUNK) {
        if (chunk != 0u) {
            __syncthreads(); /* the chunk before has been read */
        }
#pragma unroll
        for (uint32_t part = 0; part < THIN_LOADS; part++) {
            if (chunk + 512u * part + 8u * lane < H) { /* a width is a whole number of groups: no group is brought in part */
#pragma unroll
                for (uint32_t e = 0; e < THIN_EXPERTS; e++) {
                    projection_load_to_lds(weights[e] + chunk + 512u * part, window_address + ((wave * THIN_EXPERTS + e) * THIN_ROW_VALUES + 512u * part) * 2u);
                }
                if (part / (THIN_LOADS / (PROJECTION_EXPERTS / THIN_EXPERTS)) == wave) {
                    projection_load_to_lds(row + chunk + 512u * part, window_address + (PROJECTION_EXPERTS * THIN_ROW_VALUES + 512u * part) * 2u);
                }
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t groups = (H - chunk < THIN_CHUNK ? H - chunk : THIN_CHUNK) / PROJECTION_CHAINS;
        /* a batch is read while the one before it is added; past the chunk's last group the reads stay inside its place, and what
         * they give is not added (a width that is no whole 512) */
        constexpr uint32_t BATCH_BYTES = THIN_BATCH * PROJECTION_CHAINS * 2u;
        struct thin_batch batch[2];
        thin_read(w_at, x_at, batch[0]);
        for (uint32_t group = 0; group < groups; group += 2u * THIN_BATCH) {
            const uint32_t at = group * (PROJECTION_CHAINS * 2u);
            thin_read(w_at + at + BATCH_BYTES, x_at + at + BATCH_BYTES, batch[1]);
            if (group + THIN_BATCH <= groups) {
                chain = thin_add(batch[0], THIN_BATCH, chain);
            } else {
                chain = thin_add(batch[0], groups - group, chain);
            }
            if (group + THIN_BATCH >= groups) {
                break;
            }
            if (group + 2u * THIN_BATCH < groups) {
                thin_read(w_at + at + 2u * BATCH_BYTES, x_at + at + 2u * BATCH_BYTES, batch[0]);
            }
            if (group + 2u * THIN_BATCH <= groups) {
                chain = thin_add(batch[1], THIN_BATCH, chain);
            } else {
                chain = thin_add(batch[1], groups - group - THIN_BATCH, chain);
            }
        }
    }
    /* the fold, over the distances 16, 8, 4, 2 and 1 of the expert's 32 lanes */
    const float sum = lanes_sum<1u>(lanes_sum<2u>(lanes_sum<4u>(lanes_sum<8u>(lanes_sum<16u>(__fadd_rn(0.0f, chain))))));
    if (chain_of == 0u && first_expert + mine < arguments.expert_count) {
        ((float *)(arena + arguments.output_offset))[(uint64_t)blockIdx.y * arguments.expert_count + first_expert + mine] = __fadd_rn(0.0f, sum);
    }
}

extern "C" __global__ void __launch_bounds__(PROJECTION_THIN_THREADS)
    router_projection(struct router_projection_arguments arguments, unsigned char *arena)
{
    if (router_projection_by_row(arguments.row_count, arguments.expert_count)) { /* the same in every block */
        router_projection_thin(arguments, arena);
    } else {
        router_projection_block(arguments, arena);
    }
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_projection, router_projection_arguments);

/* The same scores on the matrix unit, for steps of many rows. v_mfma_f32_16x16x1_4b_f32 adds, to each of four 16 x 16
 * blocks of sums, one product a sum, each a fused multiply-add of float32 rounded once (compared bit for bit with
 * fmaf over wide exponent ranges, subnormal products and infinities): a block is a chain, its 16 x 16 sums the chains
 * of 16 experts by 16 rows, and the eight instructions of a group of 32 inputs advance the 32 chains by one input
 * each, in the definition's order. Instruction q takes the chains 8 b + q of the blocks b = 0 .. 3, so that lane
 * (b, n) needs the inputs 32 i + 8 b + {0 .. 7} of expert n (and of row n): one 16-byte piece each a group. The fold is
 * inside a lane. grid (E / 16, ceil(rows / 64)), block 256: a wavefront 16 rows.
 *
 * The pieces pass through LDS. Read by the lanes that use them they would be 64 bytes of each of sixteen rows an
 * instruction, rows a power of two apart: half-used lines that fall into the same few sets of the first-level cache, and
 * the wavefronts waited for them three quarters of their time. Instead a stage of PROJECTION_STAGE_INPUTS inputs of the
 * block's 16 experts and 64 rows (80 rows of 256 bytes) is brought by 20 loads of a wavefront that go from memory
 * straight into LDS, each 256 contiguous bytes of four rows; piece p of tile row R lies at slot p ^ (R % 16) of its row,
 * so that the eight lanes of a 16-byte read (eight rows, one piece) meet eight different bank groups. Two stages (40 KB:
 * three blocks a CU, which measured faster than three stages and two blocks): the next stage is asked for behind the
 * barrier that ends the stage before the current one. */
typedef __attribute__((ext_vector_type(16))) float float16_t;
#define PROJECTION_STAGE_ROW_BYTES (PROJECTION_STAGE_INPUTS * 2u)
#define PROJECTION_STAGE_ROWS (16u + PROJECTION_TILE_ROWS)
#define PROJECTION_STAGE_BYTES (PROJECTION_STAGE_ROWS * PROJECTION_STAGE_ROW_BYTES)
#define PROJECTION_STAGES 2u
#define PROJECTION_WAVE_LOADS (PROJECTION_STAGE_BYTES / 1024u / (PROJECTION_TILE_THREADS / WAVE)) /* 5 */

/* COUNT words of two bfloat16 each as float32. The float32 matrix instruction runs on the vector unit's own multipliers:
 * nothing else of the unit runs beside it, and every change between the two costs cycles of its own. By a probe of this
 * instruction (33.2 cycles alone, at one to three wavefronts a SIMD alike): 57 cycles with its two operands converted in
 * front of it, 53 with those of a later instruction converted behind it, 42 where the operands of eight instructions are
 * converted together and then multiplied. So conversions and matrix instructions go in blocks, fenced from each other. */
template <uint32_t COUNT>
__device__ static __forceinline__ void projection_convert(const uint32_t (&words)[COUNT], float (&values)[2u * COUNT])
{
#pragma unroll
    for (uint32_t k = 0; k < 2u * COUNT; k++) {
        values[k] = __uint_as_float(k % 2u == 0u ? words[k / 2u] << 16 : words[k / 2u] & 0xFFFF0000u);
        asm volatile("" : "+v"(values[k]));
    }
}

extern "C" __global__ void __launch_bounds__(PROJECTION_TILE_THREADS, 3) /* three blocks a CU */
    router_projection_tiles(struct router_projection_arguments arguments, unsigned char *arena)
{
    __shared__ __attribute__((aligned(1024))) unsigned char window[PROJECTION_STAGES * PROJECTION_STAGE_BYTES];
    const uint32_t lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), block = lane / 16u, index = lane % 16u;
    const uint32_t H = arguments.hidden, groups = H / PROJECTION_CHAINS;
    const uint32_t stages = groups / 4u; /* whole stages: whoever prepares the launch holds the width to a multiple of PROJECTION_STAGE_INPUTS */
    const uint32_t first_expert = blockIdx.x * 16u, block_row = blockIdx.y * PROJECTION_TILE_ROWS, first_row = block_row + wave * 16u;
    const uint32_t window_address = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)window;
    /* what this wavefront brings of a stage: the loads wave, wave + 4, ...; load d is the tile rows 4 d .. 4 d + 3 (the
     * experts' rows first, then the block's rows; a row past the last repeats the last: its sums are not stored) */
    const unsigned char *source[PROJECTION_WAVE_LOADS];
    uint32_t piece_bytes[PROJECTION_WAVE_LOADS];
#pragma unroll
    for (uint32_t part = 0; part < PROJECTION_WAVE_LOADS; part++) {
        const uint32_t tile_row = 4u * (wave + 4u * part) + lane / 16u;
        piece_bytes[part] = 16u * ((lane % 16u) ^ (tile_row % 16u));
        if (tile_row < 16u) {
            source[part] = arena + arguments.weights_offset + (uint64_t)(first_expert + tile_row) * H * 2u;
        } else {
            const uint32_t row = block_row + tile_row - 16u;
            source[part] = arena + arguments.rows_offset + (uint64_t)(row < arguments.row_count ? row : arguments.row_count - 1u) * H * 2u;
        }
    }
    auto ask = [&](uint32_t stage) {
        const uint32_t base = window_address + (stage % PROJECTION_STAGES) * PROJECTION_STAGE_BYTES;
#pragma unroll
        for (uint32_t part = 0; part < PROJECTION_WAVE_LOADS; part++) {
            projection_load_to_lds(source[part] + stage * PROJECTION_STAGE_ROW_BYTES + piece_bytes[part], base + (wave + 4u * part) * 1024u);
        }
    };
    /* where lane (b, n) reads its pieces of group i of a stage: piece 4 i + b of expert n and of the wavefront's row n */
    uint32_t w_at[4], x_at[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const uint32_t slot = 16u * ((4u * i + block) ^ index);
        w_at[i] = index * PROJECTION_STAGE_ROW_BYTES + slot;
        x_at[i] = (16u + 16u * wave + index) * PROJECTION_STAGE_ROW_BYTES + slot;
    }
    float16_t chain[8];
#pragma unroll
    for (uint32_t q = 0; q < 8u; q++) {
#pragma unroll
        for (uint32_t v = 0; v < 16u; v++) {
            chain[q][v] = 0.0f;
        }
    }
    ask(0u);
    for (uint32_t stage = 0; stage < stages; stage++) {
        /* this wavefront's loads of the stage have landed, then every wavefront's; behind the barrier every wavefront is
         * through the stage before, whose window the next stage takes */
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (stage + 1u < stages) {
            ask(stage + 1u);
        }
        const unsigned char *now = window + (stage % PROJECTION_STAGES) * PROJECTION_STAGE_BYTES;
        uint4_t w_now = *(const uint4_t *)(now + w_at[0]), x_now = *(const uint4_t *)(now + x_at[0]);
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) { /* a group of 32 inputs: eight instructions, each one input further on the four chains it takes */
            const uint32_t w_words[4] = {w_now.x, w_now.y, w_now.z, w_now.w}, x_words[4] = {x_now.x, x_now.y, x_now.z, x_now.w};
            float w_values[8], x_values[8];
            /* the further a wavefront is into its stage, the more its instructions go first: the three of a SIMD then wait for LDS
             * and the barrier at different times (8192 rows of 4096 inputs by 256 experts 219 -> 210 us, 2048 rows 66 -> 62) */
            if (i == 0u) {
                __builtin_amdgcn_s_setprio(0);
            } else if (i == 1u) {
                __builtin_amdgcn_s_setprio(1);
            } else if (i == 2u) {
                __builtin_amdgcn_s_setprio(2);
            } else {
                __builtin_amdgcn_s_setprio(3);
            }
            projection_convert(w_words, w_values);
            projection_convert(x_words, x_values);
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1u < 4u) { /* the next group's pieces are on their way behind this group's instructions */
                w_now = *(const uint4_t *)(now + w_at[i + 1u]);
                x_now = *(const uint4_t *)(now + x_at[i + 1u]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t q = 0; q < 8u; q++) {
                chain[q] = __builtin_amdgcn_mfma_f32_16x16x1f32(w_values[q], x_values[q], chain[q], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    /* register v = 4 b + r of chain[q] is chain 8 b + q of expert 4 (lane / 16) + r and row lane % 16. The fold, as the
     * definition orders it: + 0 first, then the distances 16 and 8 (blocks), 4, 2 and 1 (instructions) */
    float sums[8][8];
#pragma unroll
    for (uint32_t q = 0; q < 8u; q++) {
#pragma unroll
        for (uint32_t v = 0; v < 8u; v++) {
            sums[q][v] = __fadd_rn(__fadd_rn(0.0f, chain[q][v]), __fadd_rn(0.0f, chain[q][v + 8u]));
        }
#pragma unroll
        for (uint32_t r = 0; r < 4u; r++) {
            sums[q][r] = __fadd_rn(sums[q][r], sums[q][r + 4u]);
        }
    }
#pragma unroll
    for (uint32_t distance = 4u; distance != 0u; distance >>= 1u) {
#pragma unroll
        for (uint32_t q = 0; q < distance; q++) {
#pragma unroll
            for (uint32_t r = 0; r < 4u; r++) {
                sums[q][r] = __fadd_rn(sums[q][r], sums[q + distance][r]);
            }
        }
    }
    if (first_row + index < arguments.row_count) {
        float *out = (float *)(arena + arguments.output_offset) + (uint64_t)(first_row + index) * arguments.expert_count + first_expert + 4u * block;
        *(float4_t *)out = (float4_t){__fadd_rn(0.0f, sums[0][0]), __fadd_rn(0.0f, sums[0][1]), __fadd_rn(0.0f, sums[0][2]), __fadd_rn(0.0f, sums[0][3])};
    }
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_projection_tiles, router_projection_arguments);

/* The same scores for steps whose tiles of 16 experts by 64 rows leave CUs idle or unevenly loaded (which those are:
 * PROJECTION_SPLIT_BLOCKS_OF_TILE, with both forms' times): a block is one 16 x 16 tile, and its eight wavefronts take four
 * chains each, so that a CU's four vector units work on every score, two wavefronts a unit. The instruction of a group of 32
 * inputs takes the chains 4 wave + b of the blocks b = 0 .. 3: lane (b, n) needs the input 32 i + 4 wave + b of expert n and of
 * row n, 16 bits each, which LDS reads into the upper half of a register whose lower half is zero: a float32, and no conversion
 * that the matrix instruction would wait for. A stage is the 16 + 16 rows' 128 inputs (8 KB, laid out and swizzled as above, a
 * load a wavefront). Stages go in pairs, a barrier a pair; three pairs are in LDS or on their way (three blocks a CU), and a stage
 * is read behind the instructions of the one before it. The wavefronts' sums meet in LDS at the end, half of them folding the
 * scores. What bounds it: a unit's 256 instructions of 4096 inputs, 33 cycles each, beside 64 LDS reads a stage; the first loads'
 * way from memory; the launch. By four wavefronts of eight chains, words converted and a barrier a stage | so, us, 256 experts of
 * 4096 inputs: 32 rows 10.6 | 9.2, 203 rows 10.75 | 9.4, 300 rows 15.2 | 14.2, 700 rows 21.2 | 19.5 (eight wavefronts with a
 * barrier a stage 9.95 at 32 rows and 22.6 at 700). grid (E / 16, ceil(rows / 16)), block (256, 2): 512 threads, the 256
 * of y = 0 bring the experts' rows of the tile, those of y = 1 the rows. */
#define PROJECTION_SPLIT_STAGE_BYTES (32u * PROJECTION_STAGE_ROW_BYTES)
#define PROJECTION_SPLIT_PAIRS 3u
#define PROJECTION_SPLIT_WAVES (PROJECTION_SPLIT_SIDES * PROJECTION_TILE_THREADS / WAVE)
struct split_inputs {
    float w[4], x[4]; /* of a stage's four groups; the lower halves stay zero */
};

/* A stage's inputs out of LDS: asked for here, there behind split_landed. Assembly, as the compiler has no read of this form; it
 * takes the registers for filled where they are asked for, and one that it copied or saved in between would be taken before it
 * is filled. So the two stand in one run of instructions without a branch or a loop's end between them, with nothing but the
 * matrix instructions of the other set, and the build refuses the kernel if it spills a vector register. */
template <uint32_t STAGE> __device__ static __forceinline__ void split_read(const uint32_t (&at)[4], uint32_t place, struct split_inputs &into)
{
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const uint32_t from = at[i] + place;
        asm volatile("ds_read_u16_d16_hi %0, %1 offset:%2" : "+v"(into.w[i]) : "v"(from), "n"(STAGE * PROJECTION_SPLIT_STAGE_BYTES) : "memory");
        asm volatile("ds_read_u16_d16_hi %0, %1 offset:%2" : "+v"(into.x[i]) : "v"(from), "n"(STAGE * PROJECTION_SPLIT_STAGE_BYTES + 4096u) : "memory");
    }
}

__device__ static __forceinline__ void split_landed(struct split_inputs &inputs)
{
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(inputs.w[0]), "+v"(inputs.w[1]), "+v"(inputs.w[2]), "+v"(inputs.w[3]), "+v"(inputs.x[0]), "+v"(inputs.x[1]), "+v"(inputs.x[2]),
                   "+v"(inputs.x[3])
                 :
                 : "memory");
}

extern "C" __global__ void __launch_bounds__(PROJECTION_SPLIT_SIDES * PROJECTION_TILE_THREADS)
    router_projection_split(struct router_projection_arguments arguments, unsigned char *arena)
{
    constexpr uint32_t PAIR_BYTES = 2u * PROJECTION_SPLIT_STAGE_BYTES;
    __shared__ __attribute__((aligned(1024))) unsigned char window[PROJECTION_SPLIT_PAIRS * PAIR_BYTES];
    const uint32_t lane = threadIdx.x % WAVE, block = lane / 16u, index = lane % 16u;
    const uint32_t side = __builtin_amdgcn_readfirstlane(threadIdx.y), of_side = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t wave = PROJECTION_TILE_THREADS / WAVE * side + of_side;
    const uint32_t H = arguments.hidden, stages = H / PROJECTION_STAGE_INPUTS;
    const uint32_t first_expert = blockIdx.x * 16u, first_row = blockIdx.y * 16u;
    const uint32_t window_address = (uint32_t)(uintptr_t)(lds_bytes)window;
    /* this wavefront brings four experts' rows of a stage (side 0) or four rows (a row past the last repeats the last) */
    const uint32_t line = 4u * of_side + lane / 16u, last_row = arguments.row_count - 1u - first_row;
    const unsigned char *base = arena + (side == 0u ? arguments.weights_offset + (uint64_t)first_expert * H * 2u : arguments.rows_offset + (uint64_t)first_row * H * 2u);
    const uint32_t own = 16u * ((lane % 16u) ^ line) + (side == 0u || line < last_row ? line : last_row) * (H * 2u);
    const uint32_t lands_at = window_address + wave * 1024u;
    /* a stage past the last is the last again, into a place that nobody reads any more: every wait counts the same */
    auto ask = [&](uint32_t pair, uint32_t place) {
        const uint32_t one = 2u * pair < stages ? 2u * pair : stages - 1u, two = 2u * pair + 1u < stages ? 2u * pair + 1u : stages - 1u;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %3"
                     : : "s"(lands_at + place), "s"(lands_at + place + PROJECTION_SPLIT_STAGE_BYTES), "v"(own + one * PROJECTION_STAGE_ROW_BYTES), "s"(base),
                       "v"(own + two * PROJECTION_STAGE_ROW_BYTES) : "memory", "m0");
    };
    for (uint32_t pair = 0; pair < PROJECTION_SPLIT_PAIRS; pair++) {
        ask(pair, pair * PAIR_BYTES);
    }
    float16_t chain;
#pragma unroll
    for (uint32_t v = 0; v < 16u; v++) {
        chain[v] = 0.0f;
    }
    /* input 32 i + 4 wave + block of line `index`: piece 4 i + wave / 2, its value 4 (wave % 2) + block */
    uint32_t at[4];
    struct split_inputs inputs[2];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        at[i] = window_address + index * PROJECTION_STAGE_ROW_BYTES + 16u * ((4u * i + wave / 2u) ^ index) + 2u * (4u * (wave % 2u) + block);
        inputs[0].w[i] = inputs[0].x[i] = inputs[1].w[i] = inputs[1].x[i] = 0.0f;
    }
    /* this wavefront's loads of the first pair have landed, then every wavefront's */
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2u * (PROJECTION_SPLIT_PAIRS - 1u)) : "memory");
    __syncthreads();
    const auto multiply = [&](const struct split_inputs &of) {
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            chain = __builtin_amdgcn_mfma_f32_16x16x1f32(of.w[i], of.x[i], chain, 0, 0, 0);
        }
    };
    split_read<0>(at, 0u, inputs[0]);
    split_landed(inputs[0]);
    uint32_t place = 0;
    for (uint32_t pair = 0; pair < stages / 2u; pair++) {
        split_read<1>(at, place, inputs[1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(inputs[0]);
        __builtin_amdgcn_sched_barrier(0);
        /* every wavefront has read the pair, whose place the one to ask for takes; the next pair has landed */
        split_landed(inputs[1]);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2u * (PROJECTION_SPLIT_PAIRS - 2u)) : "memory");
        __syncthreads();
        ask(pair + PROJECTION_SPLIT_PAIRS, place);
        place = place + PAIR_BYTES < PROJECTION_SPLIT_PAIRS * PAIR_BYTES ? place + PAIR_BYTES : 0u;
        split_read<0>(at, place, inputs[0]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(inputs[1]);
        __builtin_amdgcn_sched_barrier(0);
        split_landed(inputs[0]);
    }
    if (stages % 2u != 0u) { /* a last stage alone */
        multiply(inputs[0]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* the last pairs' repeats */
    __syncthreads();
    /* register v = 4 b + r is chain 4 wave + b of expert 4 (lane / 16) + r and row lane % 16. Every wavefront leaves its four
     * chains of the experts r; wavefront r then folds those of expert 4 (lane / 16) + r as the definition orders it: + 0 first, then
     * the distances 16, 8 and 4 (wavefronts), 2 and 1 (blocks) */
    float4_t *exchange = (float4_t *)window; /* [wavefront][r][lane] */
#pragma unroll
    for (uint32_t r = 0; r < 4u; r++) {
        exchange[(wave * 4u + r) * WAVE + lane] = (float4_t){__fadd_rn(0.0f, chain[r]), __fadd_rn(0.0f, chain[4u + r]), __fadd_rn(0.0f, chain[8u + r]),
                                                             __fadd_rn(0.0f, chain[12u + r])};
    }
    __syncthreads();
    if (side != 0u || first_row + index >= arguments.row_count) {
        return;
    }
    float4_t part[PROJECTION_SPLIT_WAVES];
#pragma unroll
    for (uint32_t from = 0; from < PROJECTION_SPLIT_WAVES; from++) {
        part[from] = exchange[(from * 4u + wave) * WAVE + lane];
    }
#pragma unroll
    for (uint32_t distance = PROJECTION_SPLIT_WAVES / 2u; distance != 0u; distance >>= 1u) {
#pragma unroll
        for (uint32_t from = 0; from < distance; from++) {
#pragma unroll
            for (uint32_t b = 0; b < 4u; b++) {
                part[from][b] = __fadd_rn(part[from][b], part[from + distance][b]);
            }
        }
    }
    const float sum = __fadd_rn(__fadd_rn(part[0][0], part[0][2]), __fadd_rn(part[0][1], part[0][3]));
    ((float *)(arena + arguments.output_offset))[(uint64_t)(first_row + index) * arguments.expert_count + first_expert + 4u * block + wave] = __fadd_rn(0.0f, sum);
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_projection_split, router_projection_arguments);

extern "C" __global__ void __launch_bounds__(SELECT_THREADS)
    router_select_entry(struct router_select_arguments arguments, unsigned char *arena)
{
    __shared__ struct router_select_lds lds;
    router_select_body(arguments, arena, threadIdx.x, SELECT_THREADS, lds);
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_select_entry, router_select_arguments);

/* ---- the wide select: rows of a prefill, sorted by expert ------------------------------------------------------
 * Four launches of one record, in this order (include/anemone/router_records.h:31-47 of the reference; the kernels
 * at source/kernel_router.cu:97-459 there): the picks of every live row; the pairs of each expert counted in blocks
 * of ROUTER_SORT_ROWS rows; every pair placed (a pair's place: the pairs of lower experts, and of its expert in
 * lower rows), the runs and the tiles of at most 64 pairs; the job table of at most 8 pairs a job. The only atomic
 * operations count in LDS; the order is the rows' (sort_device.cuh). */
#define WIDE_SORT_THREADS 512u

__device__ static __forceinline__ uint32_t wide_live_rows(const struct router_wide_arguments &arguments, const unsigned char *arena)
{
    const uint32_t step_rows = ((const struct step_block *)(arena + arguments.step_offset))->row_count;
    return step_rows < arguments.row_count ? step_rows : arguments.row_count;
}

/* a lane's values of a row: its `places` experts lie next to each other, from lane * places on (0 past them) */
__device__ static __forceinline__ void router_lane_values(const float *row, uint32_t lane, uint32_t places, float (&values)[ROUTER_PLACES])
{
    typedef float4_t float4_of_words __attribute__((aligned(4)));
    float4_t four = {0.0f, 0.0f, 0.0f, 0.0f};
    if (places == 4u) {
        four = ((const float4_of_words *)row)[lane];
    }
#pragma unroll
    for (uint32_t place = 0; place < ROUTER_PLACES; place++) {
        values[place] = place < 4u ? four[place % 4u] : 0.0f;
        if (places != 4u && place < places) {
            values[place] = row[lane * places + place];
        }
    }
}

/* a row from its scores on: the affinities (LDS and memory), the keys, the picks. places: PLACES, or fewer, where the lane's
 * others hold key 0 and are never taken */
template <uint32_t PLACES>
__device__ static __forceinline__ void router_row_of_scores(const float (&scores)[ROUTER_PLACES], const float (&bias)[ROUTER_PLACES],
                                                            float *affinities, float *affinities_out, uint32_t lane, uint32_t places, uint32_t affinity_kind,
                                                            uint32_t picks, uint32_t reference_order, float route_scale, uint32_t &expert_out,
                                                            float &weight_out)
{
    uint32_t keys[PLACES];
#pragma unroll
    for (uint32_t place = 0; place < PLACES; place++) {
        keys[place] = 0u;
        if (place < places) {
            const float a = router_affinity(scores[place], affinity_kind);
            affinities[lane * places + place] = a;
            affinities_out[lane * places + place] = a;
            keys[place] = router_key(__fadd_rn(a, bias[place]));
        }
    }
    router_row<PLACES>(affinities, keys, lane, places, picks, reference_order, route_scale, expert_out, weight_out);
}

/* grid (ceil(row_count / 8)), a wavefront a row: its affinities, as the select writes them, and its picks by slot */
extern "C" __global__ void __launch_bounds__(SELECT_THREADS)
    router_wide_select(struct router_wide_arguments arguments, unsigned char *arena)
{
    __shared__ float affinities[LINEAR_MAXIMUM_ROWS * ROUTER_MOST_EXPERTS];
    const uint32_t experts = arguments.expert_count, picks = arguments.pick_count, places = experts / WAVE;
    const uint32_t wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const uint32_t row = blockIdx.x * LINEAR_MAXIMUM_ROWS + wave;
    /* asked for together: the step's rows, the lane's bias values and scores (the row is inside the scores' array or the
     * wavefront reads row 0's) */
    const uint32_t live_rows = wide_live_rows(arguments, arena);
    const uint64_t first = (uint64_t)(row < arguments.row_count ? row : 0u) * experts;
    float bias_of[ROUTER_PLACES], scores[ROUTER_PLACES];
    router_lane_values((const float *)(arena + arguments.bias_offset), lane, places, bias_of);
    router_lane_values((const float *)(arena + arguments.scores_offset) + first, lane, places, scores);
    if (row >= live_rows) {
        return; /* no barrier in this kernel: a wavefront is a row */
    }
    struct router_pick my_pick;
    float *own = affinities + wave * experts, *out = (float *)(arena + arguments.affinities_offset) + first;
    router_by_places(places, [&](auto count) {
        router_row_of_scores<count.value>(scores, bias_of, own, out, lane, places, arguments.affinity_kind, picks, arguments.reference_order,
                                          arguments.route_scale, my_pick.expert, my_pick.route_weight);
    });
    if (lane < picks) { /* lane s holds the pick of slot s */
        ((struct router_pick *)(arena + arguments.picks_offset))[(uint64_t)row * picks + lane] = my_pick;
    }
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_wide_select, router_wide_arguments);

/* the picked experts of the live rows of block `block` of ROUTER_SORT_ROWS rows, into LDS; returns their number */
__device__ static __forceinline__ uint32_t wide_block_picks(const struct router_wide_arguments &arguments, const unsigned char *arena,
                                                            uint32_t block, uint32_t live_rows, uint32_t *experts_out)
{
    return sort_block_picks((const struct router_pick *)(arena + arguments.picks_offset), arguments.pick_count, block, live_rows, experts_out);
}

/* grid (ceil(row_count / ROUTER_SORT_ROWS)): counts [block][E] */
extern "C" __global__ void __launch_bounds__(WIDE_SORT_THREADS)
    router_wide_count(struct router_wide_arguments arguments, unsigned char *arena)
{
    __shared__ __attribute__((aligned(16))) uint32_t block_experts[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    const uint32_t live_rows = wide_live_rows(arguments, arena);
    const uint32_t pairs = wide_block_picks(arguments, arena, blockIdx.x, live_rows, block_experts);
    __syncthreads();
    if (pairs == 0u) {
        return; /* a block of no live row writes nothing; the place reads no count of it */
    }
    __shared__ uint32_t histogram[ROUTER_MOST_EXPERTS];
    sort_count_picks(block_experts, pairs, arguments.expert_count, histogram);
    uint32_t *counts = (uint32_t *)(arena + arguments.counts_offset) + (uint64_t)blockIdx.x * arguments.expert_count;
    for (uint32_t expert = threadIdx.x; expert < arguments.expert_count; expert += WIDE_SORT_THREADS) {
        counts[expert] = histogram[expert];
    }
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_wide_count, router_wide_arguments);

/* What a block of the place does once it holds, in LDS, its picks (block_experts, `pairs` of them) and of every expert
 * the pairs of all blocks (totals; starts a copy of them), those of the blocks before this one (before) and its
 * tiles (tile_starts): the sorted pairs of the block's rows; block 0 also the runs and every tile. The whole block
 * calls it after a barrier. */
__device__ static __forceinline__ void wide_place_block(const struct router_wide_arguments &arguments, unsigned char *arena, uint32_t block,
                                                        const uint32_t *block_experts, uint32_t *place_of, uint32_t pairs, uint32_t *totals,
                                                        uint32_t *starts, const uint32_t *before, uint32_t *tile_starts, uint32_t *scratch,
                                                        uint32_t *first_places, uint32_t *cursors)
{
    const uint32_t experts = arguments.expert_count, picks = arguments.pick_count;
    (void)block_exclusive_scan(starts, experts, scratch);
    const struct router_pick *all_picks = (const struct router_pick *)(arena + arguments.picks_offset);
    struct wide_pair *sorted = (struct wide_pair *)(arena + arguments.pairs_offset);
    const uint32_t first_pair = block * ROUTER_SORT_ROWS * picks;
    /* every pick's place into LDS; the pairs are written behind it, a thread a pick */
    for (uint32_t expert = threadIdx.x; expert < experts; expert += WIDE_SORT_THREADS) {
        first_places[expert] = starts[expert] + before[expert];
    }
    __syncthreads();
    sort_place_picks(block_experts, pairs, experts, first_places, cursors, place_of);
    for (uint32_t index = threadIdx.x; index < pairs; index += WIDE_SORT_THREADS) {
        sorted[place_of[index]] = (struct wide_pair){first_pair + index, all_picks[first_pair + index].route_weight};
    }
    if (block != 0u) {
        return;
    }
    struct wide_run *runs = (struct wide_run *)(arena + arguments.runs_offset);
    for (uint32_t expert = threadIdx.x; expert < experts; expert += WIDE_SORT_THREADS) {
        runs[expert] = (struct wide_run){starts[expert], totals[expert]};
    }
    const uint32_t used_tiles = block_exclusive_scan(tile_starts, experts, scratch);
    if (threadIdx.x == 0u) {
        tile_starts[experts] = used_tiles;
    }
    __syncthreads();
    const uint32_t all_tiles = ROUTER_WIDE_TILES_OF(arguments.row_count, picks, experts);
    struct wide_expert_tile *tiles = (struct wide_expert_tile *)(arena + arguments.tiles_offset);
    const uint64_t *offsets = (const uint64_t *)(arena + arguments.expert_offsets_offset);
    for (uint32_t tile = threadIdx.x; tile < all_tiles; tile += WIDE_SORT_THREADS) {
        struct wide_expert_tile value = {0, 0, 0, 0, 0};
        if (tile < used_tiles) {
            uint32_t low = 0, high = experts; /* the expert whose tiles hold this one: tile_starts[e] <= tile < [e + 1] */
            while (high - low > 1u) {
                const uint32_t middle = (low + high) / 2u;
                if (tile_starts[middle] <= tile) {
                    low = middle;
                } else {
                    high = middle;
                }
            }
            const uint32_t taken = (tile - tile_starts[low]) * WIDE_TILE_PAIRS, left = totals[low] - taken;
            value.gate_offset = offsets[(uint64_t)low * MODEL_EXPERT_MATRICES + 0u];
            value.up_offset = offsets[(uint64_t)low * MODEL_EXPERT_MATRICES + 1u];
            value.down_offset = offsets[(uint64_t)low * MODEL_EXPERT_MATRICES + 2u];
            value.first_pair = starts[low] + taken;
            value.pair_count = left < WIDE_TILE_PAIRS ? left : WIDE_TILE_PAIRS;
        }
        tiles[tile] = value;
    }
}

/* block `block` of a grid as the count's: the sorted pairs of the block's rows; block 0 also the runs and every tile */
__device__ static __forceinline__ void wide_place(const struct router_wide_arguments &arguments, unsigned char *arena, uint32_t block)
{
    __shared__ __attribute__((aligned(16))) uint32_t block_experts[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    __shared__ uint32_t place_of[ROUTER_SORT_ROWS * ROUTER_MOST_PICKS];
    __shared__ uint32_t totals[ROUTER_MOST_EXPERTS], starts[ROUTER_MOST_EXPERTS], before[ROUTER_MOST_EXPERTS];
    __shared__ uint32_t tile_starts[ROUTER_MOST_EXPERTS + 1u], scratch[SORT_MOST_WAVES];
    __shared__ uint32_t first_places[ROUTER_MOST_EXPERTS], cursors[SORT_MOST_WAVES * ROUTER_MOST_EXPERTS];
    const uint32_t experts = arguments.expert_count;
    const uint32_t live_rows = wide_live_rows(arguments, arena);
    const uint32_t live_blocks = (live_rows + ROUTER_SORT_ROWS - 1u) / ROUTER_SORT_ROWS;
    const uint32_t pairs = wide_block_picks(arguments, arena, block, live_rows, block_experts);
    if (pairs == 0u && block != 0u) {
        return;
    }
    const uint32_t *counts = (const uint32_t *)(arena + arguments.counts_offset);
    for (uint32_t expert = threadIdx.x; expert < experts; expert += WIDE_SORT_THREADS) {
        uint32_t total = 0, lower = 0;
#pragma unroll 8
        for (uint32_t other = 0; other < live_blocks; other++) {
            const uint32_t count = counts[(uint64_t)other * experts + expert];
            total += count;
            lower += other < block ? count : 0u;
        }
        totals[expert] = total;
        starts[expert] = total;
        before[expert] = lower;
        tile_starts[expert] = (total + WIDE_TILE_PAIRS - 1u) / WIDE_TILE_PAIRS;
    }
    __syncthreads();
    wide_place_block(arguments, arena, block, block_experts, place_of, pairs, totals, starts, before, tile_starts, scratch, first_places,
                     cursors);
}

extern "C" __global__ void __launch_bounds__(WIDE_SORT_THREADS)
    router_wide_place(struct router_wide_arguments arguments, unsigned char *arena)
{
    wide_place(arguments, arena, blockIdx.x);
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_wide_place, router_wide_arguments);

/* Job `job` of an expert whose jobs begin at job_start and whose `total` pairs begin at first_pair of the sorted pairs:
 * pair(place, index, weight) reads one. The eight reads go together (those past the job's pairs repeat its first). */
template <typename PAIR>
__device__ static __forceinline__ void wide_job(uint32_t job, uint32_t job_start, uint32_t expert, uint32_t first_pair, uint32_t total,
                                                const uint64_t *offsets, struct expert_job_record &value, PAIR pair)
{
    const uint32_t taken = (job - job_start) * LINEAR_MAXIMUM_ROWS, left = total - taken;
    value.gate_offset = offsets[0];
    value.up_offset = offsets[1];
    value.down_offset = offsets[2];
    value.row_count = left < LINEAR_MAXIMUM_ROWS ? left : LINEAR_MAXIMUM_ROWS;
    value.expert = expert;
#pragma unroll
    for (uint32_t column = 0; column < LINEAR_MAXIMUM_ROWS; column++) {
        uint32_t index;
        float weight;
        pair(first_pair + taken + (column < value.row_count ? column : 0u), index, weight);
        value.pair_index[column] = column < value.row_count ? index : 0u;
        value.route_weight[column] = column < value.row_count ? weight : 0.0f;
    }
}

/* grid (1): the job table of the runs, a thread a job */
extern "C" __global__ void __launch_bounds__(WIDE_SORT_THREADS)
    router_wide_jobs(struct router_wide_arguments arguments, unsigned char *arena)
{
    __shared__ uint32_t job_starts[ROUTER_MOST_EXPERTS + 1u], scratch[SORT_MOST_WAVES];
    const uint32_t experts = arguments.expert_count;
    const struct wide_run *runs = (const struct wide_run *)(arena + arguments.runs_offset);
    if (threadIdx.x < experts) {
        job_starts[threadIdx.x] = (runs[threadIdx.x].pair_count + LINEAR_MAXIMUM_ROWS - 1u) / LINEAR_MAXIMUM_ROWS;
    }
    __syncthreads();
    const uint32_t used_jobs = block_exclusive_scan(job_starts, experts, scratch);
    const uint32_t all_jobs = ROUTER_WIDE_JOBS_OF(arguments.row_count, arguments.pick_count, experts);
    const struct wide_pair *sorted = (const struct wide_pair *)(arena + arguments.pairs_offset);
    const uint64_t *offsets = (const uint64_t *)(arena + arguments.expert_offsets_offset);
    struct expert_job_record *jobs = (struct expert_job_record *)(arena + arguments.jobs_offset);
    for (uint32_t job = threadIdx.x; job < all_jobs; job += WIDE_SORT_THREADS) {
        struct expert_job_record value = {};
        if (job < used_jobs) {
            uint32_t low = 0, high = experts;
            while (high - low > 1u) {
                const uint32_t middle = (low + high) / 2u;
                if (job_starts[middle] <= job) {
                    low = middle;
                } else {
                    high = middle;
                }
            }
            const struct wide_run run = runs[low];
            wide_job(job, job_starts[low], low, run.first_pair, run.pair_count, offsets + (uint64_t)low * MODEL_EXPERT_MATRICES, value,
                     [&](uint32_t place, uint32_t &index, float &weight) {
                         const struct wide_pair pair = sorted[place];
                         index = pair.pair_index;
                         weight = pair.route_weight;
                     });
        }
        jobs[job] = value;
    }
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_wide_jobs, router_wide_arguments);

/* grid (1): the count, the place and the jobs of at most ROUTER_SORT_ROWS rows in one block (the reference's
 * router_wide_small, source/kernel_router.cu there): the same pairs, runs, tiles and jobs; the counts scratch is
 * not written.
 *
 * One block's time is its round trips: everything it reads from memory is asked for at its start (the picks of all the rows
 * there is room for, beside the number of the live ones), a thread owns an expert and takes the starts of its pairs, tiles
 * and jobs from one scan of the three side by side, the jobs find their expert and their pairs in LDS: five barriers, two
 * waits for memory. 64 rows of 256 experts, 8 picks: 17.4 -> 6.0 us (three scans of nine barriers, searches, the runs and
 * the sorted pairs read back from memory, a job's pairs by way of scratch memory). */
__device__ static __forceinline__ void wide_small(const struct router_wide_arguments &arguments, unsigned char *arena)
{
    constexpr uint32_t MOST_PAIRS = ROUTER_SORT_ROWS * ROUTER_MOST_PICKS;
    static_assert(WIDE_SORT_THREADS == SORT_MOST_WAVES * SORT_WAVE && WIDE_SORT_THREADS >= ROUTER_MOST_EXPERTS, "a thread an expert");
    /* a scan's word: pairs in 12 bits, tiles and jobs in 10 each */
    static_assert(MOST_PAIRS < 4096u && MOST_PAIRS / WIDE_TILE_PAIRS + ROUTER_MOST_EXPERTS < 1024u &&
                      MOST_PAIRS / LINEAR_MAXIMUM_ROWS + ROUTER_MOST_EXPERTS < 1024u, "the three sums fit their bits");
    __shared__ uint32_t block_experts[MOST_PAIRS], sorted_index[MOST_PAIRS], cursors[SORT_MOST_WAVES * ROUTER_MOST_EXPERTS];
    __shared__ float weights[MOST_PAIRS];
    __shared__ uint64_t expert_offsets[ROUTER_MOST_EXPERTS * MODEL_EXPERT_MATRICES];
    __shared__ uint32_t starts[ROUTER_MOST_EXPERTS], totals[ROUTER_MOST_EXPERTS], job_starts[ROUTER_MOST_EXPERTS], scratch[SORT_MOST_WAVES];
    __shared__ uint16_t job_expert[1024];
    const uint32_t experts = arguments.expert_count, picks = arguments.pick_count, room = arguments.row_count * picks;
    const uint32_t wave = threadIdx.x / SORT_WAVE, expert = threadIdx.x;
    const struct router_pick *all_picks = (const struct router_pick *)(arena + arguments.picks_offset);
    const uint64_t *offsets = (const uint64_t *)(arena + arguments.expert_offsets_offset) + (uint64_t)expert * MODEL_EXPERT_MATRICES;
    const uint32_t live_rows = wide_live_rows(arguments, arena);
    struct router_pick mine[MOST_PAIRS / WIDE_SORT_THREADS];
    uint64_t own_offsets[MODEL_EXPERT_MATRICES] = {0, 0, 0};
#pragma unroll
    for (uint32_t k = 0; k < MOST_PAIRS / WIDE_SORT_THREADS; k++) {
        const uint32_t index = k * WIDE_SORT_THREADS + threadIdx.x;
        if (index < room) {
            mine[k] = all_picks[index];
        }
    }
    if (expert < experts) {
#pragma unroll
        for (uint32_t matrix = 0; matrix < MODEL_EXPERT_MATRICES; matrix++) {
            own_offsets[matrix] = offsets[matrix];
        }
    }
    for (uint32_t at = threadIdx.x; at < SORT_MOST_WAVES * experts; at += WIDE_SORT_THREADS) {
        cursors[at] = 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < MOST_PAIRS / WIDE_SORT_THREADS; k++) {
        const uint32_t index = k * WIDE_SORT_THREADS + threadIdx.x;
        if (index < room) { /* past the live rows: whatever the array holds, read no further */
            block_experts[index] = mine[k].expert;
            weights[index] = mine[k].route_weight;
        }
    }
    const uint32_t pairs = live_rows * picks;
    uint32_t begin, end;
    sort_share(pairs, wave, begin, end);
    __syncthreads();
    sort_count_share(block_experts, begin, end, cursors + wave * experts);
    __syncthreads();
    uint32_t counts[SORT_MOST_WAVES], total = 0, sums;
    if (expert < experts) {
        total = sort_counts_of(cursors, experts, expert, counts);
    }
    const uint32_t own_tiles = (total + WIDE_TILE_PAIRS - 1u) / WIDE_TILE_PAIRS, own_jobs = (total + LINEAR_MAXIMUM_ROWS - 1u) / LINEAR_MAXIMUM_ROWS;
    const uint32_t before = block_sum_before(total | own_tiles << 12 | own_jobs << 22, scratch, sums);
    const uint32_t start = before & 4095u, first_tile = before >> 12 & 1023u, first_job = before >> 22;
    const uint32_t used_tiles = sums >> 12 & 1023u, used_jobs = sums >> 22;
    struct wide_expert_tile *tiles = (struct wide_expert_tile *)(arena + arguments.tiles_offset);
    if (expert < experts) {
        sort_cursors_of(cursors, experts, expert, counts, start);
        starts[expert] = start;
        totals[expert] = total;
        job_starts[expert] = first_job;
#pragma unroll
        for (uint32_t matrix = 0; matrix < MODEL_EXPERT_MATRICES; matrix++) {
            expert_offsets[expert * MODEL_EXPERT_MATRICES + matrix] = own_offsets[matrix];
        }
        for (uint32_t k = 0; k < own_jobs; k++) {
            job_expert[first_job + k] = (uint16_t)expert;
        }
        ((struct wide_run *)(arena + arguments.runs_offset))[expert] = (struct wide_run){start, total};
        for (uint32_t k = 0; k < own_tiles; k++) {
            const uint32_t taken = k * WIDE_TILE_PAIRS, left = total - taken;
            tiles[first_tile + k] = (struct wide_expert_tile){own_offsets[0], own_offsets[1], own_offsets[2], start + taken,
                                                              left < WIDE_TILE_PAIRS ? left : WIDE_TILE_PAIRS};
        }
    }
    for (uint32_t tile = used_tiles + threadIdx.x; tile < ROUTER_WIDE_TILES_OF(arguments.row_count, picks, experts); tile += WIDE_SORT_THREADS) {
        tiles[tile] = (struct wide_expert_tile){0, 0, 0, 0, 0};
    }
    __syncthreads();
    struct wide_pair *sorted = (struct wide_pair *)(arena + arguments.pairs_offset);
    sort_place_share(block_experts, begin, end, experts, cursors + wave * experts, [&](uint32_t index, uint32_t place) {
        sorted_index[place] = index;
        sorted[place] = (struct wide_pair){index, weights[index]};
    });
    __syncthreads();
    struct expert_job_record *jobs = (struct expert_job_record *)(arena + arguments.jobs_offset);
    for (uint32_t job = threadIdx.x; job < ROUTER_WIDE_JOBS_OF(arguments.row_count, picks, experts); job += WIDE_SORT_THREADS) {
        struct expert_job_record value = {};
        if (job < used_jobs) {
            const uint32_t owner = job_expert[job];
            wide_job(job, job_starts[owner], owner, starts[owner], totals[owner], expert_offsets + owner * MODEL_EXPERT_MATRICES, value,
                     [&](uint32_t place, uint32_t &index, float &weight) {
                         index = sorted_index[place];
                         weight = weights[index];
                     });
        }
        jobs[job] = value;
    }
}

extern "C" __global__ void __launch_bounds__(WIDE_SORT_THREADS)
    router_wide_small(struct router_wide_arguments arguments, unsigned char *arena)
{
    wide_small(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_ROUTER, router_wide_small, router_wide_arguments);

/* ---- a router's last launch and the quantizer of the step's rows behind it, as one launch ----------------------
 * Neither reads what the other writes, and the router's is one block, or one for 384 rows: the first `blocks` blocks are its, the
 * others two of the quantizer's blocks each. The backend runs the pair so where it stands in a list (joined_launches.h, with
 * what that measured). Bound by the router's block, or by the quantizer's where the rows are many: each of
 * them holds the router's LDS as well (place 51 KB, small 74 KB), so that a CU has three or two, and 8192 rows of 4096 take 30 us, the quantizer
 * alone 25.5 (the rule stops joining where that costs more than a launch). */
#define QUANTIZE_JOIN_BLOCKS (WIDE_SORT_THREADS / LINEAR_ELEMENT_THREADS)
static_assert(SELECT_THREADS == WIDE_SORT_THREADS, "one block size");

template <bool WIDE_SCALES>
__device__ static __forceinline__ void joined_quantize(const struct activation_quantize_arguments &quantize, unsigned char *arena, uint32_t block, uint32_t columns,
                                                       uint32_t vectors)
{
    const uint32_t part = block * QUANTIZE_JOIN_BLOCKS + threadIdx.x / LINEAR_ELEMENT_THREADS, vector = part / columns;
    const uint32_t q = part % columns * LINEAR_ELEMENT_THREADS + threadIdx.x % LINEAR_ELEMENT_THREADS;
    if (vector >= vectors) {
        return;
    }
    if constexpr (WIDE_SCALES) {
        activation_quantize_128_body(quantize, arena, q, vector);
    } else {
        activation_quantize_body(quantize, arena, q, vector);
    }
}

#define ROUTER_JOIN(first, record, suffix, wide_scales, ...)                                                                            \
    extern "C" __global__ void __launch_bounds__(WIDE_SORT_THREADS)                                                                     \
        first##_quantize##suffix(struct record arguments, struct activation_quantize_arguments quantize, unsigned char *arena, uint32_t blocks, \
                                 uint32_t columns, uint32_t vectors)                                                                    \
    {                                                                                                                                   \
        if (blockIdx.x < blocks) {                                                                                                      \
            __VA_ARGS__;                                                                                                                \
        } else {                                                                                                                        \
            joined_quantize<wide_scales>(quantize, arena, blockIdx.x - blocks, columns, vectors);                                       \
        }                                                                                                                               \
    }                                                                                                                                   \
    ANEMONE_JOINED_KERNEL(KERNEL_FILE_ROUTER, first, KERNEL_FILE_ACTIVATION_QUANTIZE, activation_quantize##suffix##_entry, first##_quantize##suffix);
#define SELECT_LDS_BODY __shared__ struct router_select_lds lds; router_select_body(arguments, arena, threadIdx.x, SELECT_THREADS, lds)
ROUTER_JOIN(router_select_entry, router_select_arguments, , false, SELECT_LDS_BODY)
ROUTER_JOIN(router_select_entry, router_select_arguments, _128, true, SELECT_LDS_BODY)
ROUTER_JOIN(router_wide_small, router_wide_arguments, , false, wide_small(arguments, arena))
ROUTER_JOIN(router_wide_small, router_wide_arguments, _128, true, wide_small(arguments, arena))
ROUTER_JOIN(router_wide_place, router_wide_arguments, , false, wide_place(arguments, arena, blockIdx.x))
ROUTER_JOIN(router_wide_place, router_wide_arguments, _128, true, wide_place(arguments, arena, blockIdx.x))
