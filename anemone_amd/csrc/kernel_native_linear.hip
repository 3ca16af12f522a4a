/*
 * kernel_native_linear.hip -- the wide routed experts of weights stored in gfx950's own lane order
 * (WEIGHT_FORMAT_E2M1_GFX950, WEIGHT_FORMAT_E4M3_GFX950). The reference's E2M1_SCALED and E4M3_SCALED are by definition
 * the lane order of its cards' matrix instruction (include/anemone/weight_format_seam.h:22-46 there) and its seam says
 * how a backend brings its own: a new format, its kernels, its reference decode among the tests. These are the kernels:
 * what they read, write and sum is what wide_expert_gate_up_1 / wide_expert_down_1 of kernel_wide_linear.hip do for
 * the same matrix in the reference's lay-out, bit for bit (a lane's operand is the same bytes, so every sum is the same
 * chain of the same matrix instructions); only where the bytes lie in memory differs, and with it the work between the
 * load and the matrix instruction: none here.
 *
 * A block takes GROUP consecutive tiles of one expert from the wide select's table (GROUP x 64 columns) by 4 strips of
 * outputs, in the order of wide_order_device.cuh: the blocks of an expert's tiles side by side on one die.
 */
#include "kernel_registry.h"
#include "linear_device.cuh"
#include "quantize_device.cuh"

#include "native_device.cuh"
#include "wide_finish_device.cuh"
#include "wide_order_device.cuh"

/* the vectors of the columns a wavefront brings: code_vectors[part] of column lane / 8 of its group `part` of eight,
 * exponent_vectors[i] of column 16 (WAVE_BLOCKS wave + i) + lane / 4; columns past the last pair read the first pair's. The
 * wavefront leaves the pairs of its columns in LDS for the finish (behind the chain's barriers). */
template <typename CHAIN>
__device__ static __forceinline__ void native_vectors_of(const struct wide_pair *pairs, uint32_t pair_count, uint32_t divisor, uint32_t wave,
                                                         uint32_t lane, uint32_t (&code_vectors)[2u * CHAIN::WAVE_BLOCKS],
                                                         uint32_t (&exponent_vectors)[CHAIN::WAVE_BLOCKS], struct wide_pair *columns)
{
    constexpr uint32_t WAVE_BLOCKS = CHAIN::WAVE_BLOCKS;
#pragma unroll
    for (uint32_t part = 0; part < 2u * WAVE_BLOCKS; part++) {
        const uint32_t column = 8u * CHAIN::group_of(wave, part) + lane / 8u;
        code_vectors[part] = pairs[column < pair_count ? column : 0u].pair_index / divisor;
    }
#pragma unroll
    for (uint32_t i = 0; i < WAVE_BLOCKS; i++) {
        const uint32_t column = 16u * (WAVE_BLOCKS * wave + i) + lane / 4u;
        exponent_vectors[i] = pairs[column < pair_count ? column : 0u].pair_index / divisor;
    }
    const uint32_t own_column = 16u * WAVE_BLOCKS * wave + lane % (16u * WAVE_BLOCKS);
    columns[own_column] = pairs[own_column < pair_count ? own_column : 0u];
}

/* grid (ceil(output_size / (4 strips)), tile_count), block 256; a strip is STRIP tiles of gate and STRIP of up */
/* sets of weight registers and stages of columns: 4-bit weights 2 and 2, with strips of four gate and four up tiles (eight
 * of down) at two wavefronts a SIMD (241 registers, 128 of them sums): a column block's operand read from LDS and its
 * permutations serve eight matrix instructions and not four (8192 rows of 4096 x 2048 x 256 experts: gate/up 1157 -> 1096
 * us, down 651 -> 625, against strips of half as many, three sets and three wavefronts; both with columns turned in place). One-byte weights: gate/up 2 and 2
 * at three wavefronts a SIMD (143 registers, 165 with float32 scales), down 3 and 3 at two (215 and 222): 2048 rows of
 * 4096 x 2048 x 256 experts, gate/up 880 us against 900 (float32 scales 850 / 864), down 433 against 444 (444 / 453). */
template <bool BYTES, bool DOWN, uint32_t TILES> /* tiles of a wavefront, of its matrices together */
struct native_depths {
    static constexpr uint32_t SLOTS = BYTES ? (DOWN && TILES == 2u ? 3u : 2u) : TILES == 8u ? 2u : 3u;
    static constexpr uint32_t DEPTH = BYTES ? (TILES == 4u ? NATIVE_E4M3_WHOLE_STAGES : DOWN ? NATIVE_E4M3_DOWN_STAGES : NATIVE_E4M3_GATE_UP_STAGES) : NATIVE_E2M1_STAGES;
};

template <bool BYTES, uint32_t STRIP, uint32_t GROUP, bool B128 = false>
__device__ static __forceinline__ void native_expert_gate_up(const struct wide_expert_gate_up_arguments &arguments, unsigned char *arena)
{
    constexpr uint32_t COLUMN_BLOCKS = 4u * GROUP;
    typedef native_depths<BYTES, false, 2u * STRIP> depths;
    typedef native_chain<2, BYTES, STRIP, COLUMN_BLOCKS, depths::SLOTS, depths::DEPTH, B128> chain_type;
    constexpr uint32_t TILES = chain_type::TILES;
    static_assert(STRIP == 1u || STRIP % 2u == 0u, "a quantizer block of 32 outputs is two strips, or strips are whole blocks");
    extern __shared__ __attribute__((aligned(128))) unsigned char window[];
    __shared__ struct wide_pair columns[COLUMN_BLOCKS * 16u];
    const uint32_t lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    struct wide_expert_tile tile;
    uint32_t pair_count = 0, block_strip = 0;
    bool alone = false;
    const uint32_t strips = (arguments.output_size + NATIVE_WAVES * STRIP * 16u - 1u) / (NATIVE_WAVES * STRIP * 16u);
    if (!order_block_of<GROUP, false, !BYTES || chain_type::TILES == 4u>((const struct wide_expert_tile *)(arena + arguments.tiles_offset), arguments.tile_count, strips, lane, block_strip, tile, pair_count, &alone)) {
        return;
    }
    const struct wide_pair *pairs = (const struct wide_pair *)(arena + arguments.pairs_offset) + tile.first_pair;
    uint32_t code_vectors[2u * chain_type::WAVE_BLOCKS], exponent_vectors[chain_type::WAVE_BLOCKS];
    native_vectors_of<chain_type>(pairs, pair_count, arguments.pairs_per_row, wave, lane, code_vectors, exponent_vectors, columns);
    chain_type chain_of;
    chain_of.once = alone;
    const unsigned char *const matrices[2] = {arena + tile.gate_offset, arena + tile.up_offset};
    uint32_t tile0 = 0;
    chain_of.place(matrices, arguments.output_size, arguments.input_size, block_strip, arena + arguments.codes_offset,
                   arena + arguments.exponents_offset, code_vectors, exponent_vectors, (uint32_t)(uintptr_t)(lds_pointer)window, wave, lane, tile0);
    float4_t chain[TILES][COLUMN_BLOCKS];
#pragma unroll
    for (uint32_t t = 0; t < TILES; t++) {
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            chain[t][j] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    chain_of.whole(arguments.input_size / 128u, (pair_count + 15u) / 16u, chain);
    wide_gate_up_finish<STRIP, COLUMN_BLOCKS, B128>(arguments, arena, window, columns, pair_count, block_strip, tile0, wave, lane, chain);
}

template <bool BYTES, uint32_t DOWN_STRIP, uint32_t GROUP, bool B128 = false, bool BY_RUN = !BYTES || DOWN_STRIP == 4u>
__device__ static __forceinline__ void native_expert_down(const struct wide_expert_down_arguments &arguments, unsigned char *arena)
{
    constexpr uint32_t COLUMN_BLOCKS = 4u * GROUP;
    typedef native_depths<BYTES, true, DOWN_STRIP> depths;
    typedef native_chain<1, BYTES, DOWN_STRIP, COLUMN_BLOCKS, depths::SLOTS, depths::DEPTH, B128> chain_type;
    constexpr uint32_t TILES = chain_type::TILES, STRIP = chain_type::STRIP;
    extern __shared__ __attribute__((aligned(128))) unsigned char window[];
    __shared__ struct wide_pair columns[COLUMN_BLOCKS * 16u];
    const uint32_t lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    struct wide_expert_tile tile;
    uint32_t pair_count = 0, block_strip = 0;
    bool alone = false;
    const uint32_t strips = (arguments.output_size + NATIVE_WAVES * DOWN_STRIP * 16u - 1u) / (NATIVE_WAVES * DOWN_STRIP * 16u);
    if (!order_block_of<GROUP, true, BY_RUN>((const struct wide_expert_tile *)(arena + arguments.tiles_offset), arguments.tile_count, strips, lane, block_strip, tile, pair_count, &alone)) {
        return;
    }
    const struct wide_pair *pairs = (const struct wide_pair *)(arena + arguments.pairs_offset) + tile.first_pair;
    uint32_t code_vectors[2u * chain_type::WAVE_BLOCKS], exponent_vectors[chain_type::WAVE_BLOCKS]; /* the vectors are the pairs' hidden vectors */
    native_vectors_of<chain_type>(pairs, pair_count, 1u, wave, lane, code_vectors, exponent_vectors, columns);
    chain_type chain_of;
    chain_of.once = alone;
    const unsigned char *const matrices[1] = {arena + tile.down_offset};
    uint32_t tile0 = 0;
    chain_of.place(matrices, arguments.output_size, arguments.input_size, block_strip, arena + arguments.codes_offset,
                   arena + arguments.exponents_offset, code_vectors, exponent_vectors, (uint32_t)(uintptr_t)(lds_pointer)window, wave, lane, tile0);
    float4_t chain[TILES][COLUMN_BLOCKS];
#pragma unroll
    for (uint32_t t = 0; t < TILES; t++) {
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            chain[t][j] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    chain_of.whole(arguments.input_size / 128u, (pair_count + 15u) / 16u, chain);
    wide_down_finish<STRIP, COLUMN_BLOCKS>(arguments, arena, columns, pair_count, block_strip, tile0, wave, lane, chain);
}

/* E2M1_GFX950 experts: a block is one tile of pairs by 256 outputs of gate and up (512 of down); E4M3_GFX950 experts: two
 * tiles by 64 (128 of down). The LDS window is dynamic shared memory: NATIVE_WINDOW_BYTES(column blocks, stages). */
#define NATIVE_E2M1_WAVES 2 /* 256 registers */
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_E2M1_WAVES) native_expert_gate_up_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<false, 4u, NATIVE_E2M1_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_E2M1_WAVES) native_expert_down_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<false, 8u, NATIVE_E2M1_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_1, wide_expert_down_arguments);
/* the same of half the strips, at three wavefronts a SIMD: for launches of few pairs an expert whose blocks fill their last
 * round better so (anemone_amd/host/linear.c, native_takes_narrow, holds both sides' times). Down's blocks go as they are
 * dealt: its chains are short and its runs a tile, so that the two looks at the table for an order of runs cost more than
 * the order gives (down of 896 x 3072 x 128 experts, 4 pairs an expert: 42.2 -> 40.0 us; of 768 x 2048 x 384, 3: 65.5 -> 61.9;
 * loads of Zipf(1.1), 24 on average: 40.4..92.9 -> 38.0..89.5); gate/up's gain 0 to 6 % from it at 24 pairs. */
#define NATIVE_E2M1_NARROW_WAVES 3 /* 168 registers */
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_E2M1_NARROW_WAVES) native_expert_gate_up_narrow_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<false, 2u, NATIVE_E2M1_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_narrow_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_E2M1_NARROW_WAVES) native_expert_down_narrow_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<false, 4u, NATIVE_E2M1_COLUMN_BLOCKS / 4u, false, false>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_narrow_1, wide_expert_down_arguments);
#define NATIVE_BYTES_GATE_UP_WAVES 3
#define NATIVE_BYTES_DOWN_WAVES 2
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_GATE_UP_WAVES) native_expert_gate_up_e4m3_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<true, 1u, NATIVE_E4M3_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_e4m3_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_DOWN_WAVES) native_expert_down_e4m3_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<true, 2u, NATIVE_E4M3_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_e4m3_1, wide_expert_down_arguments);

/* E4M3_BLOCK128_GFX950 experts (float32 scales of 128 x 128 blocks, columns of 128-value float32 scales): the E4M3_GFX950
 * launches' shape; the gate/up launch leaves the hidden VALUES where the record names the hidden operands, and their
 * quantizer (activation_quantize_128_entry) is a launch of its own */
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_GATE_UP_WAVES) native_expert_gate_up_b128_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<true, 1u, NATIVE_E4M3_COLUMN_BLOCKS / 4u, true>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_b128_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_DOWN_WAVES) native_expert_down_b128_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<true, 2u, NATIVE_E4M3_COLUMN_BLOCKS / 4u, true>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_b128_1, wide_expert_down_arguments);

/* The one-byte launches of whole strips: twice the tiles a wavefront (gate's two and up's two, or four of down), so that a
 * block's columns, which every strip's block brings into LDS again, are brought half as often and an operand read from LDS
 * serves four matrix instructions; two sets of weights and two stages at two wavefronts a SIMD (244 to 253 registers, 128 of
 * them sums); the blocks in the order of runs, where each is a longer piece of work and the look at the table counts less. For
 * launches of many pairs an expert (native_takes_whole_bytes, with both sides' times): at 64 pairs an expert a launch is near
 * what memory gives and three wavefronts a SIMD hide more, at 128 columns were 45 % of the lines that passed the level-2 caches
 * (4096 rows of 4096 x 2048 x 256 experts, float32 scales: gate/up 1105 -> 985 us, 9.4e7 -> 7.3e7 lines, 7.3 -> 5.2 GB fetched; down
 * 598 -> 539 us, 4.8e7 -> 3.7e7 lines). */
#define NATIVE_BYTES_WHOLE_WAVES 2
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_WHOLE_WAVES) native_expert_gate_up_e4m3_whole_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<true, 2u, NATIVE_E4M3_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_e4m3_whole_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_WHOLE_WAVES) native_expert_down_e4m3_whole_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<true, 4u, NATIVE_E4M3_COLUMN_BLOCKS / 4u>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_e4m3_whole_1, wide_expert_down_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_WHOLE_WAVES) native_expert_gate_up_b128_whole_1(struct wide_expert_gate_up_arguments arguments, unsigned char *arena)
{
    native_expert_gate_up<true, 2u, NATIVE_E4M3_COLUMN_BLOCKS / 4u, true>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_gate_up_b128_whole_1, wide_expert_gate_up_arguments);
extern "C" __global__ void __launch_bounds__(NATIVE_THREADS, NATIVE_BYTES_WHOLE_WAVES) native_expert_down_b128_whole_1(struct wide_expert_down_arguments arguments, unsigned char *arena)
{
    native_expert_down<true, 4u, NATIVE_E4M3_COLUMN_BLOCKS / 4u, true>(arguments, arena);
}
ANEMONE_KERNEL(KERNEL_FILE_NATIVE_LINEAR, native_expert_down_b128_whole_1, wide_expert_down_arguments);

static_assert(native_chain<2, false, 2u, NATIVE_E2M1_COLUMN_BLOCKS, 3u, NATIVE_E2M1_STAGES>::WINDOW_BYTES == NATIVE_WINDOW_BYTES(NATIVE_E2M1_COLUMN_BLOCKS, NATIVE_E2M1_STAGES) &&
                  native_chain<2, true, 1u, NATIVE_E4M3_COLUMN_BLOCKS, 2u, NATIVE_E4M3_GATE_UP_STAGES>::WINDOW_BYTES == NATIVE_WINDOW_BYTES(NATIVE_E4M3_COLUMN_BLOCKS, NATIVE_E4M3_GATE_UP_STAGES) &&
                  native_chain<1, true, 2u, NATIVE_E4M3_COLUMN_BLOCKS, 3u, NATIVE_E4M3_DOWN_STAGES>::WINDOW_BYTES == NATIVE_WINDOW_BYTES(NATIVE_E4M3_COLUMN_BLOCKS, NATIVE_E4M3_DOWN_STAGES) &&
                  native_chain<2, true, 2u, NATIVE_E4M3_COLUMN_BLOCKS, 2u, NATIVE_E4M3_WHOLE_STAGES>::WINDOW_BYTES == NATIVE_WINDOW_BYTES(NATIVE_E4M3_COLUMN_BLOCKS, NATIVE_E4M3_WHOLE_STAGES),
              "the windows the host asks for are the kernels'");
