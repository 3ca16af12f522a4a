/*
 * native_device.cuh -- a block's pipeline over weights stored in gfx950's own lane order (WEIGHT_FORMAT_E2M1_GFX950,
 * WEIGHT_FORMAT_E4M3_GFX950): a tile's K step of 128 inputs lies in memory as the 64 lanes' A operand of
 * v_mfma_scale_f32_16x16x128_f8f6f4, 16 bytes a lane (32 of one-byte weights, as two halves of 16), and goes from memory
 * into the wavefront's registers with one 16-byte load a lane and half: no LDS stage, no vector instruction between the
 * load and the matrix instruction. Only the columns (the vectors' codes, which every wavefront of the block reads) pass
 * through LDS, as in wide_device.cuh: brought by LDS DMA and read as they landed. (4-bit weights take the B operand's bytes in
 * another order, eight permutations a column block in every wavefront, which run beside the matrix instructions. Turned
 * about in place, once a block, by the wavefront that brought them, the columns cost it an LDS round trip ahead of every
 * step's barrier: 8192 rows of 4096 x 2048 x 256 experts, with the weights asked for in the middle of a step: gate/up 1098
 * -> 1065 us, down 635 -> 606.)
 *
 * A block is COLUMN_BLOCKS x 16 columns (pairs of one expert) by four wavefronts' strips of weight tiles. A wavefront
 * keeps several sets of weight registers: while one step is multiplied, the loads of the steps behind it are on their way.
 *
 * What bounds the one-byte launches, beside the weights' way from memory, is the number of loads: with the clock read
 * around a step's parts, a third of a wavefront's time went into asking for them (six of weights and five of columns a
 * step, about 130 cycles each: the memory pipeline takes a wavefront's load a cache line a cycle and keeps a limited number
 * of lines on their way). So the words of scales, which are a line each for four bytes, come in fewer loads -- the columns'
 * four K steps together, the weights' sixty-four together, a lane a step -- and columns that hold no pair are not brought:
 * 2048 rows of 4096 x 2048 x 256 experts, float32 scales: gate/up 930 -> 852 us, down 483 -> 446; E8M0 scales: 930 -> 897,
 * 455 -> 435; 4-bit weights, 8192 rows: 1 %.
 */
#ifndef NATIVE_DEVICE_CUH
#define NATIVE_DEVICE_CUH

#include "linear_device.cuh"
#include "native_waits.h"

#define NATIVE_WAVES 4u
#define NATIVE_THREADS (NATIVE_WAVES * WAVE)

/* memory into registers, 16 bytes or a word a lane: the address is a base common to the wavefront plus the lane's own
 * byte offset (plus 1,024: the second half of a tile of one-byte weights). Assembly, like the loads into LDS beside which
 * they are counted: the compiler keeps no book on them, native_landed is the wait (so a kernel of these loads must spill
 * no vector register: one saved between its load and the wait is saved before it is filled, and the build refuses such
 * a kernel). ONCE: the bytes are read by this
 * block alone, and are asked for as a stream (native_chain::once). */
template <bool ONCE>
__device__ static __forceinline__ void load_16(uint4_t &into, const unsigned char *base, uint32_t lane_offset)
{
    if constexpr (ONCE) {
        asm volatile("global_load_dwordx4 %0, %1, %2 nt" : "=v"(into) : "v"(lane_offset), "s"(base) : "memory");
    } else {
        asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(into) : "v"(lane_offset), "s"(base) : "memory");
    }
}

template <bool ONCE>
__device__ static __forceinline__ void load_16_second(uint4_t &into, const unsigned char *base, uint32_t lane_offset)
{
    if constexpr (ONCE) {
        asm volatile("global_load_dwordx4 %0, %1, %2 offset:1024 nt" : "=v"(into) : "v"(lane_offset), "s"(base) : "memory");
    } else {
        asm volatile("global_load_dwordx4 %0, %1, %2 offset:1024" : "=v"(into) : "v"(lane_offset), "s"(base) : "memory");
    }
}

__device__ static __forceinline__ void load_4(uint32_t &into, const unsigned char *base, uint32_t lane_offset)
{
    asm volatile("global_load_dword %0, %1, %2" : "=v"(into) : "v"(lane_offset), "s"(base) : "memory");
}

/* behind wait_loads: the value the load left in the register is this statement's result, so that nothing that uses it
 * can be placed ahead of the wait */
__device__ static __forceinline__ void native_landed(uint4_t &value)
{
    asm volatile("" : "+v"(value));
}

__device__ static __forceinline__ void native_landed(uint32_t &value)
{
    asm volatile("" : "+v"(value));
}

/* SLOTS: sets of weight registers a wavefront keeps (the weights of SLOTS - 1 steps are on their way while one is
 * multiplied); DEPTH: stages of columns in LDS, likewise */
/* B128 (one-byte weights alone): float32 scales, one for every 128 outputs x 128 inputs of a matrix and one for every 128
 * values of a column, in place of the E8M0 codes (the same bytes a K step: a word where four codes were): a K step's
 * matrix instruction runs from zero with scale codes of one and its sums enter the chain by one fused multiply-add with
 * the product of the two scales, as the reference-order kernels of that scaling add them */
template <uint32_t MATRICES, bool BYTES, uint32_t STRIP_TILES, uint32_t COLUMN_BLOCKS, uint32_t SLOTS, uint32_t DEPTH, bool B128 = false>
struct native_chain {
    static_assert(BYTES || !B128, "float32 scales go with one-byte weights");
    static_assert(COLUMN_BLOCKS == 4u || COLUMN_BLOCKS == 8u, "a wavefront brings one or two column blocks");
    static constexpr uint32_t STRIP = STRIP_TILES;
    static constexpr uint32_t TILES = MATRICES * STRIP;
    static constexpr bool STREAMS = BYTES || TILES != 8u; /* whole strips of 4-bit weights are for experts of many tiles: no instance of them streams */
    static constexpr uint32_t STEP_BYTES = BYTES ? BYTE_STEP_BYTES : NIBBLE_STEP_BYTES;
    static constexpr uint32_t HALVES = STEP_BYTES / 1024u;
    static constexpr uint32_t WAVE_BLOCKS = COLUMN_BLOCKS / NATIVE_WAVES;     /* column blocks whose scale words a wavefront brings */
    static constexpr uint32_t VECTOR_BYTES = COLUMN_BLOCKS * 2048u;            /* a K step of the block's columns' codes */
    static constexpr uint32_t STAGE_BYTES = VECTOR_BYTES;
    static constexpr uint32_t SCALE_STEPS = 4u; /* K steps whose scale words of the columns come together */
    static constexpr uint32_t CHUNK_BYTES = COLUMN_BLOCKS * 16u * SCALE_STEPS * 4u; /* [column][step of the chunk] */
    static constexpr uint32_t SCALES_AT = DEPTH * STAGE_BYTES; /* two chunks behind the stages: one in use, the next on its way */
    static constexpr uint32_t WINDOW_BYTES = SCALES_AT + 2u * CHUNK_BYTES;
    /* loads of a wavefront for a step's columns of LIVE column blocks: groups of eight columns (the groups wave, wave + 4, ...
     * that LIVE blocks need), and one of scale words */
    static constexpr uint32_t groups_of(uint32_t live)
    {
        return (live + 1u) / 2u;
    }
    static constexpr uint32_t vector_loads(uint32_t live)
    {
        return groups_of(live) + 1u;
    }
    /* scales: of one-byte weights a word a tile or a matrix a K step (a row of 32 outputs' four codes, as the reference stores
     * them, or one float32), which a lane a step holds for SCALE_ROUND steps and a step takes from its lane; of
     * 4-bit weights a word a lane a matrix: its bytes are the codes of the lane's row and inputs in the four tiles of a group
     * of 64 outputs, which the matrix instruction picks by number */
    static constexpr uint32_t GROUP_TILES = STRIP < 4u ? STRIP : 4u; /* tiles of a strip that share a word of 4-bit weights' codes */
    static constexpr uint32_t GROUPS = BYTES ? 1u : STRIP / GROUP_TILES;
    static constexpr uint32_t SCALE_LOADS = BYTES && !B128 ? TILES : MATRICES * GROUPS;
    static constexpr uint32_t WEIGHT_LOADS = TILES * HALVES + (BYTES ? 0u : SCALE_LOADS);
    static constexpr uint32_t SCALE_ROUND = WAVE / SLOTS * SLOTS;
    static_assert(BYTES || STRIP == 2u || STRIP % 4u == 0u, "a strip of 4-bit weights is half a group of four tiles, or whole ones");
    static_assert((DEPTH - 1u) * vector_loads(COLUMN_BLOCKS) + (SLOTS - 1u) * WEIGHT_LOADS < 64u, "vmcnt has six bits");

    struct slot {
        uint4_t words[TILES][HALVES];
        uint32_t scale[BYTES ? 1 : SCALE_LOADS]; /* 4-bit weights */
    };

    /* STREAMS: whether the block holds all of its expert's pairs (the same in every lane). Then no other block reads these weights,
     * and they are asked for as a stream, so that they do not push the columns, which every strip's block reads, out of the level-2
     * cache; where an expert has more blocks, a streamed line is read from memory again. 4096 x 2048, gate/up and down, us, no weight
     * as a stream | every weight | by this rule: FP8 of 2048 rows, 256 experts 919 and 446 | 880 and 430 | 887 and 430; 4096 rows 1160
     * and 605 | 1350 and 658 | 1138 and 600; 4096 rows of Zipf(1.1) loads 1251 and 656 | 1414 and 700 | 1222 and 652; 2048 rows of 64
     * experts 463 and 257 | 572 and 282 | 470 and 260; 500 Zipf rows of 128 experts 421 and 219 | 410 and 211 | 403 and 209 (float32 scales:
     * the same picture). 4-bit weights in narrow strips, 300 rows of 256 experts 386 and 210 | 361 and 196 | 360 and 195; 700
     * Zipf rows 431 and 228 | 434 and 233 | 410 and 221. */
    bool once = false;
    const unsigned char *words[MATRICES], *scales[MATRICES], *codes, *exponents;
    uint32_t step_stride, scale_stride; /* from a tile's K step to its next; from a group's scale words to the next group's */
    uint32_t window, wave, tile_bytes, group_bytes, word_offset, scale_offset[BYTES && !B128 ? STRIP : 1], code_shift, codes_offset[2u * WAVE_BLOCKS], exponents_offset[WAVE_BLOCKS];
    /* 4-bit weights: strips of four tiles have no registers for a place a piece, and add three times a column block instead */
    static constexpr bool PIECES_HELD = TILES == 8u;
    uint32_t vector_at[BYTES ? 8 : PIECES_HELD ? 4 : 1], vector_scale_at, scale_shift, last_step, lane_of;

    template <typename T>
    __device__ static __forceinline__ T lds_read(uint32_t address)
    {
        return *(const __attribute__((address_space(3))) T *)(uintptr_t)address;
    }

    /* The scale words of a column lie in that column's own row: asked for a step at a time they are a cache line a column for
     * four bytes, as many lines as the columns' codes. So the words of four K steps come together, a lane a step of a
     * column: a quarter of the lines. Column block `block` of this wavefront, chunk `chunk` of four steps (a step past the
     * last repeats the last). */
    __device__ __forceinline__ void issue_scales(uint32_t chunk, uint32_t block) const
    {
        const uint32_t step = SCALE_STEPS * chunk + lane_of % SCALE_STEPS;
        const uint32_t offset = (block == 0u ? exponents_offset[0] : exponents_offset[WAVE_BLOCKS - 1u]) + 4u * (step < last_step ? step : last_step);
        load_to_lds_4(exponents, offset, window + SCALES_AT + chunk % 2u * CHUNK_BYTES + (wave * WAVE_BLOCKS + block) * (16u * SCALE_STEPS * 4u));
    }

    /* the group of eight columns that is this wavefront's part `part` */
    __device__ __forceinline__ static uint32_t group_of(uint32_t wave_index, uint32_t part)
    {
        return wave_index + NATIVE_WAVES * part;
    }

    /* the block's columns of K step `at` into stage `stage`, this wavefront's groups; and one load of scale words: the
     * next chunk's are asked for behind the barrier of a chunk's first steps, a column block a step, when every wavefront is
     * done with the chunk whose place they take (in the other steps one lane reads a word again, so that every step's loads
     * are as many) */
    template <uint32_t LIVE>
    __device__ __forceinline__ void issue_vectors(uint32_t stage, uint32_t at) const
    {
        const uint32_t base = window + stage * STAGE_BYTES;
#pragma unroll
        for (uint32_t part = 0; part < groups_of(LIVE); part++) {
            load_to_lds_16(codes + (uint64_t)at * 128u, codes_offset[part], base + group_of(wave, part) * 1024u);
        }
        const uint32_t now = at < DEPTH - 1u ? SCALE_STEPS - 1u : at - (DEPTH - 1u); /* the step that asks; ahead of the first: no chunk's first steps */
        const bool next = now % SCALE_STEPS < WAVE_BLOCKS;
        if (next || lane_of == 0u) {
            issue_scales(at < DEPTH - 1u ? 0u : now / SCALE_STEPS + (next ? 1u : 0u), next ? now % SCALE_STEPS : 0u);
        }
    }

    /* the wavefront's weights and scale codes of K step `at` into a set of registers */
    template <bool ONCE>
    __device__ __forceinline__ void issue_weights(slot &into, uint32_t at) const
    {
#pragma unroll
        for (uint32_t m = 0; m < MATRICES; m++) {
            const unsigned char *step_words = words[m] + (uint64_t)at * step_stride;
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n++) {
                /* the tile's place is scalar: one register of lane offsets serves every tile */
                const unsigned char *tile_words = step_words + n / 4u * group_bytes + n % 4u * tile_bytes;
                load_16<ONCE>(into.words[m * STRIP + n][0], tile_words, word_offset);
                if constexpr (BYTES) {
                    load_16_second<ONCE>(into.words[m * STRIP + n][1], tile_words, word_offset);
                }
            }
        }
        if constexpr (!BYTES) {
#pragma unroll
            for (uint32_t m = 0; m < MATRICES; m++) {
#pragma unroll
                for (uint32_t group = 0; group < GROUPS; group++) { /* a word a lane of a group of four tiles' codes */
                    load_4(into.scale[m * GROUPS + group], scales[m] + (uint64_t)at * 256u + group * scale_stride, scale_offset[0]);
                }
            }
        }
    }

    /* one-byte weights: the scale words of the steps first .. first + SCALE_ROUND - 1, a lane a step (past the last: the
     * last's). A load a step of words that every lane shares would cost the memory pipeline as much as a tile's */
    __device__ __forceinline__ void issue_weight_scales(uint32_t (&into)[SCALE_LOADS], uint32_t first) const
    {
        const uint32_t step = first + lane_of < last_step ? first + lane_of : last_step;
#pragma unroll
        for (uint32_t k = 0; k < SCALE_LOADS; k++) {
            load_4(into[k], scales[B128 ? k : k / STRIP], scale_offset[B128 ? 0u : k % STRIP] + 4u * step);
        }
    }

    __device__ static __forceinline__ void landed(slot &set)
    {
#pragma unroll
        for (uint32_t t = 0; t < TILES; t++) {
#pragma unroll
            for (uint32_t h = 0; h < HALVES; h++) {
                native_landed(set.words[t][h]);
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < (BYTES ? 0u : SCALE_LOADS); k++) {
            native_landed(set.scale[k]);
        }
    }

    /* the scale words of step `step` of the columns, this lane's part aside */
    __device__ __forceinline__ uint32_t scales_of(uint32_t step) const
    {
        return SCALES_AT + step / SCALE_STEPS % 2u * CHUNK_BYTES + 4u * (step % SCALE_STEPS);
    }

    /* 4-bit weights: tile T and the tiles behind it of the wavefront's strip against column block j (the number of the scale
     * code's byte is part of the instruction: a constant) */
    template <uint32_t T>
    __device__ static __forceinline__ void multiply_tiles(const slot &set, const uint32_t (&scale_a)[SCALE_LOADS], const int8_vector &b,
                                                          uint32_t scale_b, uint32_t j, float4_t (&chain)[TILES][COLUMN_BLOCKS])
    {
        const uint4_t w = set.words[T][0];
        const int8_vector a = {(int)w.x, (int)w.y, (int)w.z, (int)w.w, 0, 0, 0, 0};
        chain[T][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, chain[T][j], 4, 0, T % GROUP_TILES, (int)scale_a[T / GROUP_TILES], 0, (int)scale_b);
        if constexpr (T + 1u < TILES) {
            multiply_tiles<T + 1u>(set, scale_a, b, scale_b, j, chain);
        }
    }

    /* 4-bit weights: a column block's codes, read from the stage as they landed (a column's 128 bytes in the order the
     * quantizer writes them), and the B operand of them */
    __device__ static constexpr uint32_t piece_of(uint32_t part) /* pieces 0, 1, 4 and 5 from the lane's first: bits 4 and 6 of the place */
    {
        return 16u * (part % 2u) + 64u * (part / 2u);
    }

    __device__ __forceinline__ void read_pieces(uint32_t at, uint32_t scales, uint32_t j, uint2_t (&pieces)[4], uint32_t &scale_b) const
    {
        uint32_t first = vector_at[0];
        if constexpr (!PIECES_HELD) {
            asm volatile("" : "+v"(first)); /* anew for every block: the compiler keeps no sum of it */
        }
#pragma unroll
        for (uint32_t part = 0; part < 4u; part++) {
            pieces[part] = lds_read<uint2_t>((PIECES_HELD ? vector_at[part] : first ^ piece_of(part)) + at + j * 2048u);
        }
        scale_b = lds_read<unsigned char>(vector_scale_at + scales + j * (16u * SCALE_STEPS * 4u));
    }

    __device__ static __forceinline__ int8_vector operand_of(const uint2_t (&pieces)[4])
    {
        int8_vector b;
#pragma unroll
        for (uint32_t part = 0; part < 4u; part++) {
            b[2u * part] = (int)__builtin_amdgcn_perm(pieces[part].y, pieces[part].x, 0x05010400u);
            b[2u * part + 1u] = (int)__builtin_amdgcn_perm(pieces[part].y, pieces[part].x, 0x07030602u);
        }
        return b;
    }

    /* one K step of LIVE column blocks from a stage's columns and a set of weight registers */
    template <uint32_t LIVE>
    __device__ __forceinline__ void consume(uint32_t stage, uint32_t step, const slot &set, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        uint32_t scale_a[SCALE_LOADS];
#pragma unroll
        for (uint32_t k = 0; k < SCALE_LOADS; k++) { /* two tiles a strip: the group's upper two tiles' codes down */
            scale_a[k] = set.scale[k] >> scale_shift;
        }
        const uint32_t at = stage * STAGE_BYTES, scales = scales_of(step);
        uint2_t pieces[LIVE][4];
        uint32_t scale_b[LIVE];
        read_pieces(at, scales, 0u, pieces[0], scale_b[0]);
#pragma unroll
        for (uint32_t j = 0; j < LIVE; j++) {
            asm volatile("" ::: "memory"); /* the reads below stay below the reads above, and above those of the next block */
            if (j + 1u < LIVE) { /* a column block's codes are read while the block before it is multiplied */
                read_pieces(at, scales, j + 1u, pieces[j + 1u], scale_b[j + 1u]);
            }
            /* the further a wavefront is into its step, the more its instructions go first: the two of a SIMD then meet in
             * different phases (gate/up 1115 -> 1087 us at 8192 rows; one priority through the matrix instructions, or none: 1115) */
            if (j == 1u) {
                __builtin_amdgcn_s_setprio(1);
            } else if (j == 2u) {
                __builtin_amdgcn_s_setprio(2);
            } else if (j == 3u) {
                __builtin_amdgcn_s_setprio(3);
            }
            multiply_tiles<0>(set, scale_a, operand_of(pieces[j]), scale_b[j], j, chain);
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the stage is read before the next barrier */
    }

    /* one-byte weights: a column block's B operand, read from the stage as the codes landed: the lane's eight words lie four
     * words apart, and the slots of the pieces put the 64 lanes of a word on every bank twice */
    __device__ __forceinline__ void read_block(uint32_t at, uint32_t scales, uint32_t j, int8_vector &b, uint32_t &scale_b) const
    {
#pragma unroll
        for (uint32_t v = 0; v < 8u; v++) {
            b[v] = (int)lds_read<uint32_t>(vector_at[v] + at + j * 2048u);
        }
        const uint32_t scale_at = vector_scale_at + scales + j * (16u * SCALE_STEPS * 4u);
        scale_b = B128 ? lds_read<uint32_t>(scale_at) : lds_read<unsigned char>(scale_at); /* a float32's bits, or a code */
    }

    /* The same step of one-byte weights. A column block's operand is read while the block before it is multiplied (two or
     * three blocks ahead: the same time, and more registers); under float32 scales products enter their chains while the next
     * ones are formed. */
    template <uint32_t LIVE>
    __device__ __forceinline__ void consume_bytes(uint32_t stage, uint32_t step, const slot &set, const uint32_t (&held)[SCALE_LOADS], uint32_t holder,
                                                  float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        uint32_t scale_a[SCALE_LOADS];
#pragma unroll
        for (uint32_t k = 0; k < SCALE_LOADS; k++) {
            const uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)held[k], (int)holder);
            scale_a[k] = B128 ? word : word >> code_shift; /* a code: the instruction takes the lowest byte */
        }
        const uint32_t at = stage * STAGE_BYTES, scales = scales_of(step);
        int8_vector b[LIVE];
        uint32_t scale_b[LIVE];
        /* float32 scales: the tiles whose products wait together (one of four: two's do not fit beside the sums of eight blocks) */
        constexpr uint32_t PART = TILES > 2u ? 1u : TILES, PARTS = TILES / PART;
        float4_t products[2][PART];
        const auto add = [&](uint32_t place) { /* part place % PARTS of column block place / PARTS */
            const uint32_t j = place / PARTS, first = place % PARTS * PART;
#pragma unroll
            for (uint32_t t = 0; t < PART; t++) {
                const float scale = __fmul_rn(__uint_as_float(scale_a[(first + t) / STRIP]), __uint_as_float(scale_b[j]));
#pragma unroll
                for (uint32_t v = 0; v < 4u; v++) {
                    chain[first + t][j][v] = __fmaf_rn(products[place % 2u][t][v], scale, chain[first + t][j][v]);
                }
            }
        };
        __builtin_amdgcn_s_setprio(1);
        read_block(at, scales, 0u, b[0], scale_b[0]);
#pragma unroll
        for (uint32_t j = 0; j < LIVE; j++) {
            asm volatile("" ::: "memory"); /* the reads below stay below the reads above, and above those of the next block */
            if (j + 1u < LIVE) {
                read_block(at, scales, j + 1u, b[j + 1u], scale_b[j + 1u]);
            }
#pragma unroll
            for (uint32_t part = 0; part < PARTS; part++) {
#pragma unroll
                for (uint32_t i = 0; i < PART; i++) {
                    const uint32_t t = part * PART + i;
                    const uint4_t first = set.words[t][0], second = set.words[t][HALVES - 1u];
                    const int8_vector a = {(int)first.x, (int)first.y, (int)first.z, (int)first.w, (int)second.x, (int)second.y, (int)second.z, (int)second.w};
                    if constexpr (B128) {
                        products[(j * PARTS + part) % 2u][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[j], (float4_t){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 127, 0, 127);
                    } else {
                        chain[t][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[j], chain[t][j], 0, 0, 0, (int)scale_a[t], 0, (int)scale_b[j]);
                    }
                }
                if constexpr (B128) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (j * PARTS + part != 0u) {
                        add(j * PARTS + part - 1u);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (B128) {
            add(LIVE * PARTS - 1u);
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the stage is read before the next barrier */
    }

    /* How many loads may be outstanding at the top of a K step for its columns and weights to have landed. Inside a step the
     * weights are asked for at its top, ahead of the barrier and the columns (in the middle of the matrix instructions 4-bit
     * weights take the same time and 18 registers more, one-byte weights a quarter longer). */
    template <uint32_t LIVE> using waits = native_waits<SLOTS, DEPTH, vector_loads(LIVE), WEIGHT_LOADS>;

    /* s_waitcnt takes its count as a constant: one instruction a count that loads_behind can come to */
    template <uint32_t LIVE, uint32_t WEIGHTS = 0, uint32_t VECTORS = 0>
    __device__ static __forceinline__ void wait_behind(uint32_t count)
    {
        if (count == WEIGHTS * WEIGHT_LOADS + VECTORS * vector_loads(LIVE)) {
            wait_loads<WEIGHTS * WEIGHT_LOADS + VECTORS * vector_loads(LIVE)>();
            return;
        }
        if constexpr (VECTORS + 1u < DEPTH - 1u) {
            wait_behind<LIVE, WEIGHTS, VECTORS + 1u>(count);
        } else if constexpr (WEIGHTS + 1u < SLOTS) {
            wait_behind<LIVE, WEIGHTS + 1u, 0u>(count);
        } else {
            wait_loads<0>(); /* not reached: every count is one of the above */
        }
    }

    /* K step `step` of `total` out of set K of the wavefront's sets of weight registers; the weights of step
     * `step` + SLOTS - 1 take the set the step before this one used */
    template <uint32_t LIVE, bool ONCE, uint32_t K>
    __device__ __forceinline__ void one_step(uint32_t step, uint32_t total, slot (&sets)[SLOTS], uint32_t (&held)[SCALE_LOADS], uint32_t round, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        wait_behind<LIVE>(waits<LIVE>::loads_behind(step, total));
        landed(sets[K]);
        if constexpr (BYTES && K == 0u) { /* the words were asked for ahead of the first round's weights, or have been waited for */
#pragma unroll
            for (uint32_t k = 0; k < SCALE_LOADS; k++) {
                native_landed(held[k]);
            }
        }
        const auto ask = [&]() { /* a function of its own: the compiler spills registers of the same lines without one */
            if (step + SLOTS - 1u < total) {
                issue_weights<ONCE>(sets[(K + SLOTS - 1u) % SLOTS], step + SLOTS - 1u);
            }
        };
        ask(); /* into the set the step before this one used: nothing of the block's is waited for */
        /* where the sets and the stages go round together the stage is a constant of the instance */
        const uint32_t stage = SLOTS % DEPTH == 0u ? K % DEPTH : step % DEPTH;
        __syncthreads(); /* every wavefront has read the step before; its columns of this one have landed */
        if (step + DEPTH - 1u < total) {
            issue_vectors<LIVE>((stage + DEPTH - 1u) % DEPTH, step + DEPTH - 1u);
        }
        if constexpr (BYTES) {
            consume_bytes<LIVE>(stage, step, sets[K], held, step - round, chain);
        } else {
            consume<LIVE>(stage, step, sets[K], chain);
        }
    }

    template <uint32_t LIVE, bool ONCE, uint32_t K>
    __device__ __forceinline__ void round_of_steps(uint32_t step, uint32_t total, slot (&sets)[SLOTS], uint32_t (&held)[SCALE_LOADS], uint32_t round, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        if (step + K < total) {
            one_step<LIVE, ONCE, K>(step + K, total, sets, held, round, chain);
        }
        if constexpr (K + 1u < SLOTS) {
            round_of_steps<LIVE, ONCE, K + 1u>(step, total, sets, held, round, chain);
        }
    }

    template <bool ONCE, uint32_t K>
    __device__ __forceinline__ void first_weights(uint32_t total, slot (&sets)[SLOTS]) const
    {
        if (K < total) {
            issue_weights<ONCE>(sets[K], K);
        }
        if constexpr (K + 2u < SLOTS) {
            first_weights<ONCE, K + 1u>(total, sets);
        }
    }

    template <uint32_t LIVE, bool ONCE>
    __device__ __forceinline__ void steps(uint32_t total, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        slot sets[SLOTS];
        uint32_t held[SCALE_LOADS], round = 0; /* one-byte weights: the scale words of the steps from `round` on */
        if constexpr (BYTES) {
            issue_weight_scales(held, 0u);
        }
#pragma unroll
        for (uint32_t i = 0; i < WAVE_BLOCKS; i++) {
            issue_scales(0u, i);
        }
#pragma unroll
        for (uint32_t k = 0; k + 1u < DEPTH; k++) {
            if (k < total) {
                issue_vectors<LIVE>(k, k);
            }
        }
        first_weights<ONCE, 0>(total, sets);
        for (uint32_t step = 0; step < total; step += SLOTS) {
            if (BYTES && step == round + SCALE_ROUND) { /* inputs past 128 SCALE_ROUND */
                round = step;
                issue_weight_scales(held, round);
                wait_loads<0>();
            }
            round_of_steps<LIVE, ONCE, 0>(step, total, sets, held, round, chain);
        }
    }

    template <uint32_t LIVE>
    __device__ __forceinline__ void steps_of(uint32_t total, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        if constexpr (STREAMS) {
            if (once) {
                steps<LIVE, true>(total, chain);
                return;
            }
        }
        steps<LIVE, false>(total, chain);
    }

    /* live_blocks: the column blocks that hold a pair, the same in every lane of the block */
    __device__ __forceinline__ void whole(uint32_t total, uint32_t live_blocks, float4_t (&chain)[TILES][COLUMN_BLOCKS]) const
    {
        if constexpr (COLUMN_BLOCKS == 4u) {
            switch (live_blocks) {
            case 1u: steps_of<1>(total, chain); break;
            case 2u: steps_of<2>(total, chain); break;
            case 3u: steps_of<3>(total, chain); break;
            default: steps_of<4>(total, chain); break;
            }
        } else {
            switch (live_blocks) {
            case 1u: steps_of<1>(total, chain); break;
            case 2u: steps_of<2>(total, chain); break;
            case 3u: steps_of<3>(total, chain); break;
            case 4u: steps_of<4>(total, chain); break;
            case 5u: steps_of<5>(total, chain); break;
            case 6u: steps_of<6>(total, chain); break;
            case 7u: steps_of<7>(total, chain); break;
            default: steps_of<8>(total, chain); break;
            }
        }
    }

    /* matrices: arena addresses of the stored matrices; the block's first strip is NATIVE_WAVES block_strip;
     * code_vectors[part]: the vector of column lane / 8 of this wavefront's group `part` of eight columns (group_of);
     * exponent_vectors[i]: the vector of column lane / 4 of its i-th column block */
    __device__ __forceinline__ void place(const unsigned char *const (&matrices)[MATRICES], uint32_t outputs, uint32_t inputs,
                                          uint32_t block_strip, const unsigned char *vector_codes, const unsigned char *vector_exponents,
                                          const uint32_t (&code_vectors)[2u * WAVE_BLOCKS], const uint32_t (&exponent_vectors)[WAVE_BLOCKS], uint32_t window_address,
                                          uint32_t wave_index, uint32_t lane, uint32_t &tile0_out)
    {
        const uint32_t tiles = outputs / 16u, steps = inputs / 128u;
        const uint32_t o = lane % 16u, g = lane / 16u;
        const uint32_t strip = block_strip * NATIVE_WAVES + wave_index;
        /* a strip that reaches past the last tile reads the last tiles again; its surplus sums are not stored */
        const uint32_t tile0 = strip * STRIP + STRIP <= tiles ? strip * STRIP : tiles > STRIP ? tiles - STRIP : 0u;
        tile0_out = tile0;
        tile_bytes = steps * STEP_BYTES;
        /* a matrix of one group of four tiles under strips of two groups: the second reads the first again */
        group_bytes = STRIP > 4u && tiles < STRIP ? 0u : 4u * tile_bytes;
        scale_stride = STRIP > 4u && tiles < STRIP ? 0u : steps * 256u;
        step_stride = STEP_BYTES;
        window = window_address;
        wave = wave_index;
        codes = vector_codes;
        exponents = vector_exponents;
#pragma unroll
        for (uint32_t m = 0; m < MATRICES; m++) {
            words[m] = matrices[m] + (uint64_t)tile0 * tile_bytes;
            if constexpr (B128) { /* float32 [outputs / 128][inputs / 128] behind the codes: the strip's row, a word a K step */
                scales[m] = matrices[m] + (uint64_t)outputs * inputs + (uint64_t)(tile0 / 8u) * (inputs / 32u);
            } else if constexpr (BYTES) { /* the scale codes as the reference stores them: a row of inputs / 32 bytes for every 32 outputs */
                scales[m] = matrices[m] + (uint64_t)outputs * inputs + (uint64_t)(tile0 / 2u) * (inputs / 32u);
            } else { /* a word a lane a K step of a group of four tiles */
                scales[m] = matrices[m] + (uint64_t)outputs * inputs / 2u + (uint64_t)(tile0 / 4u) * steps * 256u;
            }
        }
        word_offset = 16u * lane;
        if constexpr (BYTES && !B128) {
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n++) {
                scale_offset[n] = ((tile0 + n) / 2u - tile0 / 2u) * (inputs / 32u);
            }
        } else {
            scale_offset[0] = B128 ? 0u : 4u * lane;
        }
        code_shift = 8u * g;
#pragma unroll
        for (uint32_t part = 0; part < 2u * WAVE_BLOCKS; part++) {
            codes_offset[part] = code_vectors[part] * inputs + 16u * ((lane % 8u) ^ (lane / 8u) ^ (group_of(wave_index, part) % 2u));
        }
#pragma unroll
        for (uint32_t i = 0; i < WAVE_BLOCKS; i++) {
            exponents_offset[i] = exponent_vectors[i] * (inputs / 32u);
        }
        last_step = steps - 1u;
        lane_of = lane;
        const uint32_t column = o % 8u, group_bytes = (o / 8u) * 1024u;
        if constexpr (BYTES) {
#pragma unroll
            for (uint32_t v = 0; v < 8u; v++) {
                vector_at[v] = window + group_bytes + 16u * (8u * column + (v ^ column ^ (o / 8u))) + 4u * g;
            }
        } else {
#pragma unroll
            for (uint32_t part = 0; part < (PIECES_HELD ? 4u : 1u); part++) {
                vector_at[part] = (window + group_bytes + 16u * (8u * column + (2u * (g % 2u) ^ column ^ (o / 8u))) + 8u * (g / 2u)) ^ piece_of(part);
            }
        }
        vector_scale_at = window + 4u * SCALE_STEPS * o + (B128 ? 0u : g);
        scale_shift = 8u * (tile0 % 4u);
    }
};

#endif
