/*
 * wide_finish_device.cuh -- what a block of the wide routed experts does with its sums, shared by the kernels of the
 * reference's weight formats (kernel_wide_linear.hip) and of gfx950's own (kernel_native_linear.hip): the gate/up
 * launch's hidden step and quantizer from the registers the sums are in, the down launch's stores. A block's columns are
 * `pair_count` sorted pairs (COLUMN_BLOCKS blocks of 16 at most), which the block holds in LDS (`columns`); chain[t][j]:
 * tile t of the wavefront's strip (gate's STRIP tiles, then up's) by column block j, a lane holding rows
 * 4 (lane / 16) .. + 3 of column lane % 16.
 *
 * A wavefront here has no other of its block to hide behind, so what a column block costs is its instructions and its
 * round trips to memory. The pairs come from LDS: a load from memory behind the stores of the column block before it waits
 * for those stores too (both count in vmcnt), which made the finish as long as a chain of 32 K steps. Values are rounded
 * two at a time, no comparison is spent on a value that is not a number or needs the quantizer's limits (one test a
 * column block, the same in every lane of the wavefront, and the definition's steps behind it), and the lanes that hold
 * a word's halves exchange them by one v_permlane32_swap, so that a lane stores 16 bytes of codes and of operands:
 * 69 -> 31 vector instructions a hidden value, 28 -> 4 stores a column block of four tiles.
 */
#ifndef WIDE_FINISH_DEVICE_CUH
#define WIDE_FINISH_DEVICE_CUH

#include "linear_device.cuh"
#include "quantize_device.cuh"

#ifndef WIDE_WAVES
#define WIDE_WAVES 4u
#endif

/* two float32 as bfloat16 in one word, to nearest even (first in the low half); a value that is not a number keeps none
 * of float_to_bf16's promises: the caller looks for those */
__device__ static __forceinline__ uint32_t wide_round_pair(float first, float second)
{
    typedef float pair_of_floats __attribute__((ext_vector_type(2)));
    typedef __bf16 pair_of_bf16 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((pair_of_floats){first, second}, pair_of_bf16));
}

__device__ static __forceinline__ float wide_low(uint32_t pair)
{
    return __uint_as_float(pair << 16);
}

__device__ static __forceinline__ float wide_high(uint32_t pair)
{
    return __uint_as_float(pair & 0xFFFF0000u);
}

/* the smaller of a value and a limit, the limit for a value that is not a number: fminf, without the copy the compiler
 * puts before it to quieten a signalling one (a value here is a conversion's result) */
__device__ static __forceinline__ float wide_at_most(float value, float limit)
{
    float result;
    asm("v_min_f32 %0, %1, %2" : "=v"(result) : "v"(limit), "v"(value));
    return result;
}

/* the largest of a value over the four lanes of a column (lane % 16), in each of them */
__device__ static __forceinline__ float wide_column_largest(float value)
{
    const auto near_rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(value), __float_as_uint(value), false, false);
    const float two = fmaxf(__uint_as_float(near_rows[0]), __uint_as_float(near_rows[1]));
    const auto far_rows = __builtin_amdgcn_permlane32_swap(__float_as_uint(two), __float_as_uint(two), false, false);
    return fmaxf(__uint_as_float(far_rows[0]), __uint_as_float(far_rows[1]));
}

/* COUNT words of a lane to consecutive addresses */
template <uint32_t COUNT>
__device__ static __forceinline__ void wide_store_words(unsigned char *to, const uint32_t (&words)[COUNT])
{
    if constexpr (COUNT % 4u == 0u) {
#pragma unroll
        for (uint32_t k = 0; k < COUNT; k += 4u) {
            *(uint4_t *)(to + 4u * k) = (uint4_t){words[k], words[k + 1u], words[k + 2u], words[k + 3u]};
        }
    } else if constexpr (COUNT == 2u) {
        *(uint2_t *)to = (uint2_t){words[0], words[1]};
    } else {
        static_assert(COUNT == 1u, "one, two or a multiple of four words");
        *(uint32_t *)to = words[0];
    }
}

/* the quantizer's step on STRIP tiles' values of one column: hidden[n][i] = values 2 i and 2 i + 1 of the lane's four of
 * tile n, code_exponent[n / 2]; `limited`, the same in every lane: some value needs the definition's limits. Codes are
 * bytes 2 (v % 2) + g / 2 of a word (g: the lane's row group), so the lanes g and g ^ 2 of a column hold the halves of the
 * same two words: the lower takes the first whole, the upper the second; the tiles of a strip are neighbouring words. */
template <uint32_t STRIP, uint32_t SCALES>
__device__ static __forceinline__ void wide_quantize_column(const uint32_t (&hidden)[STRIP][2], const uint32_t (&code_exponent)[SCALES], bool limited,
                                                            uint32_t tile0, uint32_t lane, unsigned char *codes, unsigned char *operands)
{
    const uint32_t g = lane / 16u, upper = g / 2u;
    uint32_t code_words[STRIP], operand_words[2u * STRIP];
#pragma unroll
    for (uint32_t n = 0; n < STRIP; n++) {
        const uint32_t exponent = code_exponent[SCALES == 1u ? 0u : n / 2u];
        uint32_t own, low_pair, high_pair;
        if (limited) {
            uint32_t carried[4];
            const uint32_t bits[4] = {hidden[n][0] & 0xFFFFu, hidden[n][0] >> 16, hidden[n][1] & 0xFFFFu, hidden[n][1] >> 16};
            quantize_codes4(bits, exponent, own, carried);
            low_pair = quantize_operand_pair(carried[0], carried[1], exponent);
            high_pair = quantize_operand_pair(carried[2], carried[3], exponent);
        } else { /* every value a number, every scaled value at most 448, every operand finite */
            const float down = __uint_as_float((254u - exponent) << 23), up = __uint_as_float((exponent + 100u) << 23);
            int packed = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(wide_low(hidden[n][0]), down), __fmul_rn(wide_high(hidden[n][0]), down), 0, false);
            packed = __builtin_amdgcn_cvt_pk_fp8_f32(__fmul_rn(wide_low(hidden[n][1]), down), __fmul_rn(wide_high(hidden[n][1]), down), packed, true);
            own = (uint32_t)packed;
            const auto low = __builtin_amdgcn_cvt_pk_f32_fp8(packed, false), high = __builtin_amdgcn_cvt_pk_f32_fp8(packed, true);
            low_pair = __builtin_amdgcn_perm(__float_as_uint(__fmul_rn(low[1], up)), __float_as_uint(__fmul_rn(low[0], up)), 0x07060302u);
            high_pair = __builtin_amdgcn_perm(__float_as_uint(__fmul_rn(high[1], up)), __float_as_uint(__fmul_rn(high[0], up)), 0x07060302u);
        }
        /* the lower lane's code word in every lane, and the upper lane's: (a0, b0, a1, b1) or (a2, b2, a3, b3) of them */
        const auto both = __builtin_amdgcn_permlane32_swap(own, own, false, false);
        code_words[n] = __builtin_amdgcn_perm(both[1], both[0], upper != 0u ? 0x07030602u : 0x05010400u);
        /* lower lanes: the first pairs of both; upper lanes: the second pairs of both */
        const auto pairs_of = __builtin_amdgcn_permlane32_swap(low_pair, high_pair, false, false);
        operand_words[2u * n] = pairs_of[0];
        operand_words[2u * n + 1u] = pairs_of[1];
    }
    const uint32_t word = quantize_word_of(tile0 / 4u, tile0 % 4u, 2u * (g % 2u) + upper);
    wide_store_words<STRIP>(codes + word, code_words);
    wide_store_words<2u * STRIP>(operands + 2u * word, operand_words);
}

/* window: the block's LDS window, free once the K steps are done (one tile a strip: the two wavefronts of a quantizer
 * block pass each other their halves' largest magnitude through it; every wavefront of the block calls together) */
template <uint32_t STRIP, uint32_t COLUMN_BLOCKS, bool B128>
__device__ static __forceinline__ void wide_gate_up_finish(const struct wide_expert_gate_up_arguments &arguments, unsigned char *arena,
                                                           unsigned char *window, const struct wide_pair *columns, uint32_t pair_count,
                                                           uint32_t block_strip, uint32_t tile0, uint32_t wave, uint32_t lane,
                                                           float4_t (&chain)[2u * STRIP][COLUMN_BLOCKS])
{
    static_assert(STRIP == 1u || STRIP == 2u || STRIP == 4u, "a strip is half a quantizer block of 32 outputs, one or two");
    constexpr uint32_t STRIP_OUTPUTS = STRIP * 16u;
    /* The hidden step, as expert_gate_up_1 rounds it (the one chain is added to +0 first, as S chains are), and the
     * quantizer's step on it, from the registers the sums are in. A lane holds, of a column of every column block, rows
     * 4 (lane / 16) .. + 3 of the strip's tiles. Two tiles: the 32 outputs of one quantizer block are the 8
     * values of each of the 4 lanes of a column. One tile a strip: the block is the strips of the wavefronts 2 p and
     * 2 p + 1 (the matrix holds whole blocks of 32 outputs: both are inside it or neither), which pass each other the
     * largest magnitude of their halves through LDS. A strip that reaches past the matrix has begun at the last tiles
     * again (tile0): what it stores of them is what the strip before it stores. */
    const uint32_t width = arguments.output_size;
    const bool strip_is_live = (block_strip * WIDE_WAVES + wave) * STRIP_OUTPUTS < width; /* else: a strip wholly past the matrix */
    const float limit = arguments.activation_limit;
    const uint32_t g = lane / 16u;
    /* column block j: the hidden values of the lane's rows of its column, in pairs; returns whether one of them is not a
     * number, the same in every lane */
    const auto hidden_of = [&](float weight, uint32_t j, uint32_t (&hidden)[STRIP][2]) -> bool {
        bool unordered = false;
#pragma unroll
        for (uint32_t n = 0; n < STRIP; n++) {
#pragma unroll
            for (uint32_t i = 0; i < 2u; i++) {
                const uint32_t gates = wide_round_pair(__fadd_rn(0.0f, chain[n][j][2u * i]), __fadd_rn(0.0f, chain[n][j][2u * i + 1u]));
                const uint32_t ups = wide_round_pair(__fadd_rn(0.0f, chain[STRIP + n][j][2u * i]), __fadd_rn(0.0f, chain[STRIP + n][j][2u * i + 1u]));
                /* the median of a value that is not a number and two limits is the lower: fminf(fmaxf(up, -limit), limit) */
                const float up0 = __builtin_amdgcn_fmed3f(wide_low(ups), -limit, limit), up1 = __builtin_amdgcn_fmed3f(wide_high(ups), -limit, limit);
                const float value0 = __fmul_rn(__fmul_rn(linear_silu(wide_at_most(wide_low(gates), limit)), up0), weight);
                const float value1 = __fmul_rn(__fmul_rn(linear_silu(wide_at_most(wide_high(gates), limit)), up1), weight);
                hidden[n][i] = wide_round_pair(value0, value1);
                unordered = unordered || __builtin_isunordered(value0, value1);
            }
        }
        if (__builtin_amdgcn_ballot_w64(unordered) == 0ull) {
            return false;
        }
#pragma unroll
        for (uint32_t n = 0; n < STRIP; n++) {
#pragma unroll
            for (uint32_t i = 0; i < 2u; i++) { /* float_to_bf16's one value that is not a number */
                const uint32_t low = (hidden[n][i] & 0x7FFFu) > 0x7F80u ? 0x7FC0u : hidden[n][i] & 0xFFFFu;
                const uint32_t high = (hidden[n][i] & 0x7FFF0000u) > 0x7F800000u ? 0x7FC00000u : hidden[n][i] & 0xFFFF0000u;
                hidden[n][i] = high | low;
            }
        }
        return true;
    };
    const auto tiles_largest = [&](const uint32_t (&hidden)[STRIP][2], uint32_t n) -> float {
        return fmaxf(fmaxf(fabsf(wide_low(hidden[n][0])), fabsf(wide_high(hidden[n][0]))),
                     fmaxf(fabsf(wide_low(hidden[n][1])), fabsf(wide_high(hidden[n][1]))));
    };
    if constexpr (B128) {
        /* the hidden values themselves, where the record names the hidden operands (bfloat16 [pair][width] either way):
         * this format's quantizer takes 128 values a scale, in a launch of its own */
        if (!strip_is_live) {
            return;
        }
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            const uint32_t column = 16u * j + lane % 16u;
            if (column < pair_count) {
                const struct wide_pair pair = columns[column];
                uint32_t hidden[STRIP][2];
                (void)hidden_of(pair.route_weight, j, hidden);
                uint16_t *values = (uint16_t *)(arena + arguments.hidden_operands_offset) + (uint64_t)pair.pair_index * width;
#pragma unroll
                for (uint32_t n = 0; n < STRIP; n++) {
                    *(uint2_t *)(values + (tile0 + n) * 16u + 4u * g) = (uint2_t){hidden[n][0], hidden[n][1]};
                }
            }
        }
        return;
    } else if constexpr (STRIP >= 2u) {
        if (!strip_is_live) {
            return;
        }
        /* the quantizer blocks are this wavefront's own: a column block at a time */
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            const uint32_t column = 16u * j + lane % 16u;
            if (column < pair_count) { /* the same in the four lanes of a column */
                const struct wide_pair pair = columns[column];
                uint32_t hidden[STRIP][2], code_exponent[STRIP / 2u];
                const bool unordered = hidden_of(pair.route_weight, j, hidden);
                bool large = false;
#pragma unroll
                for (uint32_t k = 0; k < STRIP / 2u; k++) {
                    code_exponent[k] = quantize_exponent_code(wide_column_largest(fmaxf(tiles_largest(hidden, 2u * k), tiles_largest(hidden, 2u * k + 1u))));
                    large = large || code_exponent[k] > 146u;
                }
                const bool limited = unordered || __builtin_amdgcn_ballot_w64(large) != 0ull;
                const uint64_t first = (uint64_t)pair.pair_index * width;
                wide_quantize_column<STRIP, STRIP / 2u>(hidden, code_exponent, limited, tile0, lane, arena + arguments.hidden_codes_offset + first,
                                                        arena + arguments.hidden_operands_offset + 2u * first);
                if (g == 0u) {
                    unsigned char *exponents = arena + arguments.hidden_exponents_offset + (first + 16u * tile0) / 32u;
#pragma unroll
                    for (uint32_t k = 0; k < STRIP / 2u; k++) {
                        exponents[k] = (unsigned char)code_exponent[k];
                    }
                }
            }
        }
        return;
    } else {
        uint32_t hidden[COLUMN_BLOCKS][STRIP][2];
        float largest[COLUMN_BLOCKS];
        bool unordered = false;
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            const uint32_t column = 16u * j + lane % 16u;
            largest[j] = 0.0f;
            if (column < pair_count && strip_is_live) {
                unordered = hidden_of(columns[column].route_weight, j, hidden[j]) || unordered;
                largest[j] = wide_column_largest(tiles_largest(hidden[j], 0u));
            }
        }
        float *halves = (float *)window; /* [wavefront][column]: the stages are done with */
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            if (g == 0u) {
                halves[wave * (COLUMN_BLOCKS * 16u) + 16u * j + lane] = largest[j];
            }
        }
        __syncthreads();
        if (!strip_is_live) {
            return;
        }
#pragma unroll
        for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
            const uint32_t column = 16u * j + lane % 16u;
            if (column < pair_count) {
                const uint32_t code_exponent[1] = {quantize_exponent_code(fmaxf(largest[j], halves[(wave ^ 1u) * (COLUMN_BLOCKS * 16u) + column]))};
                const bool limited = __builtin_amdgcn_ballot_w64(unordered || code_exponent[0] > 146u) != 0ull;
                const uint64_t first = (uint64_t)columns[column].pair_index * width;
                wide_quantize_column<STRIP, 1u>(hidden[j], code_exponent, limited, tile0, lane, arena + arguments.hidden_codes_offset + first,
                                                arena + arguments.hidden_operands_offset + 2u * first);
                if (g == 0u && tile0 % 2u == 0u) {
                    (arena + arguments.hidden_exponents_offset)[(first + 16u * tile0) / 32u] = (unsigned char)code_exponent[0];
                }
            }
        }
    }
}

/* Two tiles a time: the lanes of a column hold four rows of each, and one v_permlane16_swap a word gives each of them
 * eight rows of one of the two, so that a lane stores 16 bytes. */
template <uint32_t STRIP, uint32_t COLUMN_BLOCKS>
__device__ static __forceinline__ void wide_down_finish(const struct wide_expert_down_arguments &arguments, unsigned char *arena,
                                                        const struct wide_pair *columns, uint32_t pair_count, uint32_t block_strip,
                                                        uint32_t tile0, uint32_t wave, uint32_t lane, float4_t (&chain)[STRIP][COLUMN_BLOCKS])
{
    static_assert(STRIP % 2u == 0u, "tiles are stored two at a time");
    constexpr uint32_t STRIP_OUTPUTS = STRIP * 16u;
    if ((block_strip * WIDE_WAVES + wave) * STRIP_OUTPUTS >= arguments.output_size) {
        return; /* a strip wholly past the matrix; one that reaches past it has begun at the last tiles again (tile0) and
                 * stores of them what the strip before it stores */
    }
    const uint32_t g = lane / 16u;
#pragma unroll
    for (uint32_t j = 0; j < COLUMN_BLOCKS; j++) {
        const uint32_t column = 16u * j + lane % 16u;
        if (column < pair_count) {
            uint16_t *out = (uint16_t *)(arena + arguments.output_offset) + (uint64_t)columns[column].pair_index * arguments.output_size + tile0 * 16u;
            uint32_t words[STRIP][2];
            bool unordered = false;
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n++) {
#pragma unroll
                for (uint32_t i = 0; i < 2u; i++) {
                    const float first = __fadd_rn(0.0f, chain[n][j][2u * i]), second = __fadd_rn(0.0f, chain[n][j][2u * i + 1u]);
                    words[n][i] = wide_round_pair(first, second);
                    unordered = unordered || __builtin_isunordered(first, second);
                }
            }
            if (__builtin_amdgcn_ballot_w64(unordered) != 0ull) {
#pragma unroll
                for (uint32_t n = 0; n < STRIP; n++) {
#pragma unroll
                    for (uint32_t i = 0; i < 2u; i++) {
                        words[n][i] = (uint32_t)float_to_bf16(__fadd_rn(0.0f, chain[n][j][2u * i])) |
                                      ((uint32_t)float_to_bf16(__fadd_rn(0.0f, chain[n][j][2u * i + 1u])) << 16);
                    }
                }
            }
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n += 2u) {
                if (STRIP > 4u && n >= 4u && arguments.output_size < STRIP_OUTPUTS) {
                    continue; /* a matrix of one group of four tiles: the strip's second group is the first again */
                }
                const auto first = __builtin_amdgcn_permlane16_swap(words[n][0], words[n + 1u][0], false, false);
                const auto second = __builtin_amdgcn_permlane16_swap(words[n][1], words[n + 1u][1], false, false);
                *(uint4_t *)(out + (n + g % 2u) * 16u + 8u * (g / 2u)) = (uint4_t){first[0], second[0], first[1], second[1]};
            }
        }
    }
}

#endif
