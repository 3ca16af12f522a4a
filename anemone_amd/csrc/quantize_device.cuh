/*
 * quantize_device.cuh -- one value of the per-32 activation quantizer (source/kernel_activation_quantize.cuh:52-133,
 * include/anemone/linear_records.h:20-44 of the reference), shared by the quantizer's own kernel and by the producer
 * (gate with up and the quantization of the hidden vectors in one launch). The 32 values of a block sit in 32
 * consecutive lanes of a wavefront (lane % 32 = index % 32); every lane calls with its value.
 */
#ifndef QUANTIZE_DEVICE_CUH
#define QUANTIZE_DEVICE_CUH

#include "exl3_device.cuh"

/* the scale code of a block whose largest magnitude is `largest`: the smallest power of two at least
 * max(largest, 1e-4) / 448, as its biased exponent */
__device__ static __forceinline__ uint32_t quantize_exponent_code(float largest)
{
    const uint32_t ratio = __float_as_uint(__fmul_rn(fmaxf(largest, 1e-4f), 1.0f / 448.0f));
    return ((ratio >> 23) & 255u) + ((ratio & 0x7FFFFFu) != 0u ? 1u : 0u);
}

/* one bfloat16 value under its block's scale code: its E4M3 code (to nearest even, clamped at 448) and its operand.
 * The definition, in plain arithmetic; the kernels use quantize_codes4 below, which the library's arithmetic_selfcheck
 * kernel compares with it over every value and every scale code. */
__device__ static __forceinline__ void quantize_code_defined(uint32_t bits, uint32_t code_exponent, uint32_t &code_out, uint32_t &operand_out)
{
    const float value = bf16_to_float((uint16_t)bits);
    const float scaled = __fmul_rn(value, __uint_as_float((254u - code_exponent) << 23)); /* exact: a power of two */
    const float magnitude = fminf(fabsf(scaled), 448.0f);
    const uint32_t field = __float_as_uint(fmaxf(magnitude, 0.015625f)) >> 23; /* at least 2^-6's */
    /* units of 1/8 of the binade (2^-9 below 2^-6): 0 .. 16, to nearest even */
    const uint32_t units = (uint32_t)__builtin_rintf(__fmul_rn(magnitude, __uint_as_float((257u - field) << 23)));
    const uint32_t sign = (bits >> 8) & 0x80u;
    code_out = (((field - 120u) << 3) + units - 8u) | sign;
    /* the operand: units x 2^(field - 130) x 2^(c - 127) x 2^100, exact, its upper half a bfloat16 */
    const float carried = __fmul_rn((float)units, __uint_as_float((field + code_exponent - 30u) << 23));
    operand_out = (code_exponent <= 146u ? __float_as_uint(carried) >> 16 : 0x7F80u) | (sign << 8);
}

/* Four values of one block at once, by the card's own conversions: the scaled value, limited to 448 in magnitude (a
 * NaN becomes 448) under the value's sign, goes through v_cvt_pk_fp8_f32 (E4M3, to nearest even, subnormals of 2^-9);
 * the operand is the code converted back (v_cvt_pk_f32_fp8) times 2^(c - 27), exact, whose upper half is the
 * bfloat16. codes: byte i the code of bits[i]; carried[i]: the operand of bits[i] in the upper half of the word, to be
 * paired by quantize_operand_pair. */
__device__ static __forceinline__ void quantize_codes4(const uint32_t (&bits)[4], uint32_t code_exponent, uint32_t &codes, uint32_t (&carried)[4])
{
    const float down = __uint_as_float((254u - code_exponent) << 23);
    const float up = __uint_as_float(((code_exponent <= 146u ? code_exponent : 146u) + 100u) << 23);
    float held[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const uint32_t value = bits[i] << 16;
        const float magnitude = fminf(fabsf(__fmul_rn(__uint_as_float(value), down)), 448.0f);
        held[i] = __uint_as_float((__float_as_uint(magnitude) & 0x7FFFFFFFu) | (value & 0x80000000u));
    }
    int packed = __builtin_amdgcn_cvt_pk_fp8_f32(held[0], held[1], 0, false);
    packed = __builtin_amdgcn_cvt_pk_fp8_f32(held[2], held[3], packed, true);
    codes = (uint32_t)packed;
    const auto low = __builtin_amdgcn_cvt_pk_f32_fp8(packed, false), high = __builtin_amdgcn_cvt_pk_f32_fp8(packed, true);
    carried[0] = __float_as_uint(__fmul_rn(low[0], up));
    carried[1] = __float_as_uint(__fmul_rn(low[1], up));
    carried[2] = __float_as_uint(__fmul_rn(high[0], up));
    carried[3] = __float_as_uint(__fmul_rn(high[1], up));
}

/* two operands as one word (first in the low half); a scale code above 146 makes every operand an infinity of its sign */
__device__ static __forceinline__ uint32_t quantize_operand_pair(uint32_t first, uint32_t second, uint32_t code_exponent)
{
    const uint32_t pair = __builtin_amdgcn_perm(second, first, 0x07060302u);
    return code_exponent <= 146u ? pair : (pair & 0x80008000u) | 0x7F807F80u;
}

/* one value by the same route (the three others zero) */
__device__ static __forceinline__ void quantize_code(uint32_t bits, uint32_t code_exponent, uint32_t &code_out, uint32_t &operand_out)
{
    const uint32_t four[4] = {bits, 0u, 0u, 0u};
    uint32_t codes, carried[4];
    quantize_codes4(four, code_exponent, codes, carried);
    code_out = codes & 0xFFu;
    operand_out = quantize_operand_pair(carried[0], 0u, code_exponent) & 0xFFFFu;
}

/* The quantizer of 128 values a float32 scale: value / scale with one rounding. A division's own value from the divisor's rounded
 * reciprocal, the product with it and a correction by that product's remainder (P. Markstein, Computation of elementary
 * functions on the IBM RISC System/6000 processor, 1990), where neither the remainder nor the reciprocal leaves the normal
 * range. Of a value or a quotient below 2^-100 it may come out a place or so apart: then the quotient is below 2^-64 (a scale is
 * at least 1e-4 / 448), far under half of the smallest code. A scale of infinity divides. arithmetic_selfcheck compares it with the division over every value under every scale there is. The
 * divisions of a thread's four values were vector issue (16384 vectors of 2048 values 42 -> 37 us, 2048 of 4096 13.2 -> 11.7). */
__device__ static __forceinline__ float quantize_quotient(float value, float scale, float reciprocal)
{
    const float near = __fmul_rn(value, reciprocal);
    return scale <= 3.402823466e38f ? __fmaf_rn(__fmaf_rn(-near, scale, value), reciprocal, near) : __fdiv_rn(value, scale);
}

/* such a quotient's E4M3 code under its value's sign: limited to 448 (a not-a-number too), to nearest even */
__device__ static __forceinline__ uint32_t quantize_quotient_code(float quotient, uint32_t bits)
{
    const float magnitude = fminf(fabsf(quotient), 448.0f);
    const uint32_t field = __float_as_uint(fmaxf(magnitude, 0.015625f)) >> 23;
    const uint32_t units = (uint32_t)__builtin_rintf(__fmul_rn(magnitude, __uint_as_float((257u - field) << 23)));
    return (((field - 120u) << 3) + units - 8u) | ((bits >> 8) & 0x80u);
}

/* where the values of a vector go: value `index` = 64 load + 16 step + u lies in word ((4 load + t) 4 + step) with
 * t = (u % 8) / 2: its code at byte 2 (u % 2) + u / 8 of the word, its operand at halfword 2 (u / 8) + u % 2 of the
 * word's four */
__device__ static __forceinline__ uint32_t quantize_word_of(uint32_t load, uint32_t step, uint32_t t)
{
    return ((4u * load + t) * 4u + step) * 4u;
}

/* bits: the bfloat16 value at `index` of a vector of `width` values; codes, exponents, operands: the vector's arrays */
__device__ static __forceinline__ void quantize_value(uint32_t bits, uint32_t index, unsigned char *codes, unsigned char *exponents,
                                                      uint16_t *operands)
{
    float largest = fabsf(bf16_to_float((uint16_t)bits));
    largest = lanes_largest<1u>(lanes_largest<2u>(lanes_largest<4u>(lanes_largest<8u>(lanes_largest<16u>(largest)))));
    const uint32_t code_exponent = quantize_exponent_code(largest);
    uint32_t code, operand;
    quantize_code(bits, code_exponent, code, operand);
    const uint32_t u = index % 16u, word = quantize_word_of(index / 64u, (index % 64u) / 16u, (u % 8u) / 2u);
    codes[word + 2u * (u % 2u) + u / 8u] = (unsigned char)code;
    operands[word + 2u * (u / 8u) + u % 2u] = (uint16_t)operand;
    if (index % 32u == 0u) {
        exponents[index / 32u] = (unsigned char)code_exponent;
    }
}

/* the first of the four values +0, +1, +8, +9 of thread q of a vector: thread q = (16 l + 4 s + t) takes 64 l + 16 s + 2 t + {0, 1, 8, 9}, the
 * four codes of one word of the lane order and the four operands of one pair of words; the 32 values of a block of the
 * quantization are those of eight neighbouring threads (s = 2 b, 2 b + 1; t = 0 .. 3) */
__device__ static __forceinline__ uint32_t quantize_first_of(uint32_t q)
{
    return 64u * (q / 16u) + 16u * (q / 4u % 4u) + 2u * (q % 4u);
}

/* activation_quantize_entry's work of thread q of vector `vector` from its four values on; the eight threads of a block of
 * 32 values are neighbours in one wavefront and call together */
__device__ static __forceinline__ void activation_quantize_values(const struct activation_quantize_arguments &arguments, unsigned char *arena,
                                                                  uint32_t q, uint64_t vector, const uint32_t (&bits)[4])
{
    const uint32_t l = q / 16u, s = (q / 4u) % 4u, t = q % 4u, first = quantize_first_of(q);
    float largest = fmaxf(fmaxf(fabsf(bf16_to_float((uint16_t)bits[0])), fabsf(bf16_to_float((uint16_t)bits[1]))),
                          fmaxf(fabsf(bf16_to_float((uint16_t)bits[2])), fabsf(bf16_to_float((uint16_t)bits[3]))));
    largest = lanes_largest<1u>(lanes_largest<2u>(lanes_largest<4u>(largest)));
    const uint32_t code_exponent = quantize_exponent_code(largest);
    /* the word's bytes j = 0 .. 3 hold values +0 (j = 0), +8 (1), +1 (2), +9 (3); its operands' halfwords 2 r + h hold
     * value + h + 8 r */
    const uint32_t in_word_order[4] = {bits[0], bits[2], bits[1], bits[3]};
    uint32_t codes, carried[4];
    quantize_codes4(in_word_order, code_exponent, codes, carried);
    const uint32_t word = quantize_word_of(l, s, t);
    *(uint32_t *)(arena + arguments.codes_offset + vector * arguments.width + word) = codes;
    *(uint2_t *)((uint16_t *)(arena + arguments.operands_offset) + vector * arguments.width + word) =
        (uint2_t){quantize_operand_pair(carried[0], carried[2], code_exponent), quantize_operand_pair(carried[1], carried[3], code_exponent)};
    if (q % 8u == 0u) {
        (arena + arguments.exponents_offset)[vector * (arguments.width / 32u) + first / 32u] = (unsigned char)code_exponent;
    }
}

/* thread q of a vector's width / 4 of vector `vector` */
__device__ static __forceinline__ void activation_quantize_body(const struct activation_quantize_arguments &arguments, unsigned char *arena,
                                                                uint32_t q, uint64_t vector)
{
    const uint32_t first = quantize_first_of(q);
    if (first >= arguments.width) {
        return; /* the width is a multiple of 64: whole groups of sixteen threads leave together */
    }
    const uint16_t *values = (const uint16_t *)(arena + arguments.values_offset) + vector * arguments.width + first;
    const uint32_t near_pair = *(const uint32_t *)values, far_pair = *(const uint32_t *)(values + 8);
    const uint32_t bits[4] = {near_pair & 0xFFFFu, near_pair >> 16, far_pair & 0xFFFFu, far_pair >> 16};
    activation_quantize_values(arguments, arena, q, vector, bits);
}

/* thread q of vector `vector`: activation_quantize_128_entry's work of one thread */
__device__ static __forceinline__ void activation_quantize_128_body(const struct activation_quantize_arguments &arguments, unsigned char *arena,
                                                                    uint32_t q, uint64_t vector)
{
    /* the threads' values as in activation_quantize_entry: thread q = 16 l + 4 s + t takes 64 l + 16 s + 2 t + {0, 1, 8, 9},
     * one word of codes; the 128 values of a scale are those of 32 neighbouring threads */
    const uint32_t l = q / 16u, s = (q / 4u) % 4u, t = q % 4u, first = 64u * l + 16u * s + 2u * t;
    if (first >= arguments.width) {
        return; /* the width is a multiple of 128: whole groups of 32 threads leave together */
    }
    const uint16_t *values = (const uint16_t *)(arena + arguments.values_offset) + vector * arguments.width + first;
    const uint32_t near_pair = *(const uint32_t *)values, far_pair = *(const uint32_t *)(values + 8);
    const uint32_t bits[4] = {near_pair & 0xFFFFu, near_pair >> 16, far_pair & 0xFFFFu, far_pair >> 16};
    float largest = fmaxf(fmaxf(fabsf(bf16_to_float((uint16_t)bits[0])), fabsf(bf16_to_float((uint16_t)bits[1]))),
                          fmaxf(fabsf(bf16_to_float((uint16_t)bits[2])), fabsf(bf16_to_float((uint16_t)bits[3]))));
    largest = lanes_largest<1u>(lanes_largest<2u>(lanes_largest<4u>(lanes_largest<8u>(lanes_largest<16u>(largest)))));
    const float scale = __fdiv_rn(fmaxf(largest, 1e-4f), 448.0f);
    const float reciprocal = __fdiv_rn(1.0f, scale);
    uint32_t code[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        code[i] = quantize_quotient_code(quantize_quotient(bf16_to_float((uint16_t)bits[i]), scale, reciprocal), bits[i]);
    }
    *(uint32_t *)(arena + arguments.codes_offset + vector * arguments.width + quantize_word_of(l, s, t)) =
        code[0] | (code[2] << 8) | (code[1] << 16) | (code[3] << 24); /* bytes: values +0, +8, +1, +9 */
    if (q % 32u == 0u) {
        ((float *)(arena + arguments.exponents_offset))[vector * (arguments.width / 128u) + first / 128u] = scale;
    }
}

#endif
