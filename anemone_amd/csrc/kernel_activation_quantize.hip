/*
 * kernel_activation_quantize.hip -- the per-32 activation quantizer of the FP4 / FP8 linears on gfx950.
 * Entry name, record and every written byte follow the reference (source/kernel_activation_quantize.cuh:52-133,
 * include/anemone/linear_records.h:20-44): for each block of 32 consecutive bfloat16 values, all in float32,
 *   m = max(largest magnitude, 1e-4) x float32(1 / 448); the exponent code c is the exponent of m, one more unless
 *   m is a power of two; each value is divided by 2^(c - 127) (exact), limited to 448 and rounded to the nearest E4M3
 *   number, a tie to the even code, the sign kept also on a zero.
 * Written: codes [v][width] in LANE ORDER (byte ((4 l + t) 4 + s) 4 + j holds value 64 l + 16 s + 2 t + j / 2 +
 * 8 (j % 2)), exponents [v][width / 32], operands [v][width] (bfloat16 of the value's code x scale x 2^100, in
 * OPERAND ORDER; an infinity of the sign where c is above 146). The operands are not read by this library's own
 * kernels; they are written because the record's contract writes them on every card.
 * Launch: grid (ceil(width / 1024), vectors), block 256; a thread four values (a word of codes), eight threads a block
 * of 32 values.
 */
#include "kernel_registry.h"
#include "quantize_device.cuh"

extern "C" __global__ void __launch_bounds__(LINEAR_ELEMENT_THREADS)
    activation_quantize_entry(struct activation_quantize_arguments arguments, unsigned char *arena)
{
    activation_quantize_body(arguments, arena, blockIdx.x * LINEAR_ELEMENT_THREADS + threadIdx.x, blockIdx.y);
}
ANEMONE_KERNEL(KERNEL_FILE_ACTIVATION_QUANTIZE, activation_quantize_entry, activation_quantize_arguments);

/* The quantizer of WEIGHT_FORMAT_E4M3_BLOCK128's vectors (no counterpart in the reference): for each 128 consecutive
 * bfloat16 values, all in float32, scale = max(largest magnitude, 1e-4) / 448; each value is divided by the scale
 * (one rounding), limited to 448 and rounded to the nearest E4M3 number, a tie to the even code, the sign kept.
 * Written: codes [v][width] in the same lane order; the scales, float32 [v][width / 128], where the record names the
 * exponents (the same bytes a vector: width / 32); the operands are not written.
 * Launch: grid (ceil(width / 1024), vectors), block 256: a thread four values (a word of codes), 32 threads a scale. */
extern "C" __global__ void __launch_bounds__(LINEAR_ELEMENT_THREADS)
    activation_quantize_128_entry(struct activation_quantize_arguments arguments, unsigned char *arena)
{
    activation_quantize_128_body(arguments, arena, blockIdx.x * LINEAR_ELEMENT_THREADS + threadIdx.x, blockIdx.y);
}
ANEMONE_KERNEL(KERNEL_FILE_ACTIVATION_QUANTIZE, activation_quantize_128_entry, activation_quantize_arguments);
