/*
 * exl3_device.cuh -- device code shared by the EXL3 kernels of gfx950, and by the others for its conversions: the mul1
 * codebook in registers, the 128-point Hadamard transform of one wavefront and of a row of sixteen lanes, and the
 * deterministic exponential. The product routines, which say which lane decodes what, are exl3_stream_device.cuh's.
 *
 * Definitions followed (reference tree): codebook source/kernel_exl3.cu:58-65; transform order
 * source/kernel_exl3.cu:104-124.
 */
#ifndef EXL3_DEVICE_CUH
#define EXL3_DEVICE_CUH

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "anemone_records.h"

typedef _Float16 half_t;
typedef half_t half2_t __attribute__((ext_vector_type(2)));
typedef half_t half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));

#define WAVE 64u

__device__ static __forceinline__ float bf16_to_float(uint16_t bits)
{
    return __uint_as_float((uint32_t)bits << 16);
}

/* float32 -> bfloat16, to nearest, ties to even; a NaN becomes 0x7FC0. The card's own conversion
 * (v_cvt_pk_bf16_f32) gives, for every float32 that is a number, the bits of (bits + 0x7FFF + ((bits >> 16) & 1)) >> 16
 * (compared over all 2^32 inputs); it keeps a NaN's payload, hence the select. */
__device__ static __forceinline__ uint16_t float_to_bf16(float value)
{
    const uint16_t rounded = __builtin_bit_cast(uint16_t, (__bf16)value);
    return value != value ? (uint16_t)0x7FC0u : rounded;
}

__device__ static __forceinline__ float half_bits_to_float(uint16_t bits)
{
    return (float)__builtin_bit_cast(half_t, bits);
}

/* float32 -> fp16, to nearest even, of a value that already IS a float32: the empty asm keeps the compiler from
 * folding the multiplication that produced it into one mixed-precision instruction (v_fma_mixlo_f16), which would
 * round once where the contract rounds twice (to float32, then to fp16). */
__device__ static __forceinline__ uint16_t float_to_half_bits(float value)
{
    asm volatile("" : "+v"(value));
    return __builtin_bit_cast(uint16_t, (half_t)value); /* v_cvt_f16_f32 */
}

/* two of them in one register, the first in its low half */
__device__ static __forceinline__ uint32_t floats_to_half_bits(float low, float high)
{
    typedef float float_pair __attribute__((ext_vector_type(2)));
    asm volatile("" : "+v"(low), "+v"(high));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float_pair){low, high}, half2_t)); /* v_cvt_pk_f16_f32 */
}

/* e^x by a fixed sequence of float32 operations: k = nearest(x log2 e), r = x - k ln 2 in two pieces, a degree-6
 * polynomial in fma form, scaling by ldexp. Written without contraction so that host and card agree bit for bit.
 * det_exp_sequence is the sequence alone, for an x it is defined for (-104 <= x <= 88.8 in det_expf). */
__device__ static __forceinline__ float det_exp_sequence(float x)
{
    const float k = __builtin_rintf(__fmul_rn(x, 1.44269502162933349609375f));
    float r = __fmaf_rn(k, -0.693145751953125f, x);
    r = __fmaf_rn(k, -1.42860676533018704503775e-06f, r);
    float p = 1.9875691500e-4f;
    p = __fmaf_rn(p, r, 1.3981999507e-3f);
    p = __fmaf_rn(p, r, 8.3334519073e-3f);
    p = __fmaf_rn(p, r, 4.1665795894e-2f);
    p = __fmaf_rn(p, r, 1.6666665459e-1f);
    p = __fmaf_rn(p, r, 5.0000001201e-1f);
    const float r2 = __fmul_rn(r, r);
    float y = __fmaf_rn(p, r2, r);
    y = __fadd_rn(y, 1.0f);
    return ldexpf(y, (int)k);
}

__device__ static __forceinline__ float det_expf(float x)
{
    if (x != x) {
        return x;
    }
    if (x > 88.8f) {
        return __builtin_huge_valf();
    }
    if (x < -104.0f) {
        return 0.0f;
    }
    return det_exp_sequence(x);
}

/* value / (1 + e^x), rounded once, for a sum of 1 and an exponential: the sum is 1 or above, so all that has to be scaled is
 * the reciprocal (the card's would flush those of sums above 2^126), by a constant; a general division brings both sides into
 * range and takes them out again, and corrects the quotient once more. The reciprocal is corrected once, the quotient once by
 * its exact remainder; infinities and not-a-numbers are the last instruction's. Nine instructions in place of eleven, three of
 * which wait for a comparison's register. The bits of the division: the arithmetic_selfcheck kernel, over all float32 of both callers. */
__device__ static __forceinline__ float quotient_above_one(float value, float sum)
{
    const float quarter = __fmul_rn(sum, 0.25f);
    float reciprocal = __builtin_amdgcn_rcpf(quarter);
    reciprocal = __fmul_rn(__fmaf_rn(__fmaf_rn(-quarter, reciprocal, 1.0f), reciprocal, reciprocal), 0.25f);
    const float near = __fmul_rn(value, reciprocal);
    return __builtin_amdgcn_div_fixupf(__fmaf_rn(__fmaf_rn(-sum, near, value), reciprocal, near), sum, value);
}

/* gate / (1 + e^(-gate)): the bits of __fdiv_rn(gate, __fadd_rn(1.0f, det_expf(-gate))) for every float32 gate (a NaN
 * for a NaN), without det_expf's three tests, each of which is a branch of its own and a wait for its comparison in a
 * kernel's epilogue. The sequence's argument is held inside [-104, 89.5] instead: above 88.8 the sequence overflows to
 * infinity by itself (k >= 128 and, where k = 128, r > 0.08, so the polynomial is above 1); below -104 det_expf gives 0
 * and the sequence at -104 something below 2^-148, and 1 plus either is 1; a NaN gate divides to a NaN whatever the
 * denominator. The library's arithmetic_selfcheck kernel compares the two over all 2^32 gates. */
__device__ static __forceinline__ float det_silu(float gate)
{
    const float x = __builtin_amdgcn_fmed3f(-gate, -104.0f, 89.5f);
    return quotient_above_one(gate, __fadd_rn(1.0f, det_exp_sequence(x)));
}

/* A lane's value and that of the lane `distance` away (lane ^ distance), in some order: for operations whose two sides may
 * change places. By the lanes' own exchanges: a shuffle is an LDS round trip of some 120 cycles, and the sums and maxima of a
 * small launch are a chain of them. Every lane of a row of sixteen (of two rows for distance 16) calls. */
struct lane_pair {
    float first, second;
};

template <uint32_t distance>
__device__ static __forceinline__ lane_pair lanes_apart(float value)
{
    const int bits = (int)__float_as_uint(value);
    if constexpr (distance == 16u) { /* two rows change places */
        const auto rows = __builtin_amdgcn_permlane16_swap((uint32_t)bits, (uint32_t)bits, false, false);
        return {__uint_as_float(rows[0]), __uint_as_float(rows[1])};
    } else if constexpr (distance == 4u) { /* four lanes on, or four back: banks of four lanes in turn */
        const int on = __builtin_amdgcn_update_dpp(bits, bits, 0x104, 0xF, 0x5, false); /* row_shl:4 */
        return {value, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(on, bits, 0x114, 0xF, 0xA, false))}; /* row_shr:4 */
    } else {
        static_assert(distance == 8u || distance == 2u || distance == 1u, "a distance inside a group of 32 lanes");
        constexpr int control = distance == 8u ? 0x128 : distance == 2u ? 0x4E : 0xB1; /* row_ror:8, quad_perm:[2,3,0,1], [1,0,3,2] */
        return {value, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(bits, bits, control, 0xF, 0xF, false))};
    }
}

template <uint32_t distance>
__device__ static __forceinline__ float lanes_sum(float value)
{
    const lane_pair pair = lanes_apart<distance>(value);
    return __fadd_rn(pair.first, pair.second);
}

template <uint32_t distance>
__device__ static __forceinline__ float lanes_largest(float value)
{
    const lane_pair pair = lanes_apart<distance>(value);
    return fmaxf(pair.first, pair.second);
}

/* The 128-point transform: seven stages, the distance doubling from 1; a pair (lower, upper) becomes (lower + upper, lower -
 * upper), each rounded once. No normalisation here. Two lay-outs: a block across a wavefront, two values a lane
 * (wave_hadamard128: the fewest instructions for one block), and across a row of sixteen lanes, eight consecutive values a
 * lane (row_hadamard128: the fewest for many).
 *
 * Lanes meet by the data-parallel primitives of a vector instruction, without LDS. Inside a row those reach lane ^ 1 and ^ 2 (a
 * permutation of four lanes), ^ 7 (the mirror of eight) and ^ 8 (a rotation by eight of sixteen) in one step, so lane L of a
 * row stands for place r = row_group_of(L), whose four bits are then the four pairings. A pair's sum and difference are one
 * fused multiply-add each, own + s x other, with s = +1 in the lower lane and -1 in the upper, which is left with upper - lower,
 * the difference's exact negative; two lanes that meet in a later pairing carry the same sign, so every value ends as its own or
 * its exact negative, by the parity of r, and row_normalized takes the sign out with the factor it multiplies by (a zero becomes
 * +0 there). Rows meet by v_permlane16_swap and v_permlane32_swap of a lane's two values. */
__device__ static __forceinline__ uint32_t row_group_of(uint32_t lane)
{
    return (lane % 16u) ^ ((lane & 4u) != 0u ? 3u : 0u);
}

__device__ static __forceinline__ void row_signs(uint32_t lane, float (&signs)[4])
{
#pragma unroll
    for (uint32_t bit = 0; bit < 4u; bit++) {
        signs[bit] = ((row_group_of(lane) >> bit) & 1u) == 0u ? 1.0f : -1.0f;
    }
}

/* EXL3_NORMALIZATION with the sign that row_hadamard128 leaves the lane's values with */
__device__ static __forceinline__ float row_normalization(uint32_t lane)
{
    return (__builtin_popcount(row_group_of(lane)) & 1) == 0 ? EXL3_NORMALIZATION : -EXL3_NORMALIZATION;
}

/* value x EXL3_NORMALIZATION of a value of row_hadamard128, rounded once; a zero becomes +0 */
__device__ static __forceinline__ float row_normalized(float value, float normalization)
{
    return __fmaf_rn(value, normalization, 0.0f);
}

/* A block across a wavefront: lane l begins with the values wave_channel<SWAPPED>(l) (v0) and 64 on (v1) and ends with those of
 * wave_channel<!SWAPPED>(l): the exchanges of the rows leave the two upper bits of a lane's number the other way round. */
template <bool SWAPPED>
__device__ static __forceinline__ uint32_t wave_channel(uint32_t lane)
{
    const uint32_t row = lane / 16u % 2u, half = lane / 32u;
    return row_group_of(lane) + 16u * (SWAPPED ? half : row) + 32u * (SWAPPED ? row : half);
}

/* Seventeen instructions and their waits: 14 exchanges through LDS, each waited for, and 14 additions before. A launch of one
 * row a block of channels is its wavefront's instructions: exl3_tc_activate 6.8 -> 5.6 us (8 rows of 4096 x 2048, 8 picks), 13.1 ->
 * 11.8 (37 rows), exl3_tc_operands 9.5 -> 8.5 (37 rows); a lane-row form of these launches (eight values a lane) was slower at
 * one row a job, where eight hidden steps stand one behind the other. */
template <bool SWAPPED>
__device__ static __forceinline__ void wave_hadamard128(float &v0, float &v1, uint32_t lane)
{
    float signs[4];
    row_signs(lane, signs);
    /* written as assembly: the compiler does not fold a lane's move into a multiply-add. Two instructions or waits stand between
     * a vector write and a lane's read of it, ahead of the first stage and behind the last as well */
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %0, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\ts_nop 0\n\t"
        "v_fmac_f32_dpp %0, %0, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\ts_nop 0\n\t"
        "v_fmac_f32_dpp %0, %0, %4 row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %4 row_half_mirror row_mask:0xf bank_mask:0xf\n\ts_nop 0\n\t"
        "v_fmac_f32_dpp %0, %0, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %1, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\ts_nop 1"
        : "+v"(v0), "+v"(v1)
        : "v"(signs[0]), "v"(signs[1]), "v"(signs[2]), "v"(signs[3]));
    /* rows: a lane's two values become the two of one pair; what told them apart moves into the lane's number */
    const auto pair_rows = [&](bool halves) {
        const auto swapped = halves ? __builtin_amdgcn_permlane32_swap(__float_as_uint(v0), __float_as_uint(v1), false, false)
                                    : __builtin_amdgcn_permlane16_swap(__float_as_uint(v0), __float_as_uint(v1), false, false);
        const float lower = __uint_as_float(swapped[0]), upper = __uint_as_float(swapped[1]);
        v0 = __fadd_rn(lower, upper);
        v1 = __fsub_rn(lower, upper);
    };
    pair_rows(SWAPPED);  /* 16 */
    pair_rows(!SWAPPED); /* 32 */
    pair_rows(SWAPPED);  /* 64 */
}

/* A block across sixteen lanes: lane L of the row holds the values 8 r .. 8 r + 7 of r = row_group_of(L); distances 1, 2, 4 stay
 * inside the lane. Seven instructions a value where the lanes' part alone was ten (a sign, moves and an addition a pairing): 32768
 * pairs of 4096 x 2048: exl3_tcp_operands 148 -> 124 us, exl3_tcp_activate 184 -> 163. A row's sixteen lanes are all active or
 * all idle. */
__device__ static __forceinline__ void row_hadamard128(float (&v)[8], uint32_t lane)
{
#pragma unroll
    for (uint32_t distance = 1; distance < 8u; distance *= 2u) {
#pragma unroll
        for (uint32_t i = 0; i < 8u; i++) {
            if ((i & distance) == 0u) {
                const float lower = v[i], upper = v[i + distance];
                v[i] = __fadd_rn(lower, upper);
                v[i + distance] = __fsub_rn(lower, upper);
            }
        }
    }
    float signs[4];
    row_signs(lane, signs);
    /* as in wave_hadamard128; a value's next instruction is eight behind its last */
#define ROW_STAGE(control, sign)                                                                                           \
    "v_fmac_f32_dpp %0, %0, %" sign " " control "\n\tv_fmac_f32_dpp %1, %1, %" sign " " control "\n\t"                     \
    "v_fmac_f32_dpp %2, %2, %" sign " " control "\n\tv_fmac_f32_dpp %3, %3, %" sign " " control "\n\t"                     \
    "v_fmac_f32_dpp %4, %4, %" sign " " control "\n\tv_fmac_f32_dpp %5, %5, %" sign " " control "\n\t"                     \
    "v_fmac_f32_dpp %6, %6, %" sign " " control "\n\tv_fmac_f32_dpp %7, %7, %" sign " " control "\n\t"
    asm("s_nop 1\n\t" ROW_STAGE("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", "8") ROW_STAGE("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf", "9")
            ROW_STAGE("row_half_mirror row_mask:0xf bank_mask:0xf", "10") ROW_STAGE("row_ror:8 row_mask:0xf bank_mask:0xf", "11")
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])
        : "v"(signs[0]), "v"(signs[1]), "v"(signs[2]), "v"(signs[3]));
#undef ROW_STAGE
}

/* eight bfloat16 or fp16 values of a 16-byte load as float32; eight float32 as fp16, one rounding each */
__device__ static __forceinline__ void unpack_bf16x8(uint4_t load, float (&values)[8])
{
#pragma unroll
    for (uint32_t i = 0; i < 8u; i++) {
        values[i] = __uint_as_float(i % 2u == 0u ? load[i / 2u] << 16 : load[i / 2u] & 0xFFFF0000u);
    }
}

__device__ static __forceinline__ void unpack_half8(uint4_t load, float (&values)[8])
{
#pragma unroll
    for (uint32_t i = 0; i < 8u; i++) {
        values[i] = half_bits_to_float((uint16_t)(i % 2u == 0u ? load[i / 2u] & 0xFFFFu : load[i / 2u] >> 16));
    }
}

__device__ static __forceinline__ uint4_t pack_half8(const float (&values)[8])
{
    uint4_t packed;
#pragma unroll
    for (uint32_t word = 0; word < 4u; word++) {
        packed[word] = floats_to_half_bits(values[2u * word], values[2u * word + 1u]);
    }
    return packed;
}

/* eight values of a row (row_hadamard128's lanes) as an operand of one matrix: fp16(H128(x suh) / sqrt(128)) */
__device__ static __forceinline__ uint4_t row_operand(uint4_t load, const float (&scale)[8], uint32_t lane)
{
    float v[8];
    unpack_bf16x8(load, v);
#pragma unroll
    for (uint32_t j = 0; j < 8u; j++) {
        v[j] = __fmul_rn(v[j], scale[j]);
    }
    row_hadamard128(v, lane);
    const float normalization = row_normalization(lane);
#pragma unroll
    for (uint32_t j = 0; j < 8u; j++) {
        v[j] = row_normalized(v[j], normalization);
    }
    return pack_half8(v);
}

/* eight gate and eight up products (g, u) as a down operand: gate = H128(gate products) / sqrt(128) x svh, up the same, the
 * SwiGLU with its limit, x the down matrix's suh, H128, fp16. Bound by its instructions and by memory alike (some 460 for eight
 * values of 64 lanes, of which the three transforms 196): the limits by a branch of the whole card in place of a select a value, the
 * median for the lower and upper one, quotient_above_one and two values a conversion took 32768 pairs of 2048 from 160.4 to 153.9 us
 * (4.4 TB/s), 1624 pairs from 10.4 to 9.7. */
__device__ static __forceinline__ uint4_t row_activated(float (&g)[8], float (&u)[8], const float (&gs)[8], const float (&us)[8],
                                                        const float (&ds)[8], float limit, uint32_t lane)
{
    float v[8];
    row_hadamard128(g, lane);
    row_hadamard128(u, lane);
    const float normalization = row_normalization(lane);
    const auto scaled = [&](bool limited) {
#pragma unroll
        for (uint32_t j = 0; j < 8u; j++) {
            const float gate = __fmul_rn(__fmul_rn(g[j], normalization), gs[j]);
            const float up = __fmul_rn(__fmul_rn(u[j], normalization), us[j]);
            g[j] = limited ? fminf(gate, limit) : gate;
            /* the lower limit for a value that is not a number, as fminf(fmaxf(up, -limit), limit) */
            u[j] = limited ? __builtin_amdgcn_fmed3f(up, -limit, limit) : up;
        }
    };
    if (limit > 0.0f) { /* the same in every lane */
        scaled(true);
    } else {
        scaled(false);
    }
#pragma unroll
    for (uint32_t j = 0; j < 8u; j++) {
        v[j] = __fmul_rn(__fmul_rn(det_silu(g[j]), u[j]), ds[j]);
    }
    row_hadamard128(v, lane);
#pragma unroll
    for (uint32_t j = 0; j < 8u; j++) {
        v[j] = row_normalized(v[j], normalization);
    }
    return pack_half8(v);
}

/* mul1: two 16-bit states -> two fp16 weights in one register (low half: first) */
__device__ static __forceinline__ uint32_t exl3_decode_pair(uint32_t state_low, uint32_t state_high)
{
    const uint32_t product_low = state_low * EXL3_MUL1_MULTIPLIER;
    const uint32_t product_high = state_high * EXL3_MUL1_MULTIPLIER;
    /* byte sums with the codebook's base folded in as the accumulator: 0x6400 + b is the fp16 1024 + b. The first
     * sum lands in the low half on top of 0x64006400, the second is added into the high half. */
    const uint32_t low = __builtin_amdgcn_sad_u8(product_low, 0u, (uint32_t)EXL3_MUL1_BASE * 0x10001u);
    const uint32_t packed = __builtin_amdgcn_sad_hi_u8(product_high, 0u, low);
    const half2_t value = __builtin_bit_cast(half2_t, packed);
    const half2_t scale = __builtin_bit_cast(half2_t, (uint32_t)EXL3_MUL1_SCALE * 0x10001u);
    const half2_t bias = __builtin_bit_cast(half2_t, (uint32_t)EXL3_MUL1_BIAS * 0x10001u);
    const half2_t weight = __builtin_elementwise_fma(value, scale, bias); /* v_pk_fma_f16: one rounding each */
    return __builtin_bit_cast(uint32_t, weight);
}

__device__ static __forceinline__ uint16_t exl3_decode_one(uint32_t state)
{
    return (uint16_t)exl3_decode_pair(state & 0xFFFFu, 0u);
}

#endif
