/*
 * dense_device.cuh -- the dense product of a step's rows as device code (see kernel_dense_linear.hip for its definition),
 * shared by the dense_linear_* kernels and the fused site fronts.
 */
#ifndef DENSE_DEVICE_CUH
#define DENSE_DEVICE_CUH

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "exl3_device.cuh"

#include "publish_device.cuh"

#define DENSE_GROUP_LANES 32u
#define DENSE_GROUPS (DENSE_THREADS_VALUE / DENSE_GROUP_LANES)
#define DENSE_DIES 8u

/* the float32 nearest 1 / sqrt(operand): both steps are correctly rounded in double, whose 53 places decide a tie */
__device__ static __forceinline__ float dense_reciprocal_root(float operand)
{
    return (float)(1.0 / __dsqrt_rn((double)operand));
}

template <uint32_t distance, uint32_t ROWS, uint32_t OUTPUTS>
__device__ static __forceinline__ void dense_add_lanes(float (&chain)[OUTPUTS][ROWS], float (&squares)[ROWS], bool scaled, uint32_t live)
{
#pragma unroll
    for (uint32_t r = 0; r < ROWS; r++) {
        if (ROWS > 1u && r >= live) {
            break;
        }
#pragma unroll
        for (uint32_t o = 0; o < OUTPUTS; o++) {
            chain[o][r] = lanes_sum<distance>(chain[o][r]);
        }
        if (scaled) {
            squares[r] = lanes_sum<distance>(squares[r]);
        }
    }
}

/* what a block of DENSE_THREADS_VALUE threads keeps in LDS */
template <uint32_t ROWS, uint32_t OUTPUTS> struct dense_group_sums {
    float sums[DENSE_GROUPS][OUTPUTS + 1u][ROWS];
};

/* OUTPUTS outputs from first_output on by ROWS rows from first_row on, by the DENSE_THREADS_VALUE threads `thread` 0 ..
 * (every one of them calls, and the others of the block reach the same barrier: `active` false computes and stores
 * nothing that is read). `rows` names row 0 of the rows (memory or LDS). FRONT, of a launch of few blocks whose time is its
 * wavefronts' instructions: the places of the eight that hold no row are not computed, and the float32 outputs go through to
 * where every die sees them, for another block of the launch to read. */
template <uint32_t TYPE, uint32_t ROWS, uint32_t OUTPUTS, bool FRONT = false>
__device__ static __forceinline__ void dense_linear_body(const struct dense_linear_arguments &arguments, unsigned char *arena, const uint16_t *rows,
                                                         uint32_t first_output, uint32_t first_row, uint32_t thread, bool active,
                                                         dense_group_sums<ROWS, OUTPUTS> &lds)
{
    float (&group_sums)[DENSE_GROUPS][OUTPUTS + 1u][ROWS] = lds.sums;
    const uint32_t inputs = arguments.input_size, chunks = active ? inputs / DENSE_CHUNK_INPUTS : 0u;
    const bool scaled = (arguments.flags & DENSE_ROW_SCALE) != 0u;
    float chain[OUTPUTS][ROWS], squares[ROWS];
#pragma unroll
    for (uint32_t r = 0; r < ROWS; r++) {
        squares[r] = 0.0f;
#pragma unroll
        for (uint32_t o = 0; o < OUTPUTS; o++) {
            chain[o][r] = 0.0f;
        }
    }
    const uint32_t live = FRONT && arguments.row_count - first_row < ROWS ? arguments.row_count - first_row : ROWS;
    constexpr uint32_t WEIGHT_LOADS = TYPE == DENSE_FLOAT32 ? 2u : 1u;
    struct chunk_loads {
        uint4_t rows[ROWS], weights[OUTPUTS][WEIGHT_LOADS];
    };
    /* every row's chunk and every output's weights are asked for before any is used: a chunk costs one trip to memory, not one a row.
     * Asked for and added in two functions: written as one loop body, the front's row loop took 129 registers in place of 116
     * (ffn_front_8 at 5 rows 14.3 -> 15.95 us, at 8 of 5120 by 384 experts 19.3 -> 25.7) */
    const auto ask = [&](uint32_t chunk, chunk_loads &into) {
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) {
            /* a column from row_count on reads row 0 and is stored nowhere */
            const uint32_t row = first_row + r < arguments.row_count ? first_row + r : 0u;
            into.rows[r] = *(const uint4_t *)(rows + (uint64_t)row * inputs + chunk * DENSE_CHUNK_INPUTS);
        }
#pragma unroll
        for (uint32_t o = 0; o < OUTPUTS; o++) {
            const uint64_t at = (uint64_t)(first_output + o) * inputs + chunk * DENSE_CHUNK_INPUTS;
#pragma unroll
            for (uint32_t part = 0; part < WEIGHT_LOADS; part++) {
                into.weights[o][part] = *(const uint4_t *)(arena + arguments.weights_offset + (TYPE == DENSE_FLOAT32 ? 4u : 2u) * at + 16u * part);
            }
        }
    };
    const auto add = [&](const chunk_loads &now) {
        float weights[OUTPUTS][DENSE_CHUNK_INPUTS];
#pragma unroll
        for (uint32_t o = 0; o < OUTPUTS; o++) {
            if constexpr (TYPE == DENSE_FLOAT32) {
#pragma unroll
                for (uint32_t i = 0; i < DENSE_CHUNK_INPUTS; i++) {
                    weights[o][i] = __uint_as_float(now.weights[o][i / 4u][i % 4u]);
                }
            } else {
                unpack_bf16x8(now.weights[o][0], weights[o]);
            }
        }
        if constexpr (FRONT) { /* a row at a time, those that are one */
#pragma unroll
            for (uint32_t r = 0; r < ROWS; r++) {
                if (ROWS > 1u && r >= live) {
                    break;
                }
                float values[DENSE_CHUNK_INPUTS];
                unpack_bf16x8(now.rows[r], values);
#pragma unroll
                for (uint32_t i = 0; i < DENSE_CHUNK_INPUTS; i++) {
                    if (scaled) {
                        squares[r] = __fmaf_rn(values[i], values[i], squares[r]);
                    }
#pragma unroll
                    for (uint32_t o = 0; o < OUTPUTS; o++) {
                        chain[o][r] = __fmaf_rn(weights[o][i], values[i], chain[o][r]);
                    }
                }
            }
            return;
        }
        float values[ROWS][DENSE_CHUNK_INPUTS];
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) {
            unpack_bf16x8(now.rows[r], values[r]);
        }
        if (scaled) {
#pragma unroll
            for (uint32_t r = 0; r < ROWS; r++) {
#pragma unroll
                for (uint32_t i = 0; i < DENSE_CHUNK_INPUTS; i++) {
                    squares[r] = __fmaf_rn(values[r][i], values[r][i], squares[r]);
                }
            }
        }
#pragma unroll
        for (uint32_t o = 0; o < OUTPUTS; o++) {
#pragma unroll
            for (uint32_t r = 0; r < ROWS; r++) {
#pragma unroll
                for (uint32_t i = 0; i < DENSE_CHUNK_INPUTS; i++) {
                    chain[o][r] = __fmaf_rn(weights[o][i], values[r][i], chain[o][r]);
                }
            }
        }
    };
#pragma unroll(ROWS == 1u ? 4 : 1)
    for (uint32_t chunk = thread; chunk < chunks; chunk += DENSE_THREADS_VALUE) {
        chunk_loads now;
        ask(chunk, now);
        add(now);
    }
    const uint32_t group = thread / DENSE_GROUP_LANES, lane = thread % DENSE_GROUP_LANES;
    /* each chain's additions are the definition's: the distance halving from 16. By the lanes' own exchanges: a thread of 8 rows
     * has up to 72 sums of five distances each (2000 rows of 16384 inputs by 24 outputs, against shuffles: 57 -> 51.5 us) */
    dense_add_lanes<16u>(chain, squares, scaled, live);
    dense_add_lanes<8u>(chain, squares, scaled, live);
    dense_add_lanes<4u>(chain, squares, scaled, live);
    dense_add_lanes<2u>(chain, squares, scaled, live);
    dense_add_lanes<1u>(chain, squares, scaled, live);
    if (lane == 0u && active) {
#pragma unroll
        for (uint32_t r = 0; r < ROWS; r++) {
#pragma unroll
            for (uint32_t o = 0; o < OUTPUTS; o++) {
                group_sums[group][o][r] = chain[o][r];
            }
            if (scaled) {
                group_sums[group][OUTPUTS][r] = squares[r];
            }
        }
    }
    __syncthreads();
    const uint32_t o = thread / ROWS, r = thread % ROWS;
    if (!active || thread >= OUTPUTS * ROWS || first_row + r >= arguments.row_count) {
        return;
    }
    float sum = 0.0f, square_sum = 0.0f;
#pragma unroll
    for (uint32_t g = 0; g < DENSE_GROUPS; g++) {
        sum = __fadd_rn(sum, group_sums[g][o][r]);
        if (scaled) {
            square_sum = __fadd_rn(square_sum, group_sums[g][OUTPUTS][r]);
        }
    }
    if (scaled) {
        const float operand = __fadd_rn(__fmul_rn(square_sum, __fdiv_rn(1.0f, (float)inputs)), arguments.epsilon);
        sum = __fmul_rn(sum, dense_reciprocal_root(operand));
    }
    const uint64_t index = (uint64_t)(first_row + r) * arguments.output_size + first_output + o;
    if constexpr (FRONT) { /* a float32 that another block of this launch reads: through to where every die sees it */
        store_through((float *)(arena + arguments.output_offset) + index, __fmul_rn(sum, arguments.output_scale));
    } else if (arguments.output_type == DENSE_FLOAT32) {
        ((float *)(arena + arguments.output_offset))[index] = __fmul_rn(sum, arguments.output_scale);
    } else {
        ((uint16_t *)(arena + arguments.output_offset))[index] = float_to_bf16(__fmul_rn(bf16_to_float(float_to_bf16(sum)), arguments.output_scale));
    }
}

#endif
