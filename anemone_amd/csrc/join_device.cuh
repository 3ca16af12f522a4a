/*
 * join_device.cuh -- the join of the FFN site for eight (four, two) consecutive values of one row, which the post, the join
 * (kernel_hyper_connection.hip) and the shared join (kernel_trunk_linear.hip) share. The arithmetic of the reference's
 * source/kernel_hyper_connection.cuh:42-85 and source/kernel_expert_join.cuh:35-57, value by value, in their order:
 * every product and sum rounded on its own.
 */
#ifndef JOIN_DEVICE_CUH
#define JOIN_DEVICE_CUH

#include "exl3_device.cuh" /* bf16 helpers, vector types */

#include "anemone_records.h"

/* VALUES bfloat16 values as they lie: 16, 8 or 4 bytes */
template <uint32_t VALUES> struct join_load_of {
    static_assert(VALUES == 8u || VALUES == 4u || VALUES == 2u, "one vector load");
    typedef uint32_t type __attribute__((ext_vector_type(VALUES / 2u)));
};
template <> struct join_load_of<2u> {
    typedef uint32_t type;
};
template <uint32_t VALUES> using join_load = typename join_load_of<VALUES>::type;

/* the values of a load as float32, and float32 values rounded to bfloat16 as one */
template <uint32_t VALUES>
__device__ static __forceinline__ void join_unpack(join_load<VALUES> load, float (&values)[VALUES])
{
    const struct { uint32_t of[VALUES / 2u]; } words = __builtin_bit_cast(decltype(words), load);
#pragma unroll
    for (uint32_t v = 0; v < VALUES; v++) {
        values[v] = __uint_as_float(v % 2u == 0u ? words.of[v / 2u] << 16 : words.of[v / 2u] & 0xFFFF0000u);
    }
}

template <uint32_t VALUES>
__device__ static __forceinline__ join_load<VALUES> join_pack(const float (&values)[VALUES])
{
    struct { uint32_t of[VALUES / 2u]; } words;
#pragma unroll
    for (uint32_t word = 0; word < VALUES / 2u; word++) {
        words.of[word] = (uint32_t)float_to_bf16(values[2u * word]) | ((uint32_t)float_to_bf16(values[2u * word + 1u]) << 16);
    }
    return __builtin_bit_cast(join_load<VALUES>, words);
}

#define JOIN_SLOTS_IN_FLIGHT 8u

/* What a thread's join reads: its load of every stream, the row's post and comb ([source][target]), and its loads of the
 * first JOIN_SLOTS_IN_FLIGHT pair outputs (a slot past the last repeats the last): one trip to memory for all of them */
template <uint32_t VALUES> struct join_streams {
    join_load<VALUES> of[MODEL_STREAMS];
    float4_t post, comb[MODEL_STREAMS];
};

template <uint32_t VALUES> struct join_slots {
    join_load<VALUES> of[JOIN_SLOTS_IN_FLIGHT];
};

template <uint32_t VALUES>
__device__ static __forceinline__ join_streams<VALUES> join_read_streams(const float *post, const float *comb, const join_load<VALUES> *streams, uint64_t stride)
{
    join_streams<VALUES> read;
#pragma unroll
    for (uint32_t stream = 0; stream < MODEL_STREAMS; stream++) {
        read.of[stream] = streams[stream * stride];
        read.comb[stream] = ((const float4_t *)comb)[stream];
    }
    read.post = *(const float4_t *)post;
    return read;
}

template <uint32_t VALUES>
__device__ static __forceinline__ join_slots<VALUES> join_read_slots(const join_load<VALUES> *pairs, uint32_t pairs_per_row, uint64_t stride)
{
    join_slots<VALUES> read;
#pragma unroll
    for (uint32_t slot = 0; slot < JOIN_SLOTS_IN_FLIGHT; slot++) {
        read.of[slot] = pairs[(uint64_t)(slot < pairs_per_row ? slot : pairs_per_row - 1u) * stride];
    }
    return read;
}

/* The post of a thread's values of a row: output y as the post takes it (with the combine, the routed sums added
 * and rounded); streams the thread's load of stream 0, the streams `stride` loads apart, written in place. */
template <uint32_t VALUES>
__device__ static __forceinline__ void join_write_streams(const float (&output)[VALUES], const join_streams<VALUES> &read, join_load<VALUES> *streams,
                                                          uint64_t stride)
{
    float values[MODEL_STREAMS][VALUES];
#pragma unroll
    for (uint32_t stream = 0; stream < MODEL_STREAMS; stream++) {
        join_unpack<VALUES>(read.of[stream], values[stream]);
    }
#pragma unroll
    for (uint32_t target = 0; target < MODEL_STREAMS; target++) {
        float mixed[VALUES];
#pragma unroll
        for (uint32_t v = 0; v < VALUES; v++) {
            float sum = 0.0f;
#pragma unroll
            for (uint32_t source = 0; source < MODEL_STREAMS; source++) {
                sum = __fadd_rn(sum, __fmul_rn(read.comb[source][target], values[source][v]));
            }
            mixed[v] = __fadd_rn(__fmul_rn(read.post[target], output[v]), sum);
        }
        streams[target * stride] = join_pack<VALUES>(mixed);
    }
}

/* The join of a thread's values of a row: pairs its load of the row's first pair output, a slot `stride` loads on, slots the
 * first of them; shared_output the shared expert's output there; row_sums where their float32 sums go, or nullptr. The
 * additions go in slot order. */
template <uint32_t VALUES>
__device__ static __forceinline__ void join_values(const join_load<VALUES> *pairs, uint32_t pairs_per_row, const join_slots<VALUES> &slots,
                                                   const float (&shared_output)[VALUES], const join_streams<VALUES> &read, join_load<VALUES> *streams,
                                                   float *row_sums, uint64_t stride)
{
    float routed[VALUES], output[VALUES];
#pragma unroll
    for (uint32_t v = 0; v < VALUES; v++) {
        routed[v] = 0.0f;
    }
    const auto add = [&](join_load<VALUES> load) {
        float pair[VALUES];
        join_unpack<VALUES>(load, pair);
#pragma unroll
        for (uint32_t v = 0; v < VALUES; v++) {
            routed[v] = __fadd_rn(routed[v], pair[v]);
        }
    };
    const auto add_some = [&](const join_slots<VALUES> &some, uint32_t count) {
#pragma unroll
        for (uint32_t slot = 0; slot < JOIN_SLOTS_IN_FLIGHT; slot++) {
            if (slot < count) {
                add(some.of[slot]);
            }
        }
    };
    if (pairs_per_row >= JOIN_SLOTS_IN_FLIGHT) {
        add_some(slots, JOIN_SLOTS_IN_FLIGHT);
    } else {
        add_some(slots, pairs_per_row);
    }
    /* more slots: as many together again, so that eight cost one trip to memory. us, a slot at a time | so: expert_join of 8 rows of
     * 4096, 16 slots 4.45 | 3.5, 64 slots 11.05 | 5.65; expert_shared_join_4 of them 5.35 | 4.7 and 10.1 | 5.9; expert_join of 2048 rows, 16
     * slots 75 | 71.4, 24 slots 105 | 113 */
    uint32_t first = JOIN_SLOTS_IN_FLIGHT;
    for (; first + JOIN_SLOTS_IN_FLIGHT <= pairs_per_row; first += JOIN_SLOTS_IN_FLIGHT) {
        add_some(join_read_slots<VALUES>(pairs + first * stride, JOIN_SLOTS_IN_FLIGHT, stride), JOIN_SLOTS_IN_FLIGHT);
    }
    if (first < pairs_per_row) {
        add_some(join_read_slots<VALUES>(pairs + first * stride, pairs_per_row - first, stride), pairs_per_row - first);
    }
    if (row_sums != nullptr) {
        typedef float sums_of __attribute__((ext_vector_type(VALUES < 4u ? VALUES : 4u)));
#pragma unroll
        for (uint32_t v = 0; v < VALUES; v += VALUES < 4u ? VALUES : 4u) {
            sums_of sums;
#pragma unroll
            for (uint32_t k = 0; k < (VALUES < 4u ? VALUES : 4u); k++) {
                sums[k] = routed[v + k];
            }
            *(sums_of *)(row_sums + v) = sums;
        }
    }
#pragma unroll
    for (uint32_t v = 0; v < VALUES; v++) {
        output[v] = bf16_to_float(float_to_bf16(__fadd_rn(routed[v], shared_output[v])));
    }
    join_write_streams<VALUES>(output, read, streams, stride);
}

#endif
