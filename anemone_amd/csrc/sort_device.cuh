/*
 * sort_device.cuh -- what the sorts of pairs by expert share (the router's wide select and the prefill form of the
 * EXL3 experts): a block's picked experts into LDS, its picks counted an expert, every pick's place, and a block-wide
 * exclusive prefix sum. The only atomic operations are integer additions in LDS that count (the same sums in any order);
 * a pick's place among its expert's is formed from the lanes' ballots, in row order.
 */
#ifndef SORT_DEVICE_CUH
#define SORT_DEVICE_CUH

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "anemone_records.h"

#define SORT_WAVE 64u
#define SORT_MOST_WAVES 8u /* of a block of the sorts: 512 threads */

/* the picked experts of the live rows of block `block` of ROUTER_SORT_ROWS rows, into LDS; returns their number */
__device__ static __forceinline__ uint32_t sort_block_picks(const struct router_pick *all_picks, uint32_t picks_per_row,
                                                            uint32_t block, uint32_t live_rows, uint32_t *experts_out)
{
    const uint32_t first_row = block * ROUTER_SORT_ROWS;
    const uint32_t rows = live_rows <= first_row ? 0u : live_rows - first_row < ROUTER_SORT_ROWS ? live_rows - first_row : ROUTER_SORT_ROWS;
    const struct router_pick *picks = all_picks + (uint64_t)first_row * picks_per_row;
    for (uint32_t index = threadIdx.x; index < rows * picks_per_row; index += SORT_MOST_WAVES * SORT_WAVE) {
        experts_out[index] = picks[index].expert;
    }
    return rows * picks_per_row;
}

/* The block's picks of every expert: histogram[expert] in LDS. Integer additions in LDS: the same sums whatever their
 * order. The whole block calls it (barriers inside); block_experts is complete before the call. */
__device__ static __forceinline__ void sort_count_picks(const uint32_t *block_experts, uint32_t pairs, uint32_t experts, uint32_t *histogram)
{
    for (uint32_t expert = threadIdx.x; expert < experts; expert += SORT_MOST_WAVES * SORT_WAVE) {
        histogram[expert] = 0u;
    }
    __syncthreads();
    for (uint32_t index = threadIdx.x; index < pairs; index += SORT_MOST_WAVES * SORT_WAVE) {
        __hip_atomic_fetch_add(&histogram[block_experts[index]], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
}

/* The lanes of the wavefront that hold the same word as this lane, among the lanes where `live` (a lane that is not live
 * gets 0): one ballot a bit of the words, `bits` of them. */
__device__ static __forceinline__ uint64_t sort_equal_lanes(uint32_t word, bool live, uint32_t bits)
{
    uint64_t equal = __builtin_amdgcn_ballot_w64(live);
    for (uint32_t bit = 0; bit < bits; bit++) {
        const bool set = ((word >> bit) & 1u) != 0u;
        const uint64_t holders = __builtin_amdgcn_ballot_w64(live && set);
        equal &= set ? holders : ~holders;
    }
    return live ? equal : 0ull;
}

/* Wavefront `wave` of a block's SORT_MOST_WAVES takes the picks [begin, end) of `pairs`: whole groups of 64 in order */
__device__ static __forceinline__ void sort_share(uint32_t pairs, uint32_t wave, uint32_t &begin, uint32_t &end)
{
    const uint32_t share = ((pairs + SORT_MOST_WAVES - 1u) / SORT_MOST_WAVES + SORT_WAVE - 1u) / SORT_WAVE * SORT_WAVE;
    begin = wave * share < pairs ? wave * share : pairs;
    end = begin + share < pairs ? begin + share : pairs;
}

/* A wavefront's picks [begin, end) counted an expert into its own cursors (LDS, zero before: integer additions) */
__device__ static __forceinline__ void sort_count_share(const uint32_t *block_experts, uint32_t begin, uint32_t end, uint32_t *mine)
{
    for (uint32_t index = begin + threadIdx.x % SORT_WAVE; index < end; index += SORT_WAVE) {
        __hip_atomic_fetch_add(&mine[block_experts[index]], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

/* The wavefronts' counts of one expert (cursors[wavefront][experts]); and where each wavefront's picks of it begin, behind
 * `place` and the wavefronts before it, in their place. The reads go together: one LDS round trip, not one a wavefront. */
__device__ static __forceinline__ uint32_t sort_counts_of(const uint32_t *cursors, uint32_t experts, uint32_t expert, uint32_t (&counts)[SORT_MOST_WAVES])
{
    uint32_t total = 0;
#pragma unroll
    for (uint32_t wave = 0; wave < SORT_MOST_WAVES; wave++) {
        counts[wave] = cursors[wave * experts + expert];
    }
#pragma unroll
    for (uint32_t wave = 0; wave < SORT_MOST_WAVES; wave++) {
        total += counts[wave];
    }
    return total;
}

__device__ static __forceinline__ void sort_cursors_of(uint32_t *cursors, uint32_t experts, uint32_t expert, const uint32_t (&counts)[SORT_MOST_WAVES],
                                                       uint32_t place)
{
#pragma unroll
    for (uint32_t wave = 0; wave < SORT_MOST_WAVES; wave++) {
        cursors[wave * experts + expert] = place;
        place += counts[wave];
    }
}

/* A wavefront's picks [begin, end), 64 at a time: a pick's place is its expert's cursor plus the lanes below it that hold
 * the same expert (ballots over the expert's bits: no lane waits for another's answer), and the first of them moves the
 * cursor on. placed(index, place) for every pick. */
template <typename PLACED>
__device__ static __forceinline__ void sort_place_share(const uint32_t *block_experts, uint32_t begin, uint32_t end, uint32_t experts, uint32_t *mine,
                                                        PLACED placed)
{
    uint32_t bits = 0;
    while ((1u << bits) < experts) {
        bits++;
    }
    for (uint32_t base = begin; base < end; base += SORT_WAVE) {
        const uint32_t index = base + threadIdx.x % SORT_WAVE;
        const bool live = index < end;
        const uint32_t expert = live ? block_experts[index] : 0u;
        const uint64_t equal = sort_equal_lanes(expert, live, bits);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(equal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)equal, 0u));
        if (live) {
            const uint32_t cursor = mine[expert]; /* every lane of an expert reads it before the first of them writes it: LDS serves
                                                    a wavefront's instructions in their order */
            placed(index, cursor + below);
            if (below == 0u) {
                mine[expert] = cursor + (uint32_t)__builtin_popcountll(equal);
            }
        }
    }
}

/* Every pick's place, in LDS: place_of[index] = first[expert] + the picks of the same expert before it in the block. A
 * wavefront takes a share of the picks (sort_share, sort_place_share), its cursors begun behind the picks of the
 * wavefronts before it, which a histogram a wavefront and a thread an expert give. first: LDS, experts words (kept);
 * cursors: LDS, SORT_MOST_WAVES x experts words. The whole block of SORT_MOST_WAVES wavefronts calls it (barriers inside). */
__device__ static __forceinline__ void sort_place_picks(const uint32_t *block_experts, uint32_t pairs, uint32_t experts, const uint32_t *first,
                                                        uint32_t *cursors, uint32_t *place_of)
{
    const uint32_t wave = threadIdx.x / SORT_WAVE;
    uint32_t begin, end;
    sort_share(pairs, wave, begin, end);
    for (uint32_t at = threadIdx.x; at < SORT_MOST_WAVES * experts; at += SORT_MOST_WAVES * SORT_WAVE) {
        cursors[at] = 0u;
    }
    __syncthreads();
    sort_count_share(block_experts, begin, end, cursors + wave * experts);
    __syncthreads();
    for (uint32_t expert = threadIdx.x; expert < experts; expert += SORT_MOST_WAVES * SORT_WAVE) {
        uint32_t counts[SORT_MOST_WAVES];
        (void)sort_counts_of(cursors, experts, expert, counts);
        sort_cursors_of(cursors, experts, expert, counts, first[expert]);
    }
    __syncthreads();
    sort_place_share(block_experts, begin, end, experts, cursors + wave * experts, [&](uint32_t index, uint32_t place) { place_of[index] = place; });
    __syncthreads();
}

/* the sum of a wavefront's words up to and with the lane's own: additions of lanes 1, 2, 4 and 8 below inside rows of
 * sixteen, then of the rows' last lanes (data-parallel primitives: no LDS round trip) */
template <int control, int row_mask>
__device__ static __forceinline__ uint32_t sort_add_lanes(uint32_t value)
{
    return value + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)value, control, row_mask, 0xF, false);
}

__device__ static __forceinline__ uint32_t wave_inclusive_sum(uint32_t value)
{
    value = sort_add_lanes<0x111, 0xF>(value); /* row_shr:1 */
    value = sort_add_lanes<0x112, 0xF>(value); /* row_shr:2 */
    value = sort_add_lanes<0x114, 0xF>(value); /* row_shr:4 */
    value = sort_add_lanes<0x118, 0xF>(value); /* row_shr:8 */
    value = sort_add_lanes<0x142, 0xA>(value); /* row_bcast:15 into rows 1 and 3 */
    return sort_add_lanes<0x143, 0xC>(value);  /* row_bcast:31 into rows 2 and 3 */
}

/* The sum of the values of the threads before this one, a value a thread of a block of SORT_MOST_WAVES wavefronts; total:
 * of all of them. The wavefronts' sums meet in LDS behind one barrier (a scan over the values in LDS took one a doubling:
 * nine of them). scratch: LDS, SORT_MOST_WAVES words nobody else touches before the block's next barrier. */
__device__ static __forceinline__ uint32_t block_sum_before(uint32_t value, uint32_t *scratch, uint32_t &total)
{
    const uint32_t wave = threadIdx.x / SORT_WAVE, inclusive = wave_inclusive_sum(value);
    if (threadIdx.x % SORT_WAVE == SORT_WAVE - 1u) {
        scratch[wave] = inclusive;
    }
    __syncthreads();
    uint32_t before = 0;
    total = 0;
#pragma unroll
    for (uint32_t other = 0; other < SORT_MOST_WAVES; other++) {
        const uint32_t sum = scratch[other];
        before += other < wave ? sum : 0u;
        total += sum;
    }
    return before + inclusive - value;
}

/* exclusive prefix sums of values[0 .. count) in LDS, in their place, by a block of SORT_MOST_WAVES wavefronts, count at most
 * its threads; total returned (barriers inside, one behind the last write) */
__device__ static __forceinline__ uint32_t block_exclusive_scan(uint32_t *values, uint32_t count, uint32_t *scratch)
{
    uint32_t total;
    const uint32_t before = block_sum_before(threadIdx.x < count ? values[threadIdx.x] : 0u, scratch, total);
    if (threadIdx.x < count) {
        values[threadIdx.x] = before;
    }
    __syncthreads();
    return total;
}

#endif
