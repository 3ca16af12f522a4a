/*
 * wide_order_device.cuh -- which strip of outputs and which tile of pairs a block of the wide routed experts takes, for
 * the kernels of the reference's weight formats (kernel_wide_linear.hip) and of gfx950's own (kernel_native_linear.hip).
 *
 * What a launch reads past its algorithmic bytes is the experts' matrices again: every tile of 64 pairs reads its
 * expert's whole matrix, and whether a second tile finds it in a level-2 cache is a matter of which blocks run on one die
 * at one time. The card deals blocks to its eight dies in turn by their number, so the blocks of a number n are those of
 * die n % 8, in the order of n / 8. Die c therefore takes the c-th eighth of the launch's work in the order
 *
 *   runs of tiles of one expert (in pieces of at most ORDER_MOST_TILES)  ->  strips of outputs  ->  the run's tiles
 *
 * so that the tiles of a run that need a strip's weights are neighbours in the order of one die and walk the strip's
 * K steps side by side: the weights come from memory once a run, and the run's columns (256 KB a tile of 4,096 inputs)
 * stay in that die's cache for the strips after the first.
 *
 * The 4-bit launches take this order, but for the narrow down's (BY_RUN; 8192 rows of 4096 x 2048 x 256 experts in gfx950's lane order: 5.5 -> 3.4 GB
 * fetched by a gate/up launch). One-byte launches keep the blocks as dealt: their tiles are taken two at a time, so that
 * the matrix of an expert of up to 128 pairs is read once either way, and the second look at the table costs more (2 to 4 %).
 *
 * Where the runs begin follows from the tile table alone: tiles follow each other in a run where their offsets agree and
 * the pairs of the second follow a full first. A table's unused tiles lie behind its used ones, so the launch's work is
 * what lies before the last used tile; without that the last die would be left with the unused ones.
 */
#ifndef WIDE_ORDER_DEVICE_CUH
#define WIDE_ORDER_DEVICE_CUH

#include "exl3_device.cuh"

#define ORDER_DIES 8u
#define ORDER_MOST_TILES 16u /* a piece of a long run: 16 tiles' columns of 4,096 inputs fill a die's 4 MB */

/* used tiles of the table: one more than the number of the last tile that holds a pair (the same in every lane) */
__device__ static __forceinline__ uint32_t order_used_tiles(const struct wide_expert_tile *tiles, uint32_t tile_count, uint32_t lane)
{
    constexpr uint32_t LOOKS = 4u; /* asked for together: a table's unused tiles are at most its experts */
    for (uint32_t behind = 0; behind < tile_count; behind += LOOKS * WAVE) {
        uint32_t count[LOOKS];
#pragma unroll
        for (uint32_t k = 0; k < LOOKS; k++) {
            const uint32_t distance = behind + k * WAVE + lane + 1u; /* from the table's end */
            count[k] = distance <= tile_count ? tiles[tile_count - distance].pair_count : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < LOOKS; k++) {
            const uint64_t mask = __builtin_amdgcn_ballot_w64(count[k] != 0u);
            if (mask != 0ull) {
                return tile_count - behind - k * WAVE - (uint32_t)__builtin_ctzll(mask);
            }
        }
    }
    return 0u;
}

/* The block's strip of the grid's x and its columns: GROUP consecutive tiles of one run, fewer at the run's end. DOWN:
 * runs are tiles of one down matrix, else of one gate and up. Returns false for a block that has nothing to do. Every
 * lane of a wavefront calls; strips and tile_count: the grid's. Two round trips to the table: the used tiles, and
 * the ORDER_WINDOW tiles around the block's own, a lane a tile (runs are cut where a window ends). alone_out: whether the
 * block's tiles are all of their run (as far as the block sees: a matter of speed, not of results). */
template <uint32_t GROUP, bool DOWN, bool BY_RUN>
__device__ static __forceinline__ bool order_block_of(const struct wide_expert_tile *tiles, uint32_t tile_count, uint32_t strips, uint32_t lane, uint32_t &strip_out,
                                                      struct wide_expert_tile &tile_out, uint32_t &pair_count_out, bool *alone_out = nullptr)
{
    if constexpr (!BY_RUN && GROUP == 1u) {
        strip_out = blockIdx.x;
        tile_out = tiles[blockIdx.y];
        pair_count_out = tile_out.pair_count;
        if (alone_out != nullptr) { /* the neighbours in the table hold another matrix, or lie past it, or hold nothing */
            const auto matrix_of = [&](uint32_t index) -> uint64_t { return DOWN ? tiles[index].down_offset : tiles[index].gate_offset; };
            const uint32_t before = blockIdx.y != 0u ? blockIdx.y - 1u : 0u, behind = blockIdx.y + 1u < tile_count ? blockIdx.y + 1u : blockIdx.y;
            const uint64_t own = DOWN ? tile_out.down_offset : tile_out.gate_offset;
            *alone_out = !(before != blockIdx.y && matrix_of(before) == own) &&
                         !(behind != blockIdx.y && tiles[behind].pair_count != 0u && matrix_of(behind) == own);
        }
        return tile_out.pair_count != 0u;
    }
    uint32_t used = tile_count, at = blockIdx.y, unit = 0;
    if constexpr (BY_RUN) {
        const uint32_t number = blockIdx.x + strips * blockIdx.y;
        used = order_used_tiles(tiles, tile_count, lane);
        /* die c takes units [start, start + share) of the launch's work: shares differ by one at most, and the die holds
         * a block for each (no more units than the grid's blocks, which are dealt the same way) */
        const uint32_t work = strips * used, die = number % ORDER_DIES, place = number / ORDER_DIES;
        const uint32_t left = work % ORDER_DIES, share = work / ORDER_DIES + (die < left ? 1u : 0u);
        if (place >= share) {
            return false;
        }
        unit = die * (work / ORDER_DIES) + (die < left ? die : left) + place;
        at = unit / strips; /* a tile of the run the unit belongs to: a run of L tiles takes L x strips units */
    }
    const uint32_t window = at / WAVE * WAVE, inside = at % WAVE, index = window + lane < used ? window + lane : used - 1u;
    const struct wide_expert_tile mine = tiles[index];
    const uint64_t matrix = DOWN ? mine.down_offset : mine.gate_offset, other_matrix = DOWN ? 0u : mine.up_offset;
    /* tiles that begin a run: the matrices of the lane before, or its pairs, do not lead here */
    const uint64_t matrix_before = __shfl_up(matrix, 1u, WAVE), other_before = __shfl_up(other_matrix, 1u, WAVE);
    const uint32_t pairs_before = __shfl_up(mine.pair_count, 1u, WAVE), first_before = __shfl_up(mine.first_pair, 1u, WAVE);
    const bool begins = lane == 0u || window + lane >= used || matrix != matrix_before || other_matrix != other_before ||
                        pairs_before != WIDE_TILE_PAIRS || mine.pair_count == 0u || first_before + WIDE_TILE_PAIRS != mine.first_pair;
    const uint64_t begin_mask = __builtin_amdgcn_ballot_w64(begins);
    const uint32_t run = WAVE - 1u - (uint32_t)__builtin_clzll(begin_mask << (WAVE - 1u - inside) >> (WAVE - 1u - inside));
    const uint64_t above = inside == WAVE - 1u ? 0ull : begin_mask >> (inside + 1u);
    const uint32_t run_end = above == 0ull ? WAVE : inside + 1u + (uint32_t)__builtin_ctzll(above);
    /* pieces of a long run, in whole ORDER_MOST_TILES from its begin */
    const uint32_t first = run + (inside - run) / ORDER_MOST_TILES * ORDER_MOST_TILES;
    const uint32_t length = run_end - first < ORDER_MOST_TILES ? run_end - first : ORDER_MOST_TILES;
    uint32_t chosen = inside;
    strip_out = blockIdx.x;
    if constexpr (BY_RUN) {
        const uint32_t groups = (length + GROUP - 1u) / GROUP;
        const uint32_t place_inside = unit - (window + first) * strips; /* of the piece's units; those past its groups by strips have no work */
        strip_out = place_inside / groups;
        if (strip_out >= strips) {
            return false;
        }
        chosen = first + GROUP * (place_inside % groups);
    } else if ((inside - first) % GROUP != 0u) {
        return false; /* the block of the tile before this one takes both */
    }
    const uint32_t tile = __builtin_amdgcn_readfirstlane(chosen); /* its lane */
    const auto of_lane = [](uint32_t value, uint32_t from) -> uint32_t { return (uint32_t)__builtin_amdgcn_readlane((int)value, (int)from); };
    const auto of_lane_64 = [&](uint64_t value, uint32_t from) -> uint64_t {
        return ((uint64_t)of_lane((uint32_t)(value >> 32), from) << 32) | of_lane((uint32_t)value, from);
    };
    tile_out.gate_offset = of_lane_64(mine.gate_offset, tile);
    tile_out.up_offset = of_lane_64(mine.up_offset, tile);
    tile_out.down_offset = of_lane_64(mine.down_offset, tile);
    tile_out.first_pair = of_lane(mine.first_pair, tile);
    tile_out.pair_count = of_lane(mine.pair_count, tile);
    pair_count_out = tile_out.pair_count;
    if (alone_out != nullptr) {
        *alone_out = length <= GROUP;
    }
    if constexpr (GROUP == 2u) {
        if (tile + 1u < first + length) {
            pair_count_out += of_lane(mine.pair_count, tile + 1u);
        }
    }
    return tile_out.pair_count != 0u;
}

#endif
