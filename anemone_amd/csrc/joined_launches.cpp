/* joined_launches.cpp -- see joined_launches.h. Host code over the launches' records alone. */
#include "joined_launches.h"

#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime.h> /* what the records mark their functions with */

#include "anemone_records.h"

namespace {

constexpr uint32_t ROUTER_BLOCK = 512u;       /* threads of the router's launches that are joined, and of their joined kernels */
constexpr uint32_t QUANTIZE_UNIT = 64u, QUANTIZE_128_UNIT = 128u; /* widths of activation_quantize_entry, _128_entry: multiples */
/* Values that a router's last launch and the quantizer of the rows are joined for. Beside the place launch a quantizer's block holds that
 * launch's LDS too, so that a CU has three of them: the quantizer alone is bound by memory, joined it takes longer the more values there
 * are. Back to back, us, place + quantizer -> joined. 32 values a scale, 256 experts and 8 picks: 16 Mi values 25.1 -> 16.7, 32 Mi 38.2 -> 30.1,
 * 40 Mi 43.8 -> 36.7, 64 Mi 77.7 -> 78.7 and 78.0 -> 81.3, 128 Mi 142.8 -> 153.9; 64 experts and one pick, 32 Mi 31.4 -> 29.4, 128 Mi 130.2 ->
 * 152.1. A float32 scale: 16 Mi 25.9 -> 19.9, 24 Mi 31.8 -> 28.0, 32 Mi 38.6 -> 36.4, 40 Mi 44.6 -> 45.8, 64 Mi 63.3 -> 72.1; 128 experts and 6
 * picks, 24 Mi 30.5 -> 28.0, 32 Mi 36.0 -> 36.4; one pick, 8 Mi 12.9 -> 10.4, 16 Mi 19.4 -> 19.6, 24 Mi 24.9 -> 27.5, 128 Mi 123.6 -> 182.0 */
constexpr uint64_t MOST_VALUES = 40u << 20, MOST_VALUES_128 = 24u << 20, MOST_VALUES_128_FEW_PICKS = 16u << 20;
constexpr uint32_t FEW_PICKS = 4u; /* fewer */
constexpr uint32_t MOST_GRID_ROWS = 65534u;
constexpr uint32_t MOST_BLOCKS = 1u << 22;    /* of 512 threads: the runtime counts a grid's threads in 32 bits */

struct byte_range {
    uint64_t first, bytes;
};

bool apart(const byte_range &a, const byte_range &b)
{
    return a.bytes == 0 || b.bytes == 0 || (a.first >= b.first ? a.first - b.first >= b.bytes : b.first - a.first >= a.bytes);
}

template <size_t A, size_t B> bool all_apart(const byte_range (&a)[A], const byte_range (&b)[B])
{
    for (const byte_range &x : a) {
        for (const byte_range &y : b) {
            if (!apart(x, y)) {
                return false;
            }
        }
    }
    return true;
}

template <typename T> T record_of(const struct kernel_launch &launch)
{
    T record;
    std::memcpy(&record, launch.argument, sizeof record);
    return record;
}

bool is_plain(const struct kernel_launch &launch, uint32_t block)
{
    return launch.block[0] == block && launch.block[1] == 1 && launch.block[2] == 1 && launch.grid[2] == 1 && launch.dynamic_shared_byte_count == 0;
}

/* the quantizer's launch: its threads cover the vectors' width, and its values fit the arena (so that no product below wraps). `unit`: the
 * values that its lane order keeps together; a vector of a width that is no multiple of them is written past its end, into the next one's
 * place */
bool quantizer_is_whole(const struct kernel_launch &launch, const struct activation_quantize_arguments &record, uint32_t unit, uint64_t arena_bytes)
{
    return is_plain(launch, LINEAR_ELEMENT_THREADS) && record.width != 0 && record.width % unit == 0 &&
           (uint64_t)launch.grid[0] * LINEAR_ELEMENT_THREADS * 4u >= record.width && (uint64_t)launch.grid[1] * record.width <= arena_bytes;
}

bool join_hidden(const struct kernel_launch &first, const struct kernel_launch &second, uint64_t arena_bytes, struct joined_launch &out)
{
    const auto hidden = record_of<trunk_hidden_arguments>(first);
    const auto quantize = record_of<activation_quantize_arguments>(second);
    if (!is_plain(first, LINEAR_ELEMENT_THREADS) || !quantizer_is_whole(second, quantize, QUANTIZE_UNIT, arena_bytes) || first.grid[1] != second.grid[1] ||
        hidden.width != quantize.width || hidden.hidden_offset != quantize.values_offset ||
        (uint64_t)first.grid[0] * LINEAR_ELEMENT_THREADS * HYPER_VALUES_PER_THREAD < hidden.width) {
        return false;
    }
    const uint64_t values = (uint64_t)first.grid[1] * hidden.width;
    const byte_range outputs[] = {{quantize.codes_offset, values}, {quantize.exponents_offset, values / 32u}, {quantize.operands_offset, 2u * values}};
    const byte_range inputs[] = {{hidden.gate_offset, 2u * values}, {hidden.up_offset, 2u * values}}, own[] = {{hidden.hidden_offset, 2u * values}};
    if (!all_apart(outputs, inputs) || !all_apart(outputs, own) || !all_apart(inputs, own)) {
        return false;
    }
    out = {{second.grid[0], second.grid[1]}, LINEAR_ELEMENT_THREADS, {0, 0, 0}};
    return true;
}

/* The most blocks of gate and up that are joined with the quantizer. A block's quantizing stands behind its own product: while the card
 * is not full of blocks that costs less than the launch it saves, with many short ones it holds places that others wait for. 8 picks, 128
 * experts, us, gate and up + quantizer -> joined. 4-bit, 4 K steps a slice (2048 x 2048, four slices): 1024 blocks 25.1 -> 24.1, 1280 28.7 -> 29.3,
 * 2048 38.9 -> 41.2; 8 steps (4096 x 2048): 1280 45.7 -> 44.4, 2048 71.6 -> 69.5, in gfx950's order 71.8 -> 69.7. One byte, 4 steps: 1536 blocks
 * 32.6 -> 32.0, 2048 40.7 -> 41.0, 4096 70.6 -> 72.3; 8 steps: 1536 59.8 -> 58.5, 4096 142.7 -> 142.1; in gfx950's order 1536 56.7 -> 55.2, 2048
 * 71.5 -> 72.3, 4096 129.0 -> 130.3; one slice of 32 steps: 1536 60.4 -> 58.9, 2048 75.7 -> 80.3, 4096 116.7 -> 123.0 */
uint64_t most_gate_up_blocks(bool one_byte, bool native, uint32_t slices, uint32_t slice_steps)
{
    const bool is_long = slice_steps >= 8u;
    if (!one_byte) {
        return is_long ? 2048u : 1024u;
    }
    return is_long && !native && slices > 1u ? 4096u : 1536u;
}

bool join_gate_up(const char *function, const struct kernel_launch &first, const struct kernel_launch &second, uint64_t arena_bytes,
                  struct joined_launch &out)
{
    const auto gate_up = record_of<expert_gate_up_arguments>(first);
    const auto quantize = record_of<activation_quantize_arguments>(second);
    /* expert_gate_up_[e4m3_][gfx950_]<S>: the weights' bytes and the slices, a wavefront each */
    const char *const form = function + sizeof KERNEL_EXPERT_GATE_UP_STEM - 1u;
    const bool one_byte = std::strncmp(form, "e4m3_", 5) == 0, native = std::strstr(form, "gfx950_") != nullptr;
    const uint32_t strip = EXPERT_STRIP_OUTPUTS(one_byte), slices = (uint32_t)std::strtoul(std::strrchr(function, '_') + 1, nullptr, 10);
    /* a block quantizes the outputs of its own strip alone: there is one for every strip */
    if (slices == 0 || !is_plain(first, 64u * slices) || gate_up.output_size % strip != 0 || first.grid[0] != gate_up.output_size / strip ||
        !quantizer_is_whole(second, quantize, QUANTIZE_UNIT, arena_bytes) || gate_up.output_size != quantize.width ||
        gate_up.hidden_offset != quantize.values_offset || gate_up.pair_count != second.grid[1] || gate_up.pair_count > EXPERT_JOINED_MOST_PAIRS ||
        gate_up.pairs_per_row == 0 || gate_up.input_size > arena_bytes || first.grid[1] > MOST_GRID_ROWS ||
        (uint64_t)first.grid[0] * first.grid[1] > most_gate_up_blocks(one_byte, native, slices, gate_up.input_size / 128u / slices)) {
        return false;
    }
    const uint64_t values = (uint64_t)second.grid[1] * quantize.width, jobs = first.grid[1];
    const uint64_t inputs = ((uint64_t)gate_up.pair_count + gate_up.pairs_per_row - 1u) / gate_up.pairs_per_row * gate_up.input_size;
    const byte_range outputs[] = {{quantize.codes_offset, values}, {quantize.exponents_offset, values / 32u}, {quantize.operands_offset, 2u * values}};
    /* the matrices, which the jobs name, are nobody's output (joined_launches.h) */
    const byte_range read[] = {{gate_up.jobs_offset, jobs * sizeof(struct expert_job_record)}, {gate_up.codes_offset, inputs}, {gate_up.exponents_offset, inputs / 32u}};
    const byte_range own[] = {{gate_up.hidden_offset, 2u * values}};
    if (!all_apart(outputs, read) || !all_apart(outputs, own) || !all_apart(read, own)) {
        return false;
    }
    out = {{first.grid[0], (uint32_t)jobs + 1u}, 64u * slices, {(uint32_t)jobs, 0, 0}};
    return true;
}

bool join_router(const char *function, const char *second_function, const struct kernel_launch &first, const struct kernel_launch &second, uint64_t arena_bytes,
                 struct joined_launch &out)
{
    const bool wide_scales = std::strcmp(second_function, KERNEL_ACTIVATION_QUANTIZE_128) == 0;
    const uint32_t unit = wide_scales ? QUANTIZE_128_UNIT : QUANTIZE_UNIT;
    const auto quantize = record_of<activation_quantize_arguments>(second);
    if (!is_plain(first, ROUTER_BLOCK) || first.grid[1] != 1 || !quantizer_is_whole(second, quantize, unit, arena_bytes)) {
        return false;
    }
    const uint64_t values = (uint64_t)second.grid[1] * quantize.width;
    const byte_range read[] = {{quantize.values_offset, 2u * values}};
    /* the quantizer of 128 values a scale writes no operands: they are kept apart all the same */
    const byte_range written[] = {{quantize.codes_offset, values}, {quantize.exponents_offset, values / 32u}, {quantize.operands_offset, 2u * values}};
    const bool is_select = std::strcmp(function, KERNEL_ROUTER_SELECT) == 0;
    const uint32_t pick_count = is_select ? record_of<router_select_arguments>(first).pick_count : record_of<router_wide_arguments>(first).pick_count;
    const uint64_t picks = pick_count != 0 ? pick_count : ROUTER_DEFAULT_PICKS;
    if (values > (!wide_scales ? MOST_VALUES : picks < FEW_PICKS ? MOST_VALUES_128_FEW_PICKS : MOST_VALUES_128)) {
        return false;
    }
    if (is_select) {
        const auto select = record_of<router_select_arguments>(first);
        const uint64_t experts = select.expert_count != 0 ? select.expert_count : ROUTER_DEFAULT_EXPERTS, rows = select.row_count;
        const byte_range inputs[] = {{select.step_offset, sizeof(struct step_block)}, {select.scores_offset, rows * experts * 4u},
                                     {select.bias_offset, experts * 4u}, {select.expert_offsets_offset, experts * MODEL_EXPERT_MATRICES * 8u}};
        const byte_range outputs[] = {{select.affinities_offset, rows * experts * 4u}, {select.jobs_offset, rows * picks * sizeof(struct expert_job_record)}};
        if (!all_apart(written, inputs) || !all_apart(written, outputs) || !all_apart(read, outputs)) {
            return false;
        }
    } else {
        const auto wide = record_of<router_wide_arguments>(first);
        const uint64_t experts = wide.expert_count != 0 ? wide.expert_count : ROUTER_DEFAULT_EXPERTS, rows = wide.row_count;
        const uint64_t pairs = rows * picks;
        const byte_range inputs[] = {{wide.step_offset, sizeof(struct step_block)},
                                     {wide.expert_offsets_offset, experts * MODEL_EXPERT_MATRICES * 8u},
                                     {wide.picks_offset, pairs * sizeof(struct router_pick)},
                                     {wide.counts_offset, (rows + ROUTER_SORT_ROWS - 1u) / ROUTER_SORT_ROWS * experts * 4u}};
        const byte_range outputs[] = {{wide.pairs_offset, pairs * sizeof(struct wide_pair)},
                                      {wide.runs_offset, experts * sizeof(struct wide_run)},
                                      {wide.tiles_offset, ROUTER_WIDE_TILES_OF(rows, picks, experts) * sizeof(struct wide_expert_tile)},
                                      {wide.jobs_offset, ROUTER_WIDE_JOBS_OF(rows, picks, experts) * sizeof(struct expert_job_record)}};
        if (!all_apart(written, inputs) || !all_apart(written, outputs) || !all_apart(read, outputs)) {
            return false;
        }
    }
    constexpr uint32_t TOGETHER = ROUTER_BLOCK / LINEAR_ELEMENT_THREADS;
    const uint64_t blocks = (uint64_t)first.grid[0] + ((uint64_t)second.grid[0] * second.grid[1] + TOGETHER - 1u) / TOGETHER;
    if (blocks > MOST_BLOCKS) {
        return false;
    }
    out = {{(uint32_t)blocks, 1}, ROUTER_BLOCK, {first.grid[0], second.grid[0], second.grid[1]}};
    return true;
}

} // namespace

extern "C" bool joined_launch_of(const char *first_function, const char *second_function, const struct kernel_launch &first,
                                 const struct kernel_launch &second, uint64_t arena_bytes, struct joined_launch &out)
{
    if (std::strcmp(first_function, KERNEL_TRUNK_HIDDEN) == 0) {
        return join_hidden(first, second, arena_bytes, out);
    }
    if (std::strncmp(first_function, KERNEL_EXPERT_GATE_UP_STEM, sizeof KERNEL_EXPERT_GATE_UP_STEM - 1u) == 0) {
        return join_gate_up(first_function, first, second, arena_bytes, out);
    }
    return join_router(first_function, second_function, first, second, arena_bytes, out);
}
