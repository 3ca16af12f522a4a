/* trunk_deep.cpp -- see trunk_deep.h. Host code over the launch's record alone. */
#include "trunk_deep.h"

#include <cstring>

namespace {

uint64_t blocks_of(uint64_t size, uint64_t block)
{
    return (size + block - 1u) / block;
}

} // namespace

/* The instance of the fewest rows a block that gives every block a place on the card at once. A block of the other form has 128 outputs by
 * 64 rows, two K steps in LDS and as long a K step as memory takes to answer (0.9 us), so that a launch of a few dozen blocks is a chain of
 * such steps on as many CUs; fewer rows and outputs a block are more blocks, each of a shorter step (a wavefront alone on a SIMD reads its
 * operands out of LDS one instruction at a time), with three or four steps on their way. Gate and up, and down, us by events, that form | these:
 * 85 rows of 4096 x 896 32.6 | 19.0 and 11.8 | 8.4; 70 of 5120 x 2048 39.6 | 23.8 and 19.6 | 13.0; 158 of 3072 x 1664 26.1 | 18.1 and 16.7 |
 * 11.4; 500 of 4096 x 1024 32.6 | 23.3 and 13.1 | 12.9; 700 of 2048 x 768 19.1 | 17.2 and 11.2 | 10.8; 1100 of 2048 x 768 19.4 | 18.2. With
 * more blocks than places those behind wait for a whole chain: the other form, three blocks a CU, is then the shorter (1100 rows of 768 x
 * 2048 12.4 | 16.1 with 576 blocks). So it is where a CU holds one block alone: 64 rows a block, 7680 inputs, 512 blocks 55.8 | 49.4; 8192
 * inputs, 320 blocks 60.0 | 93.7, 512 blocks 60.2 | 94.2; 16384 inputs, 320 blocks 113.7 | 180.3 (at 256 blocks 112.1 | 93.9, and 32 rows a
 * block, two a CU, 73.7). */
extern "C" uint32_t trunk_deep_instance(const struct kernel_launch &launch, uint32_t most_shared_bytes, struct trunk_deep_launch &out)
{
    struct trunk_linear_quantized_arguments record;
    std::memcpy(&record, launch.argument, sizeof record);
    const uint32_t *const outputs = record.output_size;
    if (launch.block[0] != WIDE_BLOCK_THREADS || launch.block[1] != 1 || launch.block[2] != 1 || launch.grid[2] != 1 ||
        launch.dynamic_shared_byte_count != TRUNK_INTERLEAVED_WINDOW_BYTES || record.row_count == 0 || record.input_size == 0 ||
        record.input_size % 128u != 0 || record.input_size > TRUNK_DEEP_MOST_INPUTS ||
        launch.grid[0] != blocks_of(outputs[0], TRUNK_INTERLEAVED_BLOCK_OUTPUTS) + blocks_of(outputs[1], TRUNK_INTERLEAVED_BLOCK_OUTPUTS) ||
        launch.grid[1] != blocks_of(record.row_count, TRUNK_INTERLEAVED_ROWS)) {
        return TRUNK_DEEP_INSTANCES; /* not the whole product of its record */
    }
    const uint64_t blocks = blocks_of(outputs[0], TRUNK_DEEP_BLOCK_OUTPUTS) + blocks_of(outputs[1], TRUNK_DEEP_BLOCK_OUTPUTS);
    for (uint32_t instance = 0; instance < TRUNK_DEEP_INSTANCES; instance++) {
        const uint32_t rows = TRUNK_DEEP_ROWS(instance), window = TRUNK_DEEP_WINDOW_BYTES(record.input_size, rows);
        const uint64_t groups = blocks_of(record.row_count, rows);
        if (blocks * groups <= TRUNK_DEEP_MOST_BLOCKS(window)) {
            if (window > most_shared_bytes) {
                break;
            }
            out = {{(uint32_t)blocks, (uint32_t)groups}, window};
            return instance;
        }
    }
    return TRUNK_DEEP_INSTANCES;
}
