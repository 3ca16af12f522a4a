/*
 * trunk_deep.h -- which launches of trunk_linear_quantized_interleaved_1 the backend queues as a launch of
 * trunk_linear_quantized_deep_<rows>: the same product, bit for bit, in smaller blocks. By the launch's own record, so that a
 * caller's record of kernel handles holds what it held.
 */
#ifndef TRUNK_DEEP_H
#define TRUNK_DEEP_H

#include <hip/hip_runtime.h> /* what the records mark their functions with */

#include "anemone_backend.h"
#include "anemone_records.h"

struct trunk_deep_launch {
    uint32_t grid[2], shared_bytes;
};

/* The instance, of TRUNK_DEEP_ROWS(instance) rows a block, or TRUNK_DEEP_INSTANCES: none, the launch stays what it is.
 * most_shared_bytes: the dynamic LDS that the card grants a block. */
extern "C" uint32_t trunk_deep_instance(const struct kernel_launch &launch, uint32_t most_shared_bytes, struct trunk_deep_launch &out);

#endif
