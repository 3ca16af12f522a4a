/*
 * joined_launches.h -- which two launches next to each other in a list the backend queues as one, by a kernel that does both
 * works (ANEMONE_JOINED_KERNEL):
 *
 *   a router's select, small or place launch, then the quantizer of the step's rows    the two side by side: neither may touch what the other writes
 *   the experts' gate and up of a few pairs, then the quantizer of the hidden vectors  a block quantizes what it formed (EXPERT_JOINED_MOST_PAIRS)
 *   the shared expert's hidden step, then the quantizer of its values                  the one's values are the other's, a thread both
 *
 * Every byte that the two launches write is written, with the same value. A pair whose records do not show by themselves that this is
 * so stays two launches. A launch costs 1.3 to 1.7 us of a queue beside its work, and the router's last launch is one block, or one for
 * 384 rows, that leaves the card to the quantizer. A pass, before -> after: one row of float32-scaled FP8 50.6 -> 49.0 us, one row
 * of smaller layers 30.5 -> 28.8 and 36.2 -> 34.8, 2048 rows of FP8 1362 -> 1352, 8192 of FP4 1998 -> 1973, a site's five rows 114.9 -> 114.2.
 */
#ifndef JOINED_LAUNCHES_H
#define JOINED_LAUNCHES_H

#include "anemone_backend.h"

struct joined_launch {
    uint32_t grid[2], block;
    uint32_t numbers[3]; /* the kernel's arguments behind the records and the arena: the first launch's blocks, the second's grid */
};

/* the launches' kernels: two of those that ANEMONE_JOINED_KERNEL names together */
extern "C" bool joined_launch_of(const char *first_function, const char *second_function, const struct kernel_launch &first,
                                 const struct kernel_launch &second, uint64_t arena_bytes, struct joined_launch &out);

#endif
