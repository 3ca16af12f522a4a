/*
 * joined_launches.h -- which two launches next to each other in a list the backend queues as one, by a kernel that does both
 * works (ANEMONE_JOINED_KERNEL):
 *
 *   a router's select, small or place launch, then the quantizer of the step's rows    the two side by side: neither may touch what the other writes
 *   the experts' gate and up of a few pairs, then the quantizer of the hidden vectors  a block quantizes what it formed (EXPERT_JOINED_MOST_PAIRS)
 *   the shared expert's hidden step, then the quantizer of its values                  the one's values are the other's, a thread both
 *
 * Every byte that the two launches write is written, with the same value. A pair whose records do not show by themselves that this is
 * so stays two launches, and so does a pair so large that one kernel for both is the slower (joined_launches.cpp, with both sides'
 * times). What no record shows, the matrices that the experts' job table names, is taken to be nobody's output:
 * linear_routed_experts_prepare refuses ranges that share a byte with them. A launch costs 1.3 to 1.7 us of a queue beside its work, and
 * the router's last launch is one block, or one for 384 rows, that leaves the card to the quantizer. Back to back, us, two -> one: select
 * and quantizer of one row 6.0 -> 4.1, small of 64 rows 7.0 -> 5.1, place of 2048 rows 18.2 -> 14.3, of 8192 38.2 -> 30.1; hidden and
 * quantizer of one row 4.5 -> 2.3, of 8192 35.3 -> 27.2; gate and up and quantizer of 8 pairs of FP4 14.6 -> 12.8, of 64 71.6 -> 69.5.
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
