/*
 * router_device.cuh -- the router's select as device code: the affinity, a row's top-k choice with its route weights, and
 * the whole select of a thin step (affinities, choices, job table) by one block, shared by router_select_entry and the
 * fused FFN front. Definitions: include/anemone/router_records.h:8-31, source/kernel_router.cuh of the reference.
 */
#ifndef ROUTER_DEVICE_CUH
#define ROUTER_DEVICE_CUH

#include <type_traits>

#include "exl3_device.cuh" /* det_expf, bf16_to_float */

#define SELECT_THREADS (LINEAR_MAXIMUM_ROWS * WAVE) /* a wavefront for each row */
#define JOB_WORDS (sizeof(struct expert_job_record) / 4u)

__device__ static __forceinline__ float det_log1pf(float y) /* 0 <= y <= 1 */
{
    const float u = __fadd_rn(1.0f, y);
    const float c = __fsub_rn(y, __fsub_rn(u, 1.0f));
    float m = u, e = 0.0f;
    if (u > 1.41421354f) {
        m = __fmul_rn(u, 0.5f);
        e = 1.0f;
    }
    const float f = __fsub_rn(m, 1.0f);
    const float s = __fdiv_rn(f, __fadd_rn(2.0f, f));
    const float z = __fmul_rn(s, s);
    float r = __fmaf_rn(z, 0.222222224f, 0.285714298f);
    r = __fmaf_rn(r, z, 0.400000006f);
    r = __fmaf_rn(r, z, 0.666666687f);
    r = __fmul_rn(r, z);
    const float hfsq = __fmul_rn(__fmul_rn(0.5f, f), f);
    const float log_m = __fsub_rn(f, __fsub_rn(hfsq, __fmul_rn(s, __fadd_rn(hfsq, r))));
    const float low = __fmaf_rn(e, 9.05800061e-06f, __fdiv_rn(c, u));
    return __fmaf_rn(e, 0.693138123f, __fadd_rn(log_m, low));
}

/* 1 / (1 + e^(-score)): the bits of __fdiv_rn(1.0f, __fadd_rn(1.0f, det_expf(-score))) for every float32 score, without
 * det_expf's three tests (see det_silu: the sequence's argument held inside [-104, 89.5] gives the same sums with 1); a
 * not-a-number, which the clamp would lose, is passed through by a select. The library's arithmetic_selfcheck kernel
 * compares the two over all 2^32 scores. */
__device__ static __forceinline__ float det_sigmoid(float score)
{
    const float x = __builtin_amdgcn_fmed3f(-score, -104.0f, 89.5f);
    const float value = quotient_above_one(1.0f, __fadd_rn(1.0f, det_exp_sequence(x)));
    return score != score ? score : value;
}

__device__ static __forceinline__ float router_affinity(float score, uint32_t kind)
{
    if (kind == ROUTER_AFFINITY_SIGMOID) {
        return det_sigmoid(score);
    }
    if (score != score) {
        return score;
    }
    if (score > 20.0f) {
        return sqrtf(score); /* correctly rounded: the compiler default for float32 sqrt and divide */
    }
    const float positive = score > 0.0f ? score : 0.0f;
    return sqrtf(__fadd_rn(positive, det_log1pf(det_expf(-fabsf(score)))));
}

/* A biased affinity as an unsigned word that orders as the select orders values: a not-a-number above everything, then
 * the numbers from +infinity down to -infinity, which is 0x007FFFFF: 0 is below every key. Among equal keys the select
 * takes the lowest expert (include/anemone/router_records.h:12-16 of the reference). */
__device__ static __forceinline__ uint32_t router_key(float biased)
{
    const uint32_t bits = __float_as_uint(biased);
    return biased != biased ? 0xFFFFFFFFu : (bits & 0x80000000u) != 0u ? ~bits : bits | 0x80000000u;
}

/* The largest word of a wavefront, in every lane: a data-parallel-primitive scan (shift by 1, 2, 4, 8 inside rows of 16
 * lanes, then the row broadcasts), no LDS round trip; lane 63 holds the result. A lane without a source takes 0. */
template <int control, int row_mask>
__device__ static __forceinline__ uint32_t dpp_largest_step(uint32_t value)
{
    const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)value, control, row_mask, 0xF, false);
    return other > value ? other : value;
}

__device__ static __forceinline__ uint32_t wave_largest_u32(uint32_t value)
{
    value = dpp_largest_step<0x111, 0xF>(value); /* row_shr:1 */
    value = dpp_largest_step<0x112, 0xF>(value); /* row_shr:2 */
    value = dpp_largest_step<0x114, 0xF>(value); /* row_shr:4 */
    value = dpp_largest_step<0x118, 0xF>(value); /* row_shr:8: lane 15 of a row holds the row's */
    value = dpp_largest_step<0x142, 0xA>(value); /* row_bcast:15 into rows 1 and 3 */
    value = dpp_largest_step<0x143, 0xC>(value); /* row_bcast:31 into rows 2 and 3 */
    return (uint32_t)__builtin_amdgcn_readlane((int)value, 63);
}

#define ROUTER_PLACES (ROUTER_MOST_EXPERTS / WAVE) /* experts a lane holds at most */

/* One row by one wavefront. keys: those of the lane's `places` experts, lane * places and on (0 past them); affinities: the
 * row's, in LDS, written by this wavefront. Lane s < picks ends with the pick of slot s (the picks in ascending expert
 * order): its expert and its route weight. A wavefront that has a vector unit to itself issues an instruction in six cycles
 * whatever it is, so the row's time is its instruction count. A pick is one scan of the wavefront for the largest key: as the
 * experts of a lane lie below those of the next, the lowest lane that holds it has the lowest expert that does, and the
 * lane's own lowest was found beside the scan. The picks are kept sorted by insertion, two instructions a pick, the picks'
 * lanes side by side. (Against experts dealt lane, lane + 64, ..., a second scan for the lowest expert and slots counted behind
 * the picks, 256 experts, 8 picks, us: router_select_entry of one row 5.45 -> 4.6, of eight 5.9 -> 5.1; router_wide_select of 37
 * rows 4.65 -> 3.95, of 8192 10.6 -> 9.3; of 700 rows of 384 experts 6.95 -> 6.2.) */
template <uint32_t PLACES>
__device__ static __forceinline__ void router_row(const float *affinities, uint32_t (&keys)[PLACES], uint32_t lane, uint32_t places, uint32_t picks,
                                                  uint32_t reference_order, float route_scale, uint32_t &expert_out, float &weight_out)
{
    const uint32_t first = lane * places;
    uint32_t sorted = 0xFFFFFFFFu, in_order = 0u; /* lane s: the expert of slot s so far, above every expert where there is none; lane p: pick p */
    for (uint32_t pick = 0; pick < picks; pick++) {
        uint32_t best = keys[0];
#pragma unroll
        for (uint32_t place = 1; place < PLACES; place++) {
            best = keys[place] > best ? keys[place] : best;
        }
        const uint32_t top = wave_largest_u32(best);
        uint32_t candidate = 0u; /* the lane's lowest expert that holds its best */
#pragma unroll
        for (uint32_t place = PLACES; place-- > 0u;) {
            candidate = keys[place] == best ? place : candidate;
        }
        candidate += first;
        const uint32_t holder = (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(best == top));
        const uint32_t winner = (uint32_t)__builtin_amdgcn_readlane((int)candidate, (int)holder);
        const uint32_t taken = winner - first;
#pragma unroll
        for (uint32_t place = 0; place < PLACES; place++) {
            keys[place] = taken == place ? 0u : keys[place];
        }
        /* the slots above the winner's move up by one: slot s takes the larger of the winner and the expert of slot s - 1 (0
         * below the first) where its own is larger than that */
        const uint32_t below = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)sorted, 0x111 /* row_shr:1 */, 0xF, 0xF, false);
        const uint32_t moved = below > winner ? below : winner;
        sorted = moved < sorted ? moved : sorted;
        in_order = lane == pick ? winner : in_order;
    }
    static_assert(ROUTER_MOST_PICKS <= 16u, "the slots' lanes are one row of the wavefront");
    /* a value by readlane: its lane is the same for the whole wavefront (a shuffle is an LDS round trip each) */
    const auto of_lane = [&](float value, uint32_t from) -> float { return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(value), (int)from)); };
    const float value = lane < picks ? affinities[sorted] : 0.0f; /* one LDS read for all of them */
    float sum = 0.0f;
    if (reference_order != 0u && picks == 6u) {
        const float picked = affinities[lane < picks ? in_order : 0u];
        const float p0 = of_lane(picked, 0), p1 = of_lane(picked, 1), p2 = of_lane(picked, 2), p3 = of_lane(picked, 3), p4 = of_lane(picked, 4), p5 = of_lane(picked, 5);
        sum = __fadd_rn(__fadd_rn(__fadd_rn(p0, p4), p2), __fadd_rn(__fadd_rn(p1, p5), p3));
    } else {
#pragma unroll
        for (uint32_t slot = 0; slot < ROUTER_MOST_PICKS; slot++) { /* in slot order from +0; the zeros past the picks change no bit of it */
            sum = __fadd_rn(sum, of_lane(value, slot));
        }
    }
    expert_out = sorted;
    weight_out = __fmul_rn(__fdiv_rn(value, __fadd_rn(sum, 1e-20f)), route_scale);
}

/* A row of `places` places a lane by the narrowest instance that holds them, whose places past them have key 0 and are never
 * taken: the fewer a lane's, the fewer vector instructions a pick. */
template <typename Row> __device__ static __forceinline__ void router_by_places(uint32_t places, Row row)
{
    static_assert(ROUTER_PLACES == 8u, "three instances: up to 256 experts, to 384, to 512");
    if (places <= 4u) {
        row(std::integral_constant<uint32_t, 4u>());
    } else if (places <= 6u) {
        row(std::integral_constant<uint32_t, 6u>());
    } else {
        row(std::integral_constant<uint32_t, 8u>());
    }
}

/* what the select keeps in LDS */
struct __attribute__((aligned(16))) router_select_lds {
    float affinities[LINEAR_MAXIMUM_ROWS * ROUTER_MOST_EXPERTS];
    uint32_t keys[LINEAR_MAXIMUM_ROWS * ROUTER_MOST_EXPERTS];
    float pair_weights[LINEAR_MAXIMUM_ROWS * ROUTER_MOST_PICKS];
    uint32_t pair_experts[LINEAR_MAXIMUM_ROWS * ROUTER_MOST_PICKS];
    uint32_t rows_of[ROUTER_MOST_EXPERTS];     /* bit r: row r picked the expert */
    uint32_t picked_words[ROUTER_MOST_EXPERTS / 32u]; /* bit e % 32 of word e / 32: some row picked expert e */
    /* the experts' matrices, asked for ahead of the picks: behind them the reads stood in the launch's serial chain (with
     * one LDS read for a row's values and one for the picked words: the select of one row then 7.4 -> 6.6 us) */
    uint64_t offsets[ROUTER_MOST_EXPERTS * MODEL_EXPERT_MATRICES];
};

/* The select of a step of at most LINEAR_MAXIMUM_ROWS rows by one block of `threads` threads (whole wavefronts, at least
 * one; every thread of the block calls: two barriers inside). The block forms the affinities, a wavefront picks a row's; the
 * job table then needs of a pair only its expert's rows (a word of bits that the rows' wavefronts set in LDS: integer
 * or, the same whatever the order) and the picked experts below its own (a bit an expert). */
__device__ static __forceinline__ void router_select_body(const struct router_select_arguments &arguments, unsigned char *arena,
                                                          uint32_t thread, uint32_t threads, struct router_select_lds &lds)
{
    const uint32_t experts = arguments.expert_count != 0u ? arguments.expert_count : ROUTER_DEFAULT_EXPERTS;
    const uint32_t picks = arguments.pick_count != 0u ? arguments.pick_count : ROUTER_DEFAULT_PICKS;
    const float scale = arguments.route_scale != 0.0f ? arguments.route_scale : ROUTER_DEFAULT_SCALE;
    const uint32_t wave = thread / WAVE, lane = thread % WAVE, waves = threads / WAVE;
    const float *all_scores = (const float *)(arena + arguments.scores_offset), *bias = (const float *)(arena + arguments.bias_offset);
    /* The affinities and keys are the block's work side by side (one row: a value a thread on four wavefronts in place of four
     * values a lane on one: 4.6 -> 3.95 us, by square roots of softplus 6.15 -> 4.2, two rows of 384 experts 6.6 -> 4.5, eight 8.2 ->
     * 7.85): a row is `places` wavefronts' work, as many rows as there are wavefronts for stand beside each other,
     * and a thread takes its expert of every such row; with fewer wavefronts than places the experts `threads` on as well. Asked
     * for together: the step's rows, the thread's bias and its scores (inside the scores' array whether a row is live or not) */
    const uint32_t places = experts / WAVE;
    uint32_t beside = 0u, own_row = 0u, own_place = __builtin_amdgcn_readfirstlane(wave);
    for (uint32_t left = waves; left >= places; left -= places) { /* a division is twenty instructions, these are two turns */
        beside++;
        if (own_place >= places) {
            own_place -= places;
            own_row++;
        }
    }
    const uint32_t span = beside != 0u ? experts : threads, own_expert = own_place * WAVE + lane;
    if (beside == 0u) {
        beside = 1u;
    }
    const uint32_t step_rows = ((const struct step_block *)(arena + arguments.step_offset))->row_count;
    const uint32_t rows_of_threads = own_row < beside ? arguments.row_count : 0u;
    float scores[LINEAR_MAXIMUM_ROWS];
    const float own_bias = bias[own_expert];
#pragma unroll
    for (uint32_t turn = 0; turn < LINEAR_MAXIMUM_ROWS; turn++) {
        const uint32_t row = own_row + turn * beside;
        scores[turn] = 0.0f;
        if (row < rows_of_threads) {
            scores[turn] = all_scores[row * experts + own_expert];
        }
    }
    const uint64_t *offsets = (const uint64_t *)(arena + arguments.expert_offsets_offset);
    uint64_t own_offsets[MODEL_EXPERT_MATRICES] = {0, 0, 0};
    if (thread < experts) {
#pragma unroll
        for (uint32_t matrix = 0; matrix < MODEL_EXPERT_MATRICES; matrix++) {
            own_offsets[matrix] = offsets[(uint64_t)thread * MODEL_EXPERT_MATRICES + matrix];
        }
    }
    for (uint32_t expert = thread; expert < ROUTER_MOST_EXPERTS; expert += threads) {
        lds.rows_of[expert] = 0u;
    }
    if (thread < ROUTER_MOST_EXPERTS / 32u) {
        lds.picked_words[thread] = 0u;
    }
    const uint32_t live_rows = step_rows < arguments.row_count ? step_rows : arguments.row_count;
    const auto value_of = [&](uint32_t row, uint32_t expert, float score, float its_bias) {
        const uint32_t at = row * experts + expert;
        const float a = router_affinity(score, arguments.affinity_kind);
        lds.affinities[at] = a;
        lds.keys[at] = router_key(__fadd_rn(a, its_bias));
        ((float *)(arena + arguments.affinities_offset))[at] = a;
    };
#pragma unroll
    for (uint32_t turn = 0; turn < LINEAR_MAXIMUM_ROWS; turn++) {
        const uint32_t row = own_row + turn * beside;
        if (row < live_rows && row < rows_of_threads) {
            value_of(row, own_expert, scores[turn], own_bias);
        }
    }
    for (uint32_t expert = own_expert + span; expert < experts; expert += span) { /* fewer threads than experts: every row is this thread's */
        for (uint32_t row = 0; row < live_rows; row++) {
            value_of(row, expert, all_scores[row * experts + expert], bias[expert]);
        }
    }
    __syncthreads(); /* the keys are there, and the zeros before any row sets a bit */
    for (uint32_t row = wave; row < live_rows; row += waves) { /* a wavefront a row (every row at once with eight wavefronts) */
        uint32_t my_expert;
        float my_weight;
        router_by_places(places, [&](auto count) {
            uint32_t keys[count.value];
#pragma unroll
            for (uint32_t place = 0; place < count.value; place++) {
                keys[place] = place < places ? lds.keys[row * experts + lane * places + place] : 0u;
            }
            router_row<count.value>(lds.affinities + row * experts, keys, lane, places, picks, arguments.reference_order, scale, my_expert, my_weight);
        });
        if (lane < picks) { /* lane s holds the pick of slot s */
            lds.pair_experts[row * picks + lane] = my_expert;
            lds.pair_weights[row * picks + lane] = my_weight;
            __hip_atomic_fetch_or(&lds.rows_of[my_expert], 1u << row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_or(&lds.picked_words[my_expert / 32u], 1u << (my_expert % 32u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    for (uint32_t expert = thread; expert < experts; expert += threads) { /* a block of fewer threads than experts: the others' now */
#pragma unroll
        for (uint32_t matrix = 0; matrix < MODEL_EXPERT_MATRICES; matrix++) {
            lds.offsets[expert * MODEL_EXPERT_MATRICES + matrix] =
                expert == thread ? own_offsets[matrix] : offsets[(uint64_t)expert * MODEL_EXPERT_MATRICES + matrix];
        }
    }
    __syncthreads();
    /* The job table: at most 64 pairs, one a lane of the first wavefront. A pair's column is the number of lower rows
     * that picked its expert, its job the number of picked experts below its own, a job's rows the rows that picked its
     * expert. */
    static_assert(LINEAR_MAXIMUM_ROWS * ROUTER_MOST_PICKS <= WAVE, "a step's pairs fit one wavefront");
    const uint32_t pair = thread, pair_count = live_rows * picks;
    const bool mine = pair < pair_count;
    const uint32_t expert = mine ? lds.pair_experts[pair] : 0u;
    /* the picked experts up to the end of word `lane`, summed along the sixteen lanes of a row; a pair takes those ahead of its
     * own word from the word's lane and counts its word's bits below its own (the sixteen words by every lane: 0.2 us more) */
    static_assert(ROUTER_MOST_EXPERTS / 32u == 16u, "the words are a row of lanes");
    const uint32_t own_word = lds.picked_words[expert / 32u], bits = (uint32_t)__builtin_popcount(lds.picked_words[lane % 16u]);
    uint32_t up_to = bits;
    up_to += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)up_to, 0x111, 0xF, 0xF, false); /* row_shr:1 */
    up_to += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)up_to, 0x112, 0xF, 0xF, false); /* row_shr:2 */
    up_to += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)up_to, 0x114, 0xF, 0xF, false); /* row_shr:4 */
    up_to += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)up_to, 0x118, 0xF, 0xF, false); /* row_shr:8 */
    const uint32_t used_jobs = (uint32_t)__builtin_amdgcn_readlane((int)up_to, 15);
    const uint32_t job = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(expert / 32u * 4u), (int)(up_to - bits)) +
                         (uint32_t)__builtin_popcount(own_word & ((1u << (expert % 32u)) - 1u));
    struct expert_job_record *jobs = (struct expert_job_record *)(arena + arguments.jobs_offset);
    if (mine) {
        const uint32_t row = pair / picks, holders = lds.rows_of[expert];
        const uint32_t rows = (uint32_t)__builtin_popcount(holders), column = (uint32_t)__builtin_popcount(holders & ((1u << row) - 1u));
        jobs[job].pair_index[column] = pair;
        jobs[job].route_weight[column] = lds.pair_weights[pair];
        if (column == 0u) {
            jobs[job].gate_offset = lds.offsets[expert * MODEL_EXPERT_MATRICES];
            jobs[job].up_offset = lds.offsets[expert * MODEL_EXPERT_MATRICES + 1u];
            jobs[job].down_offset = lds.offsets[expert * MODEL_EXPERT_MATRICES + 2u];
            jobs[job].row_count = rows;
            jobs[job].expert = expert;
            for (uint32_t unused = rows; unused < LINEAR_MAXIMUM_ROWS; unused++) {
                jobs[job].pair_index[unused] = 0u;
                jobs[job].route_weight[unused] = 0.0f;
            }
        }
    }
    uint32_t *empty_words = (uint32_t *)(jobs + used_jobs);
    const uint32_t empty_count = (arguments.row_count * picks - used_jobs) * JOB_WORDS;
    for (uint32_t word = thread; word < empty_count; word += threads) {
        empty_words[word] = 0u;
    }
}

#endif
