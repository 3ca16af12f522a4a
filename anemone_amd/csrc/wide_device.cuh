/*
 * wide_device.cuh -- a block's pipeline over one tile of at most 64 vectors (four MFMA column blocks) by four
 * wavefronts' strips of weight tiles: what the wide routed experts and the trunk's many-row kernel share.
 */
#ifndef WIDE_DEVICE_CUH
#define WIDE_DEVICE_CUH

#include "linear_device.cuh"

#define WIDE_WAVES 4u
#define WIDE_THREADS (WIDE_WAVES * WAVE)
#define WIDE_COLUMN_BLOCKS (WIDE_TILE_PAIRS / 16u)
#define WIDE_BLOCKS_A_CU 3 /* as the windows allow: 168 registers */
#define WIDE_STAGES 2u /* K steps in LDS: one in use, the next on its way */

/* One block's pipeline: MATRICES matrices x STRIP tiles a wavefront, the tile's columns shared. */
/* B128: float32 scales of 128 x 128 blocks and of 128 values in place of the E8M0 codes, as in strip_device.cuh. */
/* STAGES: K steps in LDS; more than WIDE_STAGES: for a launch of few blocks (whole_deep), of tiles of ROWS columns at most. */
template <uint32_t MATRICES, bool BYTES, uint32_t STRIP_TILES, bool B128 = false, uint32_t STAGES = WIDE_STAGES, uint32_t ROWS = WIDE_TILE_PAIRS>
struct wide_chain {
    static_assert(BYTES || !B128, "float32 scales go with one-byte weights");
    static constexpr uint32_t STRIP = STRIP_TILES;
    static constexpr uint32_t STEP_BYTES = BYTES ? BYTE_STEP_BYTES : NIBBLE_STEP_BYTES;
    static constexpr uint32_t TILE_LOADS = STEP_BYTES / 1024u;
    static constexpr uint32_t TILES = MATRICES * STRIP;
    static constexpr uint32_t SCALES_AT = TILES * STEP_BYTES;                    /* inside a wavefront's part */
    static constexpr uint32_t SCALE_LANES = BYTES ? 16u : STRIP * 16u;           /* a word of the weights' scales each */
    static constexpr uint32_t WAVE_BYTES = SCALES_AT + MATRICES * SCALE_LANES * 4u; /* a wavefront's part of a stage */
    static constexpr uint32_t VECTOR_AT = WIDE_WAVES * WAVE_BYTES;               /* inside a stage */
    static constexpr uint32_t STAGE_BYTES = VECTOR_AT + ROWS * 128u;             /* and a K step of the tile's columns' codes */
    static constexpr uint32_t SCALE_STEPS = 4u; /* K steps whose scale words of the columns come together */
    static constexpr uint32_t CHUNK_BYTES = ROWS * SCALE_STEPS * 4u;             /* [column][step of the chunk] */
    static constexpr uint32_t STAGES_BYTES = STAGES * STAGE_BYTES;
    static constexpr bool DEEP = STAGES != WIDE_STAGES;                          /* every chunk has a place of its own */
    static constexpr uint32_t CHUNKS_BYTES = 2u * CHUNK_BYTES;                   /* one in use, the next on its way */
    static constexpr uint32_t WINDOW_BYTES = STAGES_BYTES + (DEEP ? 0u : CHUNKS_BYTES); /* deep: and the chunks of its inputs */
    static constexpr uint32_t WEIGHT_LOADS = TILES * TILE_LOADS + MATRICES;
    static_assert(WEIGHT_LOADS < 64u && WINDOW_BYTES <= 160u * 1024u, "vmcnt has six bits; LDS 160 KB");

    const unsigned char *words[MATRICES], *scales[MATRICES], *codes, *exponents;
    /* no other tile of the launch reads these weights: they are asked for as a stream (whoever places the chain sets it). 300
     * rows of 4096 x 2048 x 256 experts of 4-bit weights: gate/up 387 -> 348 us, down 208 -> 192; 200 rows of float32-scaled FP8
     * 702 -> 645, 361 -> 335; 2048 rows 975 -> 944, 502 -> 489. Where tiles share an expert a stream is read again: all of
     * them streamed, 2048 rows took 1050 and 555. */
    bool once;
    uint32_t tile_bytes, window, chunks, wave, piece_offset, scale_offset, codes_offset[2], exponents_offset;
    uint32_t read_at, scale_at[BYTES ? STRIP : 1], vector_at, vector_scale_at, shift, last_step, lane_of;

    /* The scale words of a column lie in that column's own row: asked for a step at a time they are a cache line a column for
     * four bytes, as many lines as the column's codes and a quarter of a wavefront's. So the words of four K steps come
     * together, a lane a step of a column of the wavefront's own block (a step past the last repeats the last): 2048 rows of
     * 4096 x 2048 x 256 experts of one-byte weights, float32 scales: gate/up 977 -> 948 us, down 493 -> 484; E8M0 scales: 998
     * -> 970, 481 -> 468; 4-bit weights the same time. */
    __device__ __forceinline__ void issue_vector_scales(uint32_t chunk) const
    {
        const uint32_t step = SCALE_STEPS * chunk + lane_of % SCALE_STEPS;
        load_to_lds_4(exponents, exponents_offset + 4u * (step < last_step ? step : last_step),
                      chunks + (DEEP ? chunk : chunk % 2u) * CHUNK_BYTES + wave * (16u * SCALE_STEPS * 4u));
    }

    /* the tile's columns of K step `at` into stage `stage` (every wavefront reads them: behind the barrier that ends the
     * reads of the stage): eight groups of eight columns, two a wavefront. Behind the barrier
     * of a chunk's first step every wavefront is done with the chunk before it, whose place the next chunk's scale words take */
    __device__ __forceinline__ void issue_vectors(uint32_t stage, uint32_t at) const
    {
        const uint32_t base = window + stage * STAGE_BYTES;
#pragma unroll
        for (uint32_t part = 0; part < 2u; part++) {
            load_to_lds_16(codes + (uint64_t)at * 128u, codes_offset[part], base + VECTOR_AT + (2u * wave + part) * 1024u);
        }
        if (!DEEP && at % SCALE_STEPS == 1u) { /* asked for by the step before it: the waits are for everything older than the weights */
            issue_vector_scales(at / SCALE_STEPS + 1u);
        }
    }

    /* the wavefront's own weights and their scales of K step `at` into its part of stage `stage` (no other wavefront
     * reads that part: once this one has read it, it may be asked for again) */
    template <bool ONCE>
    __device__ __forceinline__ void issue_weights(uint32_t stage, uint32_t at) const
    {
        const uint32_t mine = window + stage * STAGE_BYTES + wave * WAVE_BYTES;
#pragma unroll
        for (uint32_t m = 0; m < MATRICES; m++) {
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n++) {
#pragma unroll
                for (uint32_t part = 0; part < TILE_LOADS; part++) {
                    const unsigned char *piece = words[m] + (uint64_t)n * tile_bytes + (uint64_t)at * STEP_BYTES + part * 1024u;
                    const uint32_t to = mine + (m * STRIP + n) * STEP_BYTES + part * 1024u;
                    if constexpr (ONCE) {
                        load_to_lds_16_once(piece, piece_offset, to);
                    } else {
                        load_to_lds_16(piece, piece_offset, to);
                    }
                }
            }
        }
        if (SCALE_LANES == WAVE || lane_of < SCALE_LANES) {
#pragma unroll
            for (uint32_t m = 0; m < MATRICES; m++) {
                load_to_lds_4(scales[m] + (uint64_t)at * (BYTES ? 4u : 64u), scale_offset, mine + SCALES_AT + m * SCALE_LANES * 4u);
            }
        }
    }

    template <typename T>
    __device__ static __forceinline__ T lds_read(uint32_t address)
    {
        return *(const __attribute__((address_space(3))) T *)(uintptr_t)address;
    }

    /* one K step of LIVE column blocks (a constant: the MFMAs of a step stay one straight line) */
    template <uint32_t LIVE>
    __device__ __forceinline__ void consume(uint32_t stage, uint32_t step, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        /* the stage's addresses, once a step: every read below is one of them plus a constant */
        uint32_t base = window + stage * STAGE_BYTES, mine = base + wave * WAVE_BYTES;
        uint32_t vector_scales = chunks + (DEEP ? step / SCALE_STEPS : step / SCALE_STEPS % 2u) * CHUNK_BYTES + 4u * (step % SCALE_STEPS);
        asm volatile("" : "+s"(base), "+s"(mine), "+s"(vector_scales));
        /* a lane's pieces differ from its first in bits 4 to 6 of the place (stages and parts are whole 64 and 128 bytes) */
        uint32_t a_at[4], a_scale_at[BYTES ? STRIP : 1], first_a = mine + read_at, first_b = base + VECTOR_AT + vector_at, b_scale_at = vector_scales + vector_scale_at;
        asm volatile("" : "+v"(first_a), "+v"(first_b), "+v"(b_scale_at));
#pragma unroll
        for (uint32_t t = 0; t < 4u; t++) {
            a_at[t] = first_a ^ (16u * t);
            asm volatile("" : "+v"(a_at[t]));
        }
#pragma unroll
        for (uint32_t n = 0; n < (BYTES ? STRIP : 1u); n++) {
            a_scale_at[n] = mine + scale_at[n];
            asm volatile("" : "+v"(a_scale_at[n]));
        }
        /* the columns' codes as they landed (a column's 128 bytes in the order the quantizer writes them): the B operand's words
         * of one-byte weights four words apart, of 4-bit weights eight permutations a column block. Every wavefront of the
         * block does so for every column block: turned about in place, once a block, by the wavefront that brought them, the
         * columns cost it an LDS round trip ahead of the step's barrier (sizes as above: float32 scales 943 -> 930, 480 ->
         * 470; 8192 rows of 4-bit weights: gate/up 1376 -> 1350, down 755 -> 745) */
        int8_vector b[LIVE];
        uint32_t scale_b[LIVE];
        float float_scale_b[LIVE];
        constexpr uint32_t PIECES = BYTES ? 8u : 4u;
#pragma unroll
        for (uint32_t part = 0; part < PIECES; part++) { /* a place at a time (all of them first: more registers, and the 4-bit down 6 % longer) */
            uint32_t piece_at = first_b ^ (BYTES ? 16u * part : 16u * (part % 2u) + 64u * (part / 2u));
            asm volatile("" : "+v"(piece_at));
#pragma unroll
            for (uint32_t j = 0; j < LIVE; j++) {
                if constexpr (BYTES) {
                    b[j][part] = (int)lds_read<uint32_t>(piece_at + j * 2048u);
                } else {
                    const uint2_t pair = lds_read<uint2_t>(piece_at + j * 2048u);
                    b[j][2u * part] = (int)__builtin_amdgcn_perm(pair.y, pair.x, 0x05010400u);
                    b[j][2u * part + 1u] = (int)__builtin_amdgcn_perm(pair.y, pair.x, 0x07030602u);
                }
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < LIVE; j++) {
            if constexpr (B128) {
                float_scale_b[j] = lds_read<float>(b_scale_at + j * (16u * SCALE_STEPS * 4u));
            } else {
                scale_b[j] = lds_read<unsigned char>(b_scale_at + j * (16u * SCALE_STEPS * 4u));
            }
        }
        __builtin_amdgcn_s_setprio(1); /* the wavefront that feeds the matrix unit goes first at the issue */
#pragma unroll
        for (uint32_t tile = 0; tile < TILES; tile++) {
            int8_vector a = {0, 0, 0, 0, 0, 0, 0, 0};
            if constexpr (B128) {
                const float float_scale_a = lds_read<float>(mine + SCALES_AT + (tile / STRIP) * (SCALE_LANES * 4u));
#pragma unroll
                for (uint32_t v = 0; v < 8u; v++) {
                    const uint2_t w = lds_read<uint2_t>(a_at[v % 4u] + v / 4u * 1024u + tile * STEP_BYTES);
                    a[v] = (int)__builtin_amdgcn_perm(w.y, w.x, shift);
                }
#pragma unroll
                for (uint32_t j = 0; j < LIVE; j++) {
                    const float scale = __fmul_rn(float_scale_a, float_scale_b[j]);
                    const float4_t step = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[j], (float4_t){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 127, 0, 127);
#pragma unroll
                    for (uint32_t v = 0; v < 4u; v++) {
                        chain[tile][j][v] = __fmaf_rn(step[v], scale, chain[tile][j][v]);
                    }
                }
                continue;
            }
            const uint32_t scale_a = lds_read<unsigned char>(a_scale_at[BYTES ? tile % STRIP : 0u] + (BYTES ? 0u : tile % STRIP * 64u) + SCALES_AT + (tile / STRIP) * (SCALE_LANES * 4u));
            if constexpr (BYTES) {
#pragma unroll
                for (uint32_t v = 0; v < 8u; v++) {
                    const uint2_t w = lds_read<uint2_t>(a_at[v % 4u] + v / 4u * 1024u + tile * STEP_BYTES);
                    a[v] = (int)__builtin_amdgcn_perm(w.y, w.x, shift);
                }
            } else {
#pragma unroll
                for (uint32_t T = 0; T < 4u; T++) {
                    /* a byte of the result: the output's nibble of w.x below that of w.y. Rotating w.x right by 0 or 4
                     * and w.y left by 4 or 0 puts them there; the mask picks */
                    const uint2_t w = lds_read<uint2_t>(a_at[T] + tile * STEP_BYTES);
                    const uint32_t low = __builtin_amdgcn_alignbit(w.x, w.x, shift), high = __builtin_amdgcn_alignbit(w.y, w.y, 28u + shift);
                    a[T] = (int)((low & NIBBLE_MASK) | (high & ~NIBBLE_MASK));
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < LIVE; j++) {
                if constexpr (BYTES) {
                    chain[tile][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[j], chain[tile][j], 0, 0, 0, (int)scale_a, 0, (int)scale_b[j]);
                } else {
                    chain[tile][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[j], chain[tile][j], 4, 0, 0, (int)scale_a, 0, (int)scale_b[j]);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the stage is read before the next barrier */
    }

    /* all `total` K steps of LIVE live column blocks; every wavefront of the block calls it (barriers inside) */
    template <uint32_t LIVE, bool ONCE>
    __device__ __forceinline__ void steps(uint32_t total, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        /* Two stages. A wavefront's weights of a step are asked for two steps ahead, as soon as the wavefront itself has
         * read the stage they go to (its part is its own); the tile's columns one step ahead, behind the barrier that
         * ends every wavefront's reads of their stage. Outstanding at the top of step k, oldest first: the weights of k, the columns of k (and a
         * chunk of scale words), the weights of k + 1. */
        issue_vector_scales(0u);
        issue_vectors(0u, 0u);
        issue_weights<ONCE>(0u, 0u);
        if (total > 1u) {
            issue_weights<ONCE>(1u, 1u);
        }
        for (uint32_t step = 0; step < total; step++) {
            if (step + 1u < total) {
                wait_loads<WEIGHT_LOADS>();
            } else {
                wait_loads<0>();
            }
            __syncthreads(); /* every wavefront has read the step before and brought its part of this one */
            if (step + 1u < total) {
                issue_vectors((step + 1u) % 2u, step + 1u);
            }
            consume<LIVE>(step % 2u, step, chain);
            if (step + 2u < total) {
                issue_weights<ONCE>(step % 2u, step + 2u);
            }
        }
    }

    /* The same for a launch whose blocks are so few that a CU has one or two of them: a step there is as long as memory takes to answer what
     * was asked for a step before, so that STAGES - 1 steps are on their way, and the columns' scale words all from the start. A
     * wavefront brings columns where its two groups are live. The weights are asked for through the caches, also where one tile of
     * rows is all there is (`once` is not read): as a stream has not been measured here. */
    template <uint32_t LIVE>
    __device__ __forceinline__ void deep_steps(uint32_t total, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        static_assert((STAGES - 2u) * (WEIGHT_LOADS + 2u) < 64u, "vmcnt has six bits");
        const bool brings = wave < LIVE; /* the same in every lane */
        const auto ask = [&](uint32_t stage, uint32_t step) {
            if (brings) {
                issue_vectors(stage, step);
            }
            issue_weights<false>(stage, step);
        };
        if (brings) {
            for (uint32_t chunk = 0; chunk * SCALE_STEPS < total; chunk++) {
                issue_vector_scales(chunk);
            }
        }
#pragma unroll
        for (uint32_t step = 0; step + 1u < STAGES; step++) {
            if (step < total) {
                ask(step, step);
            }
        }
        uint32_t stage = 0;
        for (uint32_t step = 0; step < total; step++) {
            if (step + STAGES - 1u > total) {
                wait_loads<0>();
            } else if (brings) { /* but for the steps behind this one */
                wait_loads<(STAGES - 2u) * (WEIGHT_LOADS + 2u)>();
            } else {
                wait_loads<(STAGES - 2u) * WEIGHT_LOADS>();
            }
            __syncthreads(); /* every wavefront has read the step before, whose stage is asked for again, and brought its part of this one */
            if (step + STAGES - 1u < total) {
                ask(stage == 0u ? STAGES - 1u : stage - 1u, step + STAGES - 1u);
            }
            consume<LIVE>(stage, step, chain);
            stage = stage + 1u == STAGES ? 0u : stage + 1u;
        }
    }

    __device__ __forceinline__ void whole_deep(uint32_t total, uint32_t live_blocks, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        constexpr uint32_t MOST = ROWS / 16u; /* live column blocks */
        if (live_blocks == 1u || MOST == 1u) {
            deep_steps<1>(total, chain);
        } else if (live_blocks == 2u || MOST == 2u) {
            deep_steps<2>(total, chain);
        } else if constexpr (MOST == 4u) {
            if (live_blocks == 3u) {
                deep_steps<3>(total, chain);
            } else {
                deep_steps<4>(total, chain);
            }
        }
    }

    /* live_blocks: the tile's column blocks that hold a pair, the same in every lane of the block; the sums of the
     * others stay what they were */
    __device__ __forceinline__ void whole(uint32_t total, uint32_t live_blocks, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        static_assert(WIDE_COLUMN_BLOCKS == 4u, "one instance a count of live column blocks");
        if (once) { /* the same in every lane of the block: its own instances, and no test in the steps of the others */
            run<true>(total, live_blocks, chain);
        } else {
            run<false>(total, live_blocks, chain);
        }
    }

    template <bool ONCE>
    __device__ __forceinline__ void run(uint32_t total, uint32_t live_blocks, float4_t (&chain)[TILES][WIDE_COLUMN_BLOCKS]) const
    {
        switch (live_blocks) {
        case 1u:
            steps<1, ONCE>(total, chain);
            break;
        case 2u:
            steps<2, ONCE>(total, chain);
            break;
        case 3u:
            steps<3, ONCE>(total, chain);
            break;
        default:
            steps<4, ONCE>(total, chain);
            break;
        }
    }

    /* matrices: arena addresses of the stored matrices; block_strip: the block's first strip (of STRIP tiles) is
     * WIDE_WAVES block_strip; vector_codes / vector_exponents: vector 0's codes and scale codes; vectors: this lane's
     * two columns' vectors for the codes' loads (lane / 8 of groups 2 wave, 2 wave + 1) and its column's for the scale
     * words' load (column 16 wave + lane / 4); window_address and chunks_address: LDS, STAGES_BYTES and CHUNKS_BYTES */
    __device__ __forceinline__ void place(const unsigned char *const (&matrices)[MATRICES], uint32_t outputs, uint32_t inputs,
                                          uint32_t block_strip, const unsigned char *vector_codes, const unsigned char *vector_exponents,
                                          const uint32_t (&code_vectors)[2], uint32_t exponent_vector, uint32_t window_address, uint32_t chunks_address,
                                          uint32_t wave_index, uint32_t lane, uint32_t &tile0_out)
    {
        const uint32_t tiles = outputs / 16u;
        const uint32_t o = lane % 16u, g = lane / 16u, G = o % 8u, parity = o / 8u, ld = g / 2u, q = g % 2u;
        const uint32_t strip = block_strip * WIDE_WAVES + wave_index;
        /* a strip that reaches past the last tile reads the last tiles again; its surplus sums are not stored */
        const uint32_t tile0 = strip * STRIP + STRIP <= tiles ? strip * STRIP : tiles - STRIP;
        tile0_out = tile0;
        const uint32_t steps = inputs / 128u;
        tile_bytes = steps * STEP_BYTES;
        window = window_address;
        chunks = chunks_address;
        wave = wave_index;
        codes = vector_codes;
        exponents = vector_exponents;
        if constexpr (BYTES) {
            const uint32_t scale_rows = (outputs + 31u) / 32u, row0 = B128 ? tile0 / 8u : tile0 / 2u;
#pragma unroll
            for (uint32_t m = 0; m < MATRICES; m++) {
                words[m] = matrices[m] + (uint64_t)tile0 * steps * STEP_BYTES;
                scales[m] = matrices[m] + (uint64_t)outputs * inputs + (uint64_t)row0 * (inputs / 32u);
            }
            piece_offset = 16u * (lane ^ ((lane >> 3) & 3u));
            /* the strip's tiles lie in one or two rows of scales (32 outputs a row): lanes past them ask for the last again,
             * so that a load touches two cache lines and not one a lane */
            const uint32_t rows_needed = (tile0 + STRIP - 1u) / 2u - row0;
            static_assert(STRIP <= 2u, "a strip of one-byte weights spans two rows of scales at most");
            (void)scale_rows;
            scale_offset = B128 ? 0u : (lane < rows_needed ? lane : rows_needed) * (inputs / 32u);
            read_at = 16u * (32u * (g / 2u) + 4u * G + G / 2u) + 8u * (g % 2u); /* word v: t = v % 4, 32 pieces on for v / 4 */
#pragma unroll
            for (uint32_t n = 0; n < STRIP; n++) {
                scale_at[n] = 4u * ((tile0 + n) / 2u - row0) + g;
            }
            shift = parity == 0u ? 0x06020400u : 0x07030501u;
        } else {
            const uint32_t loads = inputs / 64u;
#pragma unroll
            for (uint32_t m = 0; m < MATRICES; m++) {
                words[m] = matrices[m] + (uint64_t)tile0 * steps * STEP_BYTES;
                scales[m] = matrices[m] + (uint64_t)outputs * inputs / 2u + (uint64_t)tile0 * loads * 32u;
            }
            /* piece p of a tile's K step lands in slot p ^ ((p / 8) % 4): LDS has 32 banks of 4 bytes, and the eight 8-byte
             * reads of sixteen lanes (G = 0 .. 7, twice) then fall on sixteen different banks */
            piece_offset = 16u * (lane ^ ((lane >> 3) & 3u));
            /* lanes past the strip's tiles read its last tile's words again */
            scale_offset = (lane / 16u < STRIP ? lane / 16u : STRIP - 1u) * (loads * 32u) + (lane % 16u) * 4u;
            read_at = 16u * (32u * ld + 4u * G + G / 2u) + 8u * q;
            scale_at[0] = (8u * ld + G) * 4u + 2u * q + parity; /* tile n of the strip: 64 bytes on */
            shift = 4u * parity;
        }
        /* the columns' codes: lane L of a load holds slot L % 8 of column L / 8 of its group of eight and asks for
         * that column's piece (L % 8) ^ (L / 8) ^ (the group's parity); a column block of 16 columns is two groups
         * (2,048 bytes). With the parity the 32 lanes of a pass of consume's reads fall on every bank pair of
         * their half twice, not four times */
#pragma unroll
        for (uint32_t part = 0; part < 2u; part++) {
            codes_offset[part] = code_vectors[part] * inputs + 16u * ((lane % 8u) ^ (lane / 8u) ^ part);
        }
        exponents_offset = exponent_vector * (inputs / 32u);
        last_step = steps - 1u;
        lane_of = lane;
        const uint32_t column = o % 8u, group_bytes = (o / 8u) * 1024u;
        vector_at = group_bytes + 16u * (8u * column + ((BYTES ? 0u : 2u * (g % 2u)) ^ column ^ (o / 8u))) + (BYTES ? 4u * g : 8u * (g / 2u));
        vector_scale_at = 4u * SCALE_STEPS * o + (B128 ? 0u : g);
    }
};

#endif
