// Which kernel, and which instance of it, the RoPE / Q-K norm + RoPE and the
// attention launchers take for a given shape, as host functions free of HIP.
// The launchers call these and nothing else to decide, so a host test can
// check every decision (each head layout of the Qwen3 family and of its
// tensor-parallel shards) without a GPU.
#pragma once

#include "launch_limits.hpp"

#include <initializer_list>

namespace q3k
{
    // ---- RoPE and Q/K norm + RoPE over [tokens, heads, 128] rows ------------

    constexpr int kRopeHeadDim = 128;
    // Below this many (token, head) rows (kSmallLaunchBytes of 256-byte rows)
    // a launch is small (decode): one head per lane group, so more and
    // shorter waves fill more CUs, and write-through stores.
    constexpr int64_t kRopeSmallLaunchRows = kSmallLaunchBytes / (2 * kRopeHeadDim);

    struct RopePlan
    {
        bool fast = false; // rope_heads_kernel; otherwise the generic kernels
        int hg_q = 1;      // heads per lane of Q's waves (1, 2 or 4)
        int hg_k = 1;      // heads per lane of K's waves
        int any_heads = 0; // bit 0 (Q) / bit 1 (K): head count not a multiple of 4, rows per lane group
        bool small = false; // a small launch: write-through stores
    };

    // Waves over a tensor's rows, hg heads per lane; the last one partial when
    // the head count is not a multiple of 4 hg.
    inline int64_t rope_waves(int64_t tokens, int32_t heads, int hg)
    {
        return blocks_for(tokens * heads, static_cast<int64_t>(kRopeHeadsPerWave) * hg);
    }

    // 4 heads per lane when the head count allows it (32 or 64 query heads),
    // else 2 (8 KV heads), else 1.
    inline int rope_heads_per_lane(int32_t heads) { return heads % 16 == 0 ? 4 : heads % 8 == 0 ? 2 : 1; }

    // Every tensor's rows below 2^31 and the grid of the most waves the
    // launcher makes (one head per lane group) within one dispatch.
    inline bool rope_grid_ok(int64_t tokens, int32_t hq, int32_t hk)
    {
        if (!rope_heads_fit(tokens, hq) || (hk > 0 && !rope_heads_fit(tokens, hk)) || !rope_heads_fit(tokens, hq + hk))
            return false;
        const int64_t waves = rope_waves(tokens, hq, 1) + rope_waves(tokens, hk, 1);
        return launch_fits(blocks_for(waves, kRopeWavesPerBlock), kRopeBlock);
    }

    // hk = 0 for one tensor (q3k_rope_bf16).  aligned: every tensor, the table
    // and the norm weights 16-byte aligned.  A head count that is not a
    // multiple of 4 takes one row per lane group, with per-row tokens and
    // positions.  (Two or four such rows per lane group, every load first,
    // did not pay at config 4's tensor-parallel-8 shards: Q/K norm + RoPE at
    // 4/1 heads 7.0 and 8.1 us against 7.2 us with one row, at 8/1 heads
    // 11.3 and 12.1 us against 10.0 us.)
    inline RopePlan plan_rope(int64_t tokens, int32_t hq, int32_t hk, int32_t head_dim, bool aligned)
    {
        RopePlan p;
        if (head_dim != kRopeHeadDim || !aligned || hq <= 0 || hk < 0 || !rope_grid_ok(tokens, hq, hk))
            return p;
        p.fast = true;
        const bool small = tokens * (static_cast<int64_t>(hq) + hk) < kRopeSmallLaunchRows;
        p.small = small;
        p.any_heads = (hq % kRopeHeadsPerWave != 0 ? 1 : 0) | (hk > 0 && hk % kRopeHeadsPerWave != 0 ? 2 : 0);
        if (p.any_heads != 0)
            return p;
        p.hg_q = small ? 1 : rope_heads_per_lane(hq);
        p.hg_k = small ? 1 : (hk == 0 ? p.hg_q : rope_heads_per_lane(hk));
        return p;
    }

    // ---- grouped-query attention ---------------------------------------------

    constexpr int kAttHeadDim = 128;
    constexpr int kAttKeyTile = 64;               // keys per pipeline step
    constexpr int kAttWavesPerBlock = 4;          // waves of a matrix-core block
    constexpr int kAttColsPerWave = 32;           // (position, head) columns of a wave
    constexpr int kAttMaxSplits = 64;             // key slices the combine kernel merges
    // Grids of fewer blocks leave CUs idle: their keys may be split.
    constexpr int64_t kAttSplitTargetBlocks = 512;
    // Decode slices of up to this many keys run as one-wave blocks.
    constexpr int32_t kAttMaxOneWaveSplitKeys = 2 * kAttKeyTile;
    constexpr int32_t kAttDecodeTile = 32; // keys of a decode wave's tile
    // Most blocks a decode step's slices make: of 3593 shapes of up to 511 pairs and
    // 32768 keys the estimate below wanted more for two.
    constexpr int64_t kAttDecodeMaxBlocks = 2048;

    struct AttnSplit
    {
        int32_t splits = 1;
        int32_t split_keys = INT32_MAX;
        int32_t key_groups = 1; // groups of waves of a block that share its columns and divide its keys (1, 2 or 4)
        int32_t decode_waves = 0; // waves of a decode block (1, 2 or 4); 0: not the decode kernel
        int64_t bytes = 0; // workspace of the split (unnormalised O^T, max and sum of each slice, fp32); 0: splits == 1
    };

    // Columns of a block and keys of a step for each number of key groups: four
    // waves side by side and 64-key tiles with one or two groups, two waves and
    // 32-key tiles with four (LDS: 64 KiB, two blocks a CU, or 128 KiB, one).
    constexpr int32_t attn_block_cols(int key_groups) { return kAttColsPerWave * (key_groups == 4 ? 2 : 4); }

    // Estimated time in us of a prefill or chunk (S > 1) with `key_groups` and
    // its keys cut into slices of split_keys, from what the three kernels
    // measured alone and side by side on a CU (1.8-2.1 GHz): a 64-key tile of a
    // 128-column block takes 1.6 us alone on its CU and 1.25 us of CU time beside
    // another block; with two key groups 1.4 us of CU time; with four (64
    // columns) 0.82 us alone, 0.9 us when blocks queue.  A block costs another
    // 3.5-5 us of start and end (Q, the first tiles, the store), which with one
    // key group the other block on the CU hides.  Blocks start longest first, ids
    // i and i + 256 on one CU, and their key counts fall evenly from the last
    // query block's to the first's.  A merge costs a launch and a write and a
    // read of the fp32 slices.
    //
    // Over 31 shapes the plan took within 5% of the best of the 9 to 30 forms
    // timed for 24 of them and within 20% for all (the far ones: one KV head and
    // long split prefills).  One group / two / four, unsplit, in us: 512 tokens of 32 / 8
    // heads 17.7 / 17.6 / 13.0; 1000 of 16 / 8 34 / 27 / 18; 2048 of 16 / 8
    // 52 / 45 / 39; 2048 of 32 / 8 64 / 60 / 75; 2 x 1001 of 32 / 8 41 / 38 / 51;
    // 2048 of 64 / 8 99 / 117 / 146; 4 x 2048 of 32 / 8 200 / 241 / 304.
    inline double attn_prefill_us(int64_t pairs, int64_t cols, int32_t G, int64_t S, int64_t cached, int key_groups,
                                  int64_t split_keys)
    {
        constexpr double kCus = 256.0;
        const int32_t block_cols = attn_block_cols(key_groups);
        const int64_t qblocks = blocks_for(cols, block_cols);
        // tiles of the longest and the shortest block (64 keys each)
        const double last = static_cast<double>(cached);
        double first = static_cast<double>(cached - S + (block_cols + G - 1) / G);
        if (first > last)
            first = last;
        const bool split = split_keys < cached;
        double longest = (last + 63.0) / 64.0, shortest = first / 64.0 + 0.5;
        double blocks = static_cast<double>(pairs * qblocks);
        const double mean_keys = 0.5 * (first + last);
        double merge = 0.0;
        if (split)
        {
            // slices of a block, on average: of four blocks spread over the range
            double slices = 0.0;
            for (int i = 0; i < 4; ++i)
            {
                const int64_t keys = static_cast<int64_t>(first + (last - first) * i / 3.0);
                slices += 0.25 * static_cast<double>(blocks_for(keys, split_keys));
            }
            blocks *= slices;
            longest = static_cast<double>(split_keys) / 64.0;
            // the mean slice is the mean range over the slices
            const double mean = mean_keys / 64.0 / slices;
            shortest = 2.0 * mean > longest ? 2.0 * mean - longest : 0.0;
            merge = 3.5 + slices * static_cast<double>(pairs * cols) * (kAttHeadDim * 4) / 2.0e6;
        }
        const double total = blocks * 0.5 * (longest + shortest);
        auto length = [&](double rank) { return longest - (longest - shortest) * rank / blocks; };
        double us;
        if (key_groups == 1)
        {
            if (blocks <= kCus)
                us = 4.0 + 1.6 * longest;
            else if (blocks <= 2 * kCus)
                us = 5.0 + 1.25 * (longest + length(kCus));
            else
                us = 5.0 + 1.25 * total / kCus + 0.3 * longest;
        }
        else
        {
            const double step = key_groups == 2 ? 1.4 : blocks <= kCus ? 0.82 : 0.9; // us a tile
            const double block_us = key_groups == 2 ? 5.0 : 3.5;
            const double rounds = blocks <= kCus ? 1.0 : blocks <= 2 * kCus ? 2.0 : blocks / kCus + 0.5;
            double work = longest;
            if (blocks > 2 * kCus)
                work = total / kCus > longest ? total / kCus : longest;
            else if (blocks > kCus && 2.0 * length(kCus) > longest)
                work = 2.0 * length(kCus);
            us = rounds * block_us + step * work;
        }
        return us + merge;
    }

    // Key groups and, when can_split, the key split of a prefill or chunk.
    inline AttnSplit plan_attention_prefill(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int64_t cached,
                                            bool can_split)
    {
        AttnSplit best;
        const int32_t G = Hq / Hkv;
        const int64_t cols = S * G, pairs = B * Hkv;
        double best_us = -1.0;
        auto consider = [&](int key_groups, int64_t split_keys) {
            const double us = attn_prefill_us(pairs, cols, G, S, cached, key_groups, split_keys);
            if (best_us >= 0.0 && us >= best_us)
                return;
            best_us = us;
            best = AttnSplit{};
            best.key_groups = key_groups;
            if (split_keys < cached)
            {
                best.splits = static_cast<int32_t>(blocks_for(cached, split_keys));
                best.split_keys = static_cast<int32_t>(split_keys);
                best.bytes = best.splits * pairs * cols * (kAttHeadDim + 2) * 4;
            }
        };
        // one tile of keys: nothing to divide (16 tokens of 32 / 8 heads: 6.8 us
        // with one group, 7.5 with four); two tiles and few columns: as long as the
        // groups' merge (13 tokens after 95: 7.9 us against 8.3)
        if (cached <= kAttKeyTile || (cached <= 2 * kAttKeyTile && cols <= 2 * kAttColsPerWave))
            return best;
        for (int key_groups : {1, 2, 4})
            consider(key_groups, cached);
        best_us -= 0.5; // a split has to give more than the estimates' grain
        // with a block to each CU and more a split gained nothing (2 x 700 tokens
        // after 3000, 352 blocks: 134 us whole, 140-147 us in two to four slices)
        const int64_t blocks = pairs * blocks_for(cols, attn_block_cols(1));
        if (!can_split || blocks > kAttSplitTargetBlocks / 2)
            return best;
        for (const int slices : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64})
        {
            if (slices > kAttMaxSplits || slices > kAttSplitTargetBlocks / blocks + 1)
                break;
            const int64_t keys = blocks_for(blocks_for(cached, slices), kAttKeyTile) * kAttKeyTile;
            if (keys >= 2 * kAttKeyTile && keys < cached)
                consider(1, keys);
            const int64_t step_keys = blocks_for(blocks_for(cached, slices), 2 * kAttKeyTile) * 2 * kAttKeyTile;
            if (step_keys < cached)
                consider(4, step_keys);
        }
        return best;
    }

    // Estimated time in us of attention over at most 32 columns to a (batch, KV
    // head) pair (decode), blocks of `waves` waves and slices of split_keys keys.
    // The measurements behind it: a wave takes 0.95 us a 32-key tile when alone,
    // c busy CUs read 8.6 c / (c + 90) TB/s together up to 5.9, and one CU 31 GB/s
    // beside the others, so uneven CUs cost; one, two or four waves a block put
    // four, two or one block on a CU; start and end take 2.7 us with one wave, 3.3
    // with two and 4.5 with four (the groups' merge), another round of short blocks
    // 2 us, the merge launch 3.8 us with its share of the host.  Of more than 8 columns
    // (several positions) the slices' fp32 results count too, 17 KB for 32 columns beside
    // 33 KB of 64 keys: the first 12 MB written and read hide behind the slices, the rest
    // goes at 6 TB/s (3 x 4 positions after 1843, 64 / 8 heads: 15.3 us in the slices taken
    // without it, 13.3 with; over 220 shapes of 2 to 16 positions 0.7% less, none more
    // than 2% slower, where counting every byte at 5 TB/s made 23 of them so).
    inline double attn_decode_us(int64_t pairs, int64_t cols, int64_t cached, int waves, int64_t split_keys)
    {
        const int64_t keys = split_keys < cached ? split_keys : cached;
        const int64_t slices = blocks_for(cached, keys);
        const int64_t blocks = pairs * slices, slots = 256 * (waves == 1 ? 4 : waves == 2 ? 2 : 1);
        const double chain = 0.95 * static_cast<double>(blocks_for(blocks_for(keys, kAttDecodeTile), waves));
        const double bytes = static_cast<double>(keys) * (4 * kAttHeadDim);
        auto round_us = [&](int64_t n) {
            const double cus = static_cast<double>(n < 256 ? n : 256);
            const double rate = 8.6e6 * cus / (cus + 90.0);
            double us = static_cast<double>(n) * bytes / ((rate < 5.9e6 ? rate : 5.9e6) * (waves == 4 ? 1.0 : 0.95));
            const double cu = n > 256 ? static_cast<double>(blocks_for(n, 256)) * bytes / 31.0e3 : 0.0;
            us = us > cu ? us : cu;
            return us > chain ? us : chain;
        };
        const int64_t full = blocks / slots, rest = blocks % slots;
        double us = waves == 4 ? 4.5 : waves == 2 ? 3.3 : 2.7;
        if (full > 0)
            us += static_cast<double>(full) * round_us(slots);
        if (rest > 0)
            us += round_us(rest);
        const int64_t more = blocks_for(blocks, slots) - 1;
        if (more > 0 && round_us(slots) < 20.0)
            us += 2.0 * static_cast<double>(more);
        if (slices > 1)
        {
            us += 3.8 + 0.006 * static_cast<double>(slices);
            const double moved = static_cast<double>(blocks * cols) * (2 * (kAttHeadDim + 2) * 4);
            if (cols > 8 && moved > 12.0e6)
                us += (moved - 12.0e6) / 6.0e6;
        }
        return us;
    }

    // Waves to a block and, when can_split, the key split of a decode step (or
    // any attention of at most 32 columns a pair).  One launch beats split and
    // merge up to about 600 keys a pair (1 sequence of 250 keys: 6.3 us against
    // 8.6; 16 x 300: 9.0 against 10.6; 1 x 1023: 12.0 against 9.2); 64 x 511 keys
    // of 32 / 8 heads took 27.2 us with two waves a block and 29.6 with four, 40 x
    // 3000 of 16 / 8 105 us whole and 88 in three slices of four-wave blocks.
    inline AttnSplit plan_attention_decode(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int64_t cached, bool can_split)
    {
        const int64_t pairs = B * Hkv, cols = S * (Hq / Hkv);
        AttnSplit best, best_split;
        double best_us = -1.0, best_split_us = -1.0;
        for (const int waves : {4, 2, 1})
        {
            if (waves == 1 && cached > kAttDecodeTile)
                continue;
            const double us = attn_decode_us(pairs, cols, cached, waves, cached);
            if (best_us >= 0.0 && us >= best_us)
                continue;
            best_us = us;
            best.decode_waves = waves;
        }
        if (pairs >= kAttSplitTargetBlocks || cached < 2 * kAttKeyTile)
            return best;
        for (const int slices : {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64})
        {
            if (slices > kAttDecodeMaxBlocks / pairs)
                break;
            const int64_t keys = blocks_for(blocks_for(cached, slices), kAttDecodeTile) * kAttDecodeTile;
            if (keys >= cached || keys < 2 * kAttDecodeTile)
                continue;
            for (const int waves : {4, 2, 1})
            {
                if ((waves == 1) != (keys <= kAttMaxOneWaveSplitKeys))
                    continue;
                const double us = attn_decode_us(pairs, cols, cached, waves, keys);
                if (best_split_us >= 0.0 && us >= best_split_us)
                    continue;
                best_split_us = us;
                best_split.decode_waves = waves;
                best_split.split_keys = static_cast<int32_t>(keys);
                best_split.splits = static_cast<int32_t>(blocks_for(cached, keys));
                best_split.bytes = static_cast<int64_t>(best_split.splits) * B * S * Hq * (kAttHeadDim + 2) * 4;
            }
        }
        if (can_split && best_split_us >= 0.0 && best_split_us < best_us)
            return best_split;
        return best;
    }

    // The key split of a call with a workspace.
    inline AttnSplit plan_attention_split(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int64_t cached)
    {
        if (S * (Hq / Hkv) <= kAttColsPerWave)
            return plan_attention_decode(B, S, Hq, Hkv, cached, true);
        return plan_attention_prefill(B, S, Hq, Hkv, cached, true);
    }

    // Workspace of the most slices a call of these B and S and up to `cached` keys may
    // be cut into: a caller that sizes it once for the length of its cache never has
    // too little for a shorter context.  (The plan's own slices go up and down with the
    // length: 64 sequences of 4 / 1 heads take 4 slices at 16384 keys and 16 at 1924.)
    // With no keys before the S positions there is no shorter context, and it is the
    // call's own: 0 for a prefill of 2048 tokens of 16 / 8 heads, where the bound is 49 MiB.
    inline int64_t attention_workspace_bytes(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int64_t cached)
    {
        const int64_t pairs = B * Hkv, cols = S * (Hq / Hkv);
        if (cached == S)
            return plan_attention_split(B, S, Hq, Hkv, cached).bytes;
        int64_t most, keys; // slices, and the fewest keys of one
        if (cols <= kAttColsPerWave)
        {
            if (pairs >= kAttSplitTargetBlocks || cached < 2 * kAttKeyTile)
                return 0;
            most = kAttDecodeMaxBlocks / pairs;
            keys = 2 * kAttDecodeTile;
        }
        else
        {
            const int64_t blocks = pairs * blocks_for(cols, attn_block_cols(1));
            if (blocks > kAttSplitTargetBlocks / 2)
                return 0;
            most = kAttSplitTargetBlocks / blocks + 1;
            keys = 2 * kAttKeyTile;
        }
        for (const int64_t bound : {static_cast<int64_t>(kAttMaxSplits), blocks_for(cached, keys)})
            most = most < bound ? most : bound;
        return most < 2 ? 0 : most * B * S * Hq * (kAttHeadDim + 2) * 4;
    }

    // Which kernel merges the slices of the query rows.
    enum class AttnMerge
    {
        BlockRow, // a block of four waves a row: few rows (decode), their slices many
        LaneRow,  // 16 lanes a row: many rows of few slices
        WaveRow   // a wave a row: many rows of more slices
    };
    // Up to this many rows a row takes a block (its loads all in flight), above it a
    // wave or 16 lanes: 16384 rows of 4 slices took 13.0 us with a block each and 9.6 us
    // with a wave each, and the whole launch 98.5 with those and 96.1 with 16 lanes.
    constexpr int64_t kAttBlockMergeRows = 2048;
    // Slices that a lane of the 16 holds at once.
    constexpr int32_t kAttLaneMergeSplits = 8;

    inline AttnMerge attn_merge(int64_t S, int64_t rows, int32_t splits)
    {
        if (S == 1 || rows <= kAttBlockMergeRows)
            return AttnMerge::BlockRow;
        return splits <= kAttLaneMergeSplits ? AttnMerge::LaneRow : AttnMerge::WaveRow;
    }

    struct AttnPlan
    {
        bool mfma = false;   // attn_mfma_kernel; otherwise attn_generic_kernel
        int g_instance = 0;  // the compiled group size (1, 2, 4, 8, 16, 32) of a whole-block prefill, or 0: taken at run time
        int waves = kAttWavesPerBlock; // waves that divide a block's columns or, in decode, its keys
        AttnSplit split;     // key groups; splits > 1: the key range is split and attn_combine_kernel merges
    };

    // ks / vs: element strides (batch, position, head, dim) of the K / V
    // views.  aligned: q, k and v 16-byte aligned and out 8-byte aligned.
    // workspace_bytes: what the caller passes (0 without a workspace), and
    // whether that workspace is 16-byte aligned.
    inline AttnPlan plan_attention(int64_t B, int64_t S, int32_t Hq, int32_t Hkv, int32_t D, int64_t start,
                                   const int64_t ks[4], const int64_t vs[4], bool aligned, int64_t workspace_bytes,
                                   bool workspace_aligned)
    {
        AttnPlan p;
        if (Hkv <= 0 || Hq <= 0 || Hq % Hkv != 0)
            return p;
        const int32_t G = Hq / Hkv;
        // tile loads use 32-bit byte offsets of up to kAttKeyTile rows
        const int64_t row_limit = (INT32_MAX - 2 * kAttHeadDim) / (2 * kAttKeyTile);
        p.mfma = G >= 1 && G <= kAttColsPerWave && D == kAttHeadDim && start + S <= INT32_MAX && ks[1] <= row_limit &&
                 vs[1] <= row_limit && ks[3] == 1 && vs[3] == 1 && ks[0] % 8 == 0 && ks[1] % 8 == 0 &&
                 ks[2] % 8 == 0 && vs[0] % 8 == 0 && vs[1] % 8 == 0 && vs[2] % 8 == 0 && aligned;
        if (!p.mfma)
            return p;
        p.split = plan_attention_split(B, S, Hq, Hkv, start + S);
        if (p.split.splits > 1 &&
            (p.split.splits > kAttMaxSplits || workspace_bytes < p.split.bytes || !workspace_aligned))
            p.split = S * G <= kAttColsPerWave ? plan_attention_decode(B, S, Hq, Hkv, start + S, false)
                                               : plan_attention_prefill(B, S, Hq, Hkv, start + S, false);
        if (p.split.decode_waves > 0)
            p.waves = p.split.decode_waves;
        else if (p.split.key_groups == 1 && (G == 1 || G == 2 || G == 4 || G == 8 || G == 16 || G == 32))
            p.g_instance = G;
        return p;
    }
} // namespace q3k
