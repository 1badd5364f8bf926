// Host-side planning shared by the runtime and the kernel launchers: how a world's selections are cut
// into units, what the count kernel needs of LDS, how many work items the cast-back kernel has to
// cover.  Plain C++ (no device code), so that the runtime's bookkeeping can also be built and exercised on
// a machine without a GPU.
#include "ep_kernels.h"

namespace mcep {

size_t count_lds_bytes(const Dims& d) {
    // per wave of the unit and per expert: a 64-bit lane mask and a 16-bit prefix
    return (size_t)(d.plan.selections() / 64) * d.E * (8 + 2) + 64;
}

void plan_units(Dims& d, const Tuning& t) {
    const long long per_rank_sel = (long long)d.max_tokens * d.K;
    const long long big = (per_rank_sel + kBigUnitSelections - 1) / kBigUnitSelections;
    const size_t big_lds = (size_t)(kBigUnitSelections / 64) * d.E * (8 + 2) + 64;
    UnitPlan p;
    if (t.routing_sum != 0 && d.Tgrid > 0 && big * d.R <= kMaxSummedUnits && big_lds <= kMaxCountLdsBytes) {
        p.per_rank = (int)big;
        p.shift = 10;
        p.summed = 1;
        p.carried = t.routing_sum == 1 ? 1 : 0;
    } else {
        p.per_rank = (int)((per_rank_sel + kUnitSelections - 1) / kUnitSelections);
        p.shift = 8;
        p.summed = 0;
    }
    p.total = d.R * p.per_rank;
    d.plan = p;
}

bool scales_direct(const Dims& d, bool use_fp8, const Tuning& t) {
    // Scales straight into their columns, 4-byte stores R * max_tokens floats apart, against a staging row per token and the
    // launch that transposes them, in thousands of scales (selections x groups).  Dispatch / the cycle with the packed
    // combine, us, transposed -> direct: 41 (640 tokens, hidden 1024, top-8) 9.8 / 18.2 -> 7.4 / 15.3; 110 (2 x 858, 1024, top-8,
    // hot experts) 11.0 / 20.8 -> 8.8 / 18.6; 122 (1020, 3072, top-5) 11.2 / 36.9 -> 9.5 / 35.0; 262 (8 x 128, 4096, top-8)
    // 14.4 / 28.4 -> 13.2 / 25.9; 351 (32 x 87, 1792, top-9) 19.8 / 42.4 -> 16.9 / 38.2; 459 (8 x 128, 7168, top-8) 22.1 /
    // 38.6 -> 22.6 / 39.4, (2 x 1024, 7168, top-4) 24.8 / 46.9 -> 24.3 / 46.0; 524 (16 x 128, 4096, top-8) 25.3 / 42.6 ->
    // 24.4 / 42.6.  A large world's 1.8 million take 30 us.  Rows of half a slab and less have not been measured.
    constexpr long long kMostScales = 320 * 1024;
    // (the variants exist with written-through rows only, which payloads of that size have by default)
    return use_fp8 && t.scales_direct != 0 && (t.pack_nt < 0 || (t.pack_nt & 4)) && d.H > 512 &&
           (long long)d.R * d.Tgrid * d.K * (d.H / 128) <= kMostScales;
}

SmallPlan plan_small(const int32_t* num_tokens, int R, int K, int hidden, bool use_fp8, const Tuning& t) {
    long long tokens = 0, lists = 0;           // tokens; rounds of kSmallListRound entries, each rank's list by itself
    int most = 0;
    for (int r = 0; r < R; ++r) {
        tokens += num_tokens[r];
        lists += ((long long)num_tokens[r] * K + kSmallListRound - 1) / kSmallListRound;
        if (num_tokens[r] > most) most = num_tokens[r];
    }
    SmallPlan p;
    if (t.fused_small == 0 || most == 0) return p;
    const bool chosen = t.fused_small_rounds >= 0;      // the option replaces the measured lines
    const long long walked = (long long)R * (((long long)most * K + kSmallListRound - 1) / kSmallListRound);
    const int together = small_block_tokens(hidden);
    if (tokens * K > (long long)t.fused_small_max) {
        // Too many for a token a block.  Up to hidden 4096 several tokens share one: the lists are read that many times
        // less, by eight waves.  Priced by the rounds of all blocks together.  Dispatch, us, apart / in one: fp8, 640
        // tokens of hidden 2048, top-8 (1600) 8.2 / 6.8, 16 x 112, 1024, top-4 (3584) 7.6 / 6.7, 4 x 256, 2048, top-8 (4096)
        // 9.3 / 8.9, 1020, 3072, top-5 (5100) 9.5 / 8.3, 2 x 860, 1024, top-8 (6020) 8.8 / 7.9; (8192) 2048, 1024, top-8
        // 9.2 / 10.3, 8 x 128, 4096 13.1 / 12.6, 4096, 1024, top-2 8.8 / 14.9; (14256) 9.6 / 10.6.  bf16 8.4 / 6.8, 7.5 / 6.4,
        // 10.7 / 8.8, 10.0 / 8.5, 9.5 / 8.1; 10.3 / 10.0, 14.8 / 13.1, 8.0 / 13.6; 10.2 / 10.2.  Every token naming the same
        // experts, or nine in ten an eighth of them, gains as much from top-3 up (2000, 640, top-3 of 3: fp8 9.8 / 6.1, bf16
        // 6.8 / 5.8); not top-1 and top-2, whose selections may all name one expert and queue for its counter.  Many
        // selections are many in the block too: bf16, 500, 1024, top-9 7.0 / 6.4, 8 x 80, 640, top-11 7.2 / 7.1, but
        // 2 x 250, 1024, top-16 8.1 / 8.6 (fp8, with two launches saved, 10.2 / 8.9).
        // A program that set "fused_small_max" has said how many selections the one launch may have.
        const bool pays = t.fused_small_max == kFusedSmallMax && tokens * K <= (long long)t.fused_shared_max && !chosen && K > 2 &&
                          (use_fp8 || K <= 12) &&
                          hidden > 512 && together > 1 && R <= kSmallRanks && walked <= 4 * kSmallWaves &&
                          tokens * walked <= 6144ll * together;
        if (pays) {
            p.fused = p.could = true;
            p.block_tokens = together;
        }
        return p;
    }
    const long long limit = chosen ? t.fused_small_rounds : (use_fp8 ? 6 : 4);
    const int waves = small_block_waves(hidden);
    p.single = R <= kSmallWaveRanks && lists <= limit;
    if (p.single) {
        p.fused = true;
        // Every wave counting by itself (dispatch_alone_kernel): nothing to set up and no barrier, but each entry is
        // compared with each of the token's K experts.  Dispatch, us, alone / shared: one round of one rank's list, 8
        // tokens of hidden 7168, fp8, top-4 4.1 / 4.6, top-8 5.0 / 5.1 (hidden 4096 4.9 / 4.7); bf16, top-8 4.6 / 5.2 (4096
        // 4.6 / 4.5), top-16 6.2 / 6.8.  More rounds: top-1, 2048 tokens of hidden 1024, fp8 6.0 / 8.2 (12.4 when nine
        // tokens in ten name one expert, for whose LDS counter the shared count queues); top-2, 1024 tokens 5.6 / 6.2;
        // top-4, 512 tokens 6.4 / 5.5.  Several ranks, top-1: 4 x 512 tokens 6.4 / 8.4, 2 x 256 4.6 / 4.9, but 4 x 64, where
        // most of a round is missing, 5.6 / 4.3.
        if (R == 1 && (long long)most * K <= kSmallListRound)
            p.alone = K <= 4 || (K <= 8 && !use_fp8) || waves > 4;
        else
            p.alone = K <= 2 && (R == 1 || most * K >= 256);
        return p;
    }
    // The waves of a block share the lists, and go through as many rounds of every rank as the longest list has.  Two
    // prices, against the launches saved (two for fp8, one for bf16).  The rounds a wave of a late token reads one after
    // another; dispatches apart / in one, us: fp8, one to six 10.3 / 4.5 to 12.2 / 8.6 (24 ranks of 20 tokens, hidden
    // 3072), eight 13.0 / 11.2 (32 ranks of 16, 4096); 12 ranks of 8 and one of 256 top-8 tokens, twelve 12.0 / 14.7; bf16,
    // two 8.9 / 7.1 (8 ranks of 64, 2048), four 9.0 / 8.1.  And the rounds of all tokens together, which fill the chip: top-4,
    // 1024 tokens of one rank (8192) fp8 11.1 / 7.9, bf16 8.1 / 7.5 at hidden 1024 and 13.3 / 9.1, 11.5 / 9.2 at 4096;
    // top-2, 2048 tokens (16384) 11.4 / 10.1 and 16.0 / 12.4, bf16 8.1 / 9.6 and 13.6 / 12.9, with one hot expert in eight
    // 11.5 / 13.1, 8.4 / 12.4; top-1, 4096 tokens (32768) 12.5 / 15.1 and 19.6 / 18.3, hot 12.8 / 33.3.  Rows of half a slab
    // and less have not been measured over that range, and stay with the separate launches.
    p.could = hidden > 512 && R <= kSmallRanks && R <= kSmallWaveRanks * waves && (lists + waves - 1) / waves <= limit;
    p.fused = hidden > 512 && R <= kSmallRanks && R <= kSmallWaveRanks * waves &&
              (walked + waves - 1) / waves <= limit && (chosen || tokens * walked <= (use_fp8 ? 16384 : 8192));
    // Several tokens a block, where the blocks' reading of the lists is what takes the time.  One token a block / several,
    // us, by rounds of all tokens: 12 ragged ranks of 70, hidden 1152, top-5 (10080) 7.3 / 5.9; 24 x 20, 3072, top-8 (11520)
    // 8.3 / 7.4; 16 x 32, 2048, bf16 (8192) 7.5 / 6.9; 1024 tokens of 768, top-4 (8192) 7.1 / 5.4; but 8 x 64, 4096, top-6
    // (4096) 6.9 / 7.1, 4 x 128, 2048, top-4, bf16 (2048) 4.9 / 5.3: the others' selections in the block are a step more, and
    // a longer one above top-8: 16 x 24, 1024, top-9 (6144) 6.8 / 7.2, 24 x 12, 1024, top-11 (6912) 7.9 / 7.9.
    if (tokens * walked >= (K <= 8 ? 6144 : 8192)) p.block_tokens = together;
    return p;
}

bool combine_reads_table(const CombineSource& src, bool direct) {
    if (src.tokens < 0 || src.out.base == 0) return true;
    // rows come as addresses from the routes, except that the packed combine looks its tensors up either way
    if (!direct && src.search && (src.src_info.base == 0 || src.layout_range.base == 0)) return true;
    if (!direct && !src.search) return src.x.base == 0 || (src.packed_fp8 && src.scales.base == 0);
    return src.topk_idx.base == 0 || src.topk_weights.base == 0 || src.active.base == 0 || src.x.base == 0 ||
           (src.packed_fp8 && src.scales.base == 0);
}

long long cast_back_chunks(long long max_rows, int num_experts) {
    // every row is in one chunk, each expert has at most one partly filled chunk, and no chunk is empty
    const long long chunks = max_rows / kCastRows + num_experts;
    return chunks < max_rows ? chunks : max_rows;
}

bool cast_back_listed(long long max_rows, int num_experts, int hidden) {
    // Every block reads a thread's run of counts after each other, ceil(E / 256) of them.  Listed / searched, us, by
    // blocks x run: 1024 experts, 128 tokens of hidden 1024, top-8 (4096) 8.6 / 6.8; 8 x 20 tokens of hidden 6784, top-7, 768
    // experts (22344) 12.3 / 13.0, 1024 experts 13.0 / 18.3; 2048 experts, 128 tokens of 7168 (57344) 15.4 / 34.3.
    const long long run = (num_experts + kCastWaves * 64 - 1) / (kCastWaves * 64);
    const long long blocks = cast_back_chunks(max_rows, num_experts) * ((hidden + kCastCols - 1) / kCastCols);
    return run > 2 && blocks * run > 16384;
}

}  // namespace mcep
