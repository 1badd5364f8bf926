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
    // 400 drawn worlds of 190 to 328 thousand, direct over transposed: dispatches into three sets of outputs in turn geomean
    // 0.85, the slowest 0.99; cycles with combine 0.93, 0.995, with the packed one 0.92, 0.996.  Dispatches into the same outputs
    // over and over, with nothing in between, are slower at top-5 and top-6 from 32 MiB of payload on (24 x 83, 4096, top-5
    // 16.7 / 19.4, 8 x 167, 5120, top-5 15.0 / 17.9; cycles of the first 32.5 / 32.1): the line is drawn by the cycles.
    constexpr long long kMostScales = 320 * 1024;
    // (the variants exist with written-through rows only, which payloads of that size have by default)
    return use_fp8 && t.scales_direct != 0 && (t.pack_nt < 0 || (t.pack_nt & 4)) && d.H > 512 &&
           (long long)d.R * d.Tgrid * d.K * (d.H / 128) <= kMostScales;
}

SmallPlan plan_small(const int32_t* num_tokens, int R, int E, int K, int hidden, bool use_fp8, const Tuning& t) {
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
    // Blocks a CU gets, with a token a block and with several: its 256-fold steps are what the time goes by.  The experts'
    // blocks, eight experts each, walk all the lists.
    long long shared_blocks = 0;
    for (int r = 0; r < R; ++r) shared_blocks += ((num_tokens[r] > 0 ? num_tokens[r] : 0) + together - 1) / together;
    const long long expert_blocks = ((long long)E + kSmallExperts - 1) / kSmallExperts;
    const long long apart_layers = (tokens + expert_blocks + kCUs - 1) / kCUs;
    const long long layers = (shared_blocks + expert_blocks + kCUs - 1) / kCUs;
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
        // Those figures have few experts, whose blocks find room beside the tokens' on the 256 CUs.  A second block on a CU
        // walks all the lists once more, which separate launches do not up to 1024 experts (beyond, they have a prefix launch
        // and cost more): 32 x 46, 1024, top-8, 512 / 640 experts bf16 9.8 / 8.7, 10.0 / 10.5, fp8 9.5 / 9.1, 9.7 / 11.2;
        // 24 x 42, 2048, 528 experts 10.9 / 10.5, 10.1 / 10.6; 2 x 860, 1024, 512 experts 10.3 / 9.5, 9.7 / 10.1; 8 x 72, 4096,
        // 768 experts, walking 16 rounds 11.7 / 9.9, 12.6 / 10.3; 32 x 46, 1024 experts 12.2 / 10.9, 12.1 / 11.4.
        // Short rows in the lists of many ranks, each a round of its own, are packed sooner than the rounds are walked, in
        // bf16, by selections x hidden: 32 x 17, 640 (2.8 million) 6.6 / 7.4, 1024 (4.5) 7.0 / 7.8, 2048 (8.9) 8.4 / 7.9;
        // 32 x 32, 1024 (8.4) 7.9 / 8.1; 28 x 24, 1024 (5.5) 7.2 / 7.4; 24 x 24 (4.7) 6.9 / 7.2, 24 x 30 (5.9) 7.3 / 7.3, 12 x 100,
        // top-6 (7.4) 7.9 / 7.2; walking 20 rounds 20 x 28 (4.6) 7.0 / 6.9; with 512 experts 32 x 22, 1024 (5.8) 8.0 / 7.9;
        // top-4 32 x 33, 640 (2.7) 6.6 / 6.8, 1024 (4.3) 6.9 / 7.0, 32 x 40 (5.2) 7.3 / 7.0, 28 x 40, 640 (2.9) 6.7 / 6.4.
        // Above top-8 a token's place among the block's other selections takes longer, and short rows lose by the elements
        // that a round of the lists stands for, in thousands: bf16, top-12, 12 x 44, 1024 (270) 7.9 / 8.9, 16 x 28, 1024
        // (344) 7.6 / 8.3, 32 x 17, 896, 512 experts (209) 8.6 / 9.4, top-10, 12 x 53, 1024 (271) 7.9 / 8.5, but 8 x 92, 1024,
        // top-9 (424) 8.1 / 7.6, and lists of few ranks, whose rounds are full: 2 x 471, 896, top-10 8.4 / 8.0.  fp8, whose rows
        // are half as long: 32 x 25, 896, top-12 (269) 8.6 / 10.3, 16 x 57, 768, top-9 (197) 8.0 / 9.3, 12 x 61, 768, top-10
        // (234) 7.6 / 8.6, and with them from top-5 up 16 x 71, 640, top-8 (182) 8.1 / 9.1, 32 x 19, 896, top-7 (119) 7.6 / 8.2.
        // With a second block on a CU, from 24 rounds on: bf16, 24 x 78, 640, top-4, 384 experts (199) 8.0 / 8.9, 8 x 251, 640,
        // top-6 (321) 8.3 / 9.1, 24 x 37, 1152, top-8 (340) 8.7 / 9.2.
        // A program that set "fused_small_max" has said how many selections the one launch may have.
        const long long per_round = tokens * K * hidden / walked;
        const bool crowded = E < 1024 && layers > 1 &&
                             (layers * walked > (use_fp8 ? 32 : 56) || (walked >= 24 && per_round <= 7 << 16));
        bool short_rows = false;
        if (use_fp8)
            short_rows = E < 1024 && (K > 8 ? walked >= 16 && per_round <= 7 << 16 : K > 4 && walked >= 24 && per_round <= 1 << 18);
        else if (K > 8)
            short_rows = E < 1024 && R >= 8 && walked >= 12 && per_round <= (K > 10 ? 15 << 15 : 5 << 16);
        else if (E < 512)
            short_rows = K > 4 ? walked > 20 && per_round <= 1 << 18 : walked > 28 && tokens * K * hidden <= (1ll << 22);
        const bool pays = t.fused_small_max == kFusedSmallMax && tokens * K <= (long long)t.fused_shared_max && !chosen && K > 2 &&
                          (use_fp8 || K <= 12) &&
                          hidden > 512 && together > 1 && R <= kSmallRanks && walked <= 4 * kSmallWaves &&
                          tokens * walked <= 6144ll * together && !crowded && !short_rows;
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
    // 8.3 / 7.4; 16 x 32, 1024, bf16 (8192) 7.5 / 6.6; 1024 tokens of 768, top-4 (8192) 7.1 / 5.4; but 8 x 64, 4096, top-6
    // (4096) 6.9 / 7.1, 4 x 128, 2048, top-4, bf16 (2048) 4.9 / 5.3: the others' selections in the block are a step more, and
    // a longer one above top-8: 16 x 24, 1024, top-9 (6144) 6.8 / 7.2, 24 x 12, 1024, top-11 (6912) 7.9 / 7.9.
    // And only where a CU gets that many fewer of the blocks, which are eight waves and not four.  fp8, blocks a CU gets: one for
    // two 16 x 24, 2048, top-8 (6144) 6.7 / 6.8, 16 x 26 (6656) 6.9 / 6.8; two for three, hidden 2048 and less: 16 x 32, 2048, 1280
    // experts 8.2 / 8.7, 24 x 16, 1152, top-5, 1296 experts 8.1 / 8.5, from hidden 2049 on, in smaller blocks: 24 x 20, 3072, 528
    // experts 9.3 / 9.1; three for five 12 x 64, 1024, 3588 experts 9.5 / 9.0; two for two 20 x 20, 3072, 520 experts 7.7 / 8.5,
    // three for three 9.1 / 10.8.  bf16: one for two 16 x 26, 2048 (6656) 6.5 / 6.7, hidden 4096 7.3 / 7.8; two for four 4 x 200, 3072,
    // top-4 6.6 / 6.8, but up to hidden 2048 16 x 32, 2560 experts 9.2 / 8.8; three for five 1024, 4096, top-4 8.1 / 8.4; two for five 1024 of 768, top-4, 1280 experts 7.2 / 6.3, one for
    // three 16 x 32, 1024 7.5 / 6.6, one for four 8 x 96, 2048, top-5 6.8 / 6.2.  Top-1 and top-2, every token naming one expert
    // or not: 12 x 64, 1024, top-1, fp8 6.3 / 5.0; 2048, 1024, top-2 9.1 / 6.0, one expert 12.4 / 7.3.
    // fp8, two tokens a block, in the eight waves of four slabs: one for two 12 x 55, 4096, top-2 6.8 / 7.4, three for five 8 x
    // 158, 3328, top-1 7.5 / 8.2, four for seven 8 x 222, 3456, top-1 9.2 / 10.5, two for four with eight rounds of lists 8 x 109,
    // 3968, top-2 7.0 / 7.2, with more of them 16 x 51, 3328, top-1 8.2 / 7.5; in the six of three slabs three for five with
    // eight rounds 8 x 134, 2560, top-1 7.1 / 7.3, with twelve 12 x 101, 2304, top-2 9.1 / 8.6, two for three with twelve 12 x 49,
    // 3072, top-2 6.5 / 6.9.
    bool fewer;
    if (!use_fp8)
        fewer = 2 * apart_layers >= 5 * layers || (hidden <= 2048 && layers >= 2 && apart_layers >= 2 * layers);
    else if (hidden <= 2048 || (hidden > 3072 && K > 5))
        fewer = 3 * apart_layers >= 5 * layers;
    else if (hidden > 3072)
        fewer = apart_layers >= 2 * layers && (K > 3 || walked > 8);
    else
        fewer = 2 * apart_layers >= 3 * layers && (K > 2 || walked > 8) && (K > 5 || walked > 16 || apart_layers > 3);
    const int line = K > 8 ? 8192 : (use_fp8 && apart_layers < 3 * layers ? 6400 : 6144);
    if (fewer && tokens * walked >= line) p.block_tokens = together;
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
