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

}  // namespace mcep
