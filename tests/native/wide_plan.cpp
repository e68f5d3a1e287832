// wide_plan (wide_plan.h) and what its launch deals out, for callers without HIP.
#include "wide_plan.h"

using namespace slai;

// out: form, column ranges, then of the share-out of the launch's own row units: whole rounds, tiles of a die's last round, most rests a workgroup has, super-blocks of the
// workgroup with the most, super-blocks of whole rounds
extern "C" void wide_plan_of(const uint32_t *nrows, int nseg, uint32_t ntokens, uint32_t ncb, int splits, int gated, int may_share, uint32_t *out) {
    const WidePlan p = wide_plan(nrows, nseg, ntokens, ncb, (WideSplits)splits, gated, may_share);
    uint32_t units = 0;
    for (int i = 0; i < nseg; ++i) units += wide_row_units(nrows[i], p.form, gated);
    const wide::TileShare s(units, (ntokens + 63) / 64, ncb);
    const uint32_t values[7] = {(uint32_t)p.form, p.ksplit, s.rounds, s.rest, s.mains, s.longest(), (s.rounds + (s.rest ? 1u : 0u)) * ncb};
    for (int i = 0; i < 7; ++i) out[i] = values[i];
}
