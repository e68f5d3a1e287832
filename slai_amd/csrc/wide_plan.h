// Which form a launch of a wide prompt pass (kernels_prompt_wide.hip) takes.  Plain C++ (no HIP), so that the choice and the share-out of tiles that follows from it
// are checked on the host.
#pragma once

#include <algorithm>
#include <cstdint>

#include "wide_layout.h"

namespace slai {

// Form and number of column ranges for nseg matrices over one input (a gated pair is one, of the rows of either).  WIDE_WHOLE: no ranges; WIDE_SUMMED: partial results are summed by the next norm;
// WIDE_READ: by each of their readers
enum { WIDE_LARGE = 0, WIDE_SMALL, WIDE_SLIM4, WIDE_SLIM8, WIDE_SHARE };
enum WideSplits { WIDE_WHOLE, WIDE_SUMMED, WIDE_READ };
struct WidePlan { int form; uint32_t ksplit; };

// Rows of a matrix that a workgroup of a form has (gated: of the gate matrix and of the up matrix each), and row units of a matrix: what a launch is made of and
// what the choice has to count
inline uint32_t wide_unit_rows(int form, bool gated) { return (gated ? 32u : 64u) * (form == WIDE_SLIM4 || form == WIDE_SLIM8 ? 1u : form == WIDE_SMALL ? 4u : 8u); }
inline uint32_t wide_row_units(uint32_t nrows, int form, bool gated) { return (nrows + wide_unit_rows(form, gated) - 1) / wide_unit_rows(form, gated); }

// The forms of a launch: large, 512 rows x 64 tokens (one workgroup fills a compute unit); small, 256 rows x 32 tokens; and slim, 64 rows x
// 32 tokens with the super-blocks shared out among four waves, or eight where that fills the device no more than once.  The columns are
// cut into ranges as long as that gives more compute units a workgroup (512 small ones; a range has at least two super-blocks of a large one, four of a slim one).
// The form is the one with the smallest estimate.  us a launch in a kernel trace, large or small / slim:
//   7B shape, Q4_K      q/k/v          output         gate + up       down
//     64 tokens     27.8 / 23.9      14.0 / 10.6      52.8 / 37.7      26.0 / 20.3
//    128 tokens     41.6 / 36.8      24.7 / 15.8      87.2 / 69.9      50.1 / 33.4
//    192 tokens     54.4 / 58.0      26.1 / 24.4     115.4 / 102.5     52.7 / 50.1
//    256 tokens     68.8 / 71.3      27.6 / 26.7     121.3 / 128.0     56.9 / 61.9
//    512 tokens    119.3 / 144.1     42.2 / 51.2     232.1 / 261.3     94.9 / 122.9
//    640 tokens    127.7 / 194.6     53.9 / 67.8     246.2 / 361.8    119.8 / 173.1
//    704 tokens    227.1 / 243.8     64.5 / 82.7     351.7 / 446.8    156.4 / 218.7
//    832 tokens    227.5 / 354.6     65.1 / 114.7    356.1 / 641.7    157.2 / 308.6
//   1024 tokens    245.6 / 500.0     74.0 / 166.4    388.0 / 889.9    180.5 / 407.3
// and whole prompts without / with slim launches: GPT-2 small, 64 tokens 857 / 553, 680: 1596 / 1296; the 288-wide model, 36 tokens 326 / 229.
// A slim launch takes 6 us and 2.9 ns (2.6 dealt out in ranges, see below) per 64 rows x 32 tokens x super-block over the whole device (gate + up of the 7B shape by counters: requests to the L2
// at 8.9 TB/s for 23 tokens, 12.8 for 64, so the caches are not at their end; 51 and 68 % of the compute units' time is busy), from 576 tokens on the more the
// more tokens there are (eight super-blocks of columns or more: 704 tokens 3.6 ns, 832: 4.4, 1024: 5.0; four: 3.5 at 1024), and at least 5.2 us for each super-block that a wave takes, which counts where
// it takes more than four.  A large workgroup has a compute unit to itself and a row unit's workgroups one die: as many rounds as the die with the most needs,
// of 3 us and 7.2 us per super-block (6.9 Q4_K, 7.8 Q8_0), and 10 us; a small one 2.8 us alone on its compute unit and 5 beside another, and 8 us; what
// sums partial results (the norm) takes 1 us more and 0.4 us per million of them, what reads each several times (bias + RoPE + cache rows, attention) 2 us per million.
// Over twelve shapes and formats and 64 to 1024 tokens in steps of 64 the picks cost 0.3 % more than the better form of every launch would (3.2 % without the
// many tokens, the dies and the readers in the estimate: 7B shape, Q8_0, two layers, 832 tokens 1411 us for 1193).
inline WidePlan wide_plan(const uint32_t *nrows, int nseg, uint32_t ntokens, uint32_t ncb, WideSplits splits, bool gated, bool may_share) {
    uint32_t r8 = 0, r4 = 0, r1 = 0, rows = 0;
    for (int i = 0; i < nseg; ++i) {
        r8 += wide_row_units(nrows[i], WIDE_LARGE, gated); r4 += wide_row_units(nrows[i], WIDE_SMALL, gated); r1 += wide_row_units(nrows[i], WIDE_SLIM4, gated);
        rows += nrows[i];
    }
    const uint32_t large = r8 * ((ntokens + 63) / 64), small = r4 * ((ntokens + 31) / 32), slim = r1 * ((ntokens + 31) / 32);
    const auto ranges = [&](uint32_t units, uint32_t most) { return splits != WIDE_WHOLE ? std::max(1u, std::min(std::min(units, most), 8u)) : 1u; };
    const uint32_t ks_large = ranges(256u / large, ncb / 2), ks_small = ranges(512u / small, ncb), ks_fill = ranges(256u / slim, (ncb + 3) / 4);
    // A launch that fills the device a little more than once, with four waves, not eight, leaves compute units with one workgroup waiting for those with two: two or
    // four ranges of columns are dealt out more evenly.  us a launch with one / two / four, what sums the results takes up to 1 us more:
    //   Q4_K, down    7B 320 workgroups 53.4 / 45.5 / 41.4, 384: 55.2 / 46.6 / 47.9;  Qwen2-7B 280: 80.5 / 69.5 / 62.5, 336: 86.1 / 71.5 / 73.8
    //   Q4_K, output  7B 320: 20.8 / 18.0 / 18.8, 384: 21.0 / 18.6 / 22.2;  Qwen2-7B 280: 20.5 / 17.4 / 18.0;  Q8_0, 320: 24.8 / 22.4 / 22.7
    //   GPT-2 small, down, 264: 22.1 / 18.4 / 17.6, 348: 27.6 / 20.7 / 20.4
    // From 392 to 512 workgroups two cost as much as one.  (Where partial results are read several times, two pay for long columns alone: q/k/v of the 7B shape at
    // 63 tokens 27.2 / 23.5, and 3.1 for the readers.)
    const bool uneven = ks_fill == 1 && slim > 256 && slim <= 384 && (ncb > 32 ? splits != WIDE_WHOLE : ncb >= 8 && splits == WIDE_SUMMED);
    const uint32_t ks_slim = uneven ? (ncb > 32 && slim <= 320 ? 4u : 2u) : ks_fill;
    // (waves without a super-block help to add up and write: 7B output, 22 tokens 6.9 us with four waves, 6.6 with eight; GPT-2 small, 36 tokens, q/k/v 6.2 / 5.9, output
    // 6.1 / 5.7, MLP 7.3 / 6.7; the 288-wide model, q/k/v 5.7 / 5.3)
    const bool eight = slim * ks_slim <= 256;
    const auto parts = [&](uint32_t ks) {
        if (ks <= 1) return 0.0f;
        return splits == WIDE_SUMMED ? 1.0f + (float)ntokens * (float)rows * (float)(ks - 1) * 4e-7f : (float)ntokens * (float)rows * (float)ks * 2e-6f;
    };
    const bool wide = large * ks_large >= 128;
    const uint32_t rounds = ((r8 * ks_large + 7) / 8 * ((ntokens + 63) / 64) + 31) / 32;
    const float t_wide = wide ? 10.0f + (float)rounds * (7.2f * (float)ncb / (float)ks_large + 3.0f) + parts(ks_large)
                              : 8.0f + (small * ks_small <= 256 ? 2.8f : 5.0f * (float)((small * ks_small + 511) / 512)) * (float)((ncb + ks_small - 1) / ks_small) + parts(ks_small);
    const uint32_t turns = ((ncb + ks_slim - 1) / ks_slim + (eight ? 7 : 3)) / (eight ? 8 : 4);
    const uint32_t tile_tokens = (ntokens + 31) / 32 * 32;
    const float many = tile_tokens > 576 && ncb > 2 ? 1.0f + 0.0003f * (float)(tile_tokens - 576) * (float)(std::min(ncb, 8u) - 2) : 1.0f;
    const float t_slim = std::max(6.0f + (uneven ? 0.0026f : 0.0029f) * (float)slim * (float)ncb * many, turns > 4 ? 5.2f * (float)turns : 0.0f) + parts(ks_slim);
    // Shared tiles, where the longest share is at most nine tenths of whole rounds and nobody has the rests of more than four tiles to finish (320 tokens: six): 7.6 us per super-block, and 21 us (with 20, which the launches below take, the 21 picks nearest to the other forms were no faster than those, and 1024 x 4096 of GPT-2 at 993 tokens 6 us slower).  us a launch, large or slim / shared, gate + up of
    // the 7B shape (43 row units):
    //   tokens      192        256        320        384        448        512        576        640        768        896       1024
    //   Q4_K     112 / 90   130 / 111  132 / 131  214 / 192  235 / 198  247 / 207  255 / 229  264 / 245  367 / 326  383 / 344  404 / 390
    //   Q8_0     126 / 101  144 / 123  138 / 142  243 / 209  264 / 221  271 / 234  281 / 257  293 / 273  394 / 362  414 / 386  (968: 428 / 434)
    // (with every compute unit busy each is slower, 8.3 us per super-block at 1024 tokens, by its clock and not by waits: requests in flight over a
    // super-block's end instead of waiting for them there changed 1.5 %)
    // Not where large workgroups in column ranges are the other choice and fill one round: they cut every tile in two as well, and nobody meets anybody.  q/k/v, us
    // of the prompt that sharing took more: 7B shape, 257 to 320 tokens, Q4_K 14 to 17, Q5_K 11 to 18, Q4_0 8, Q8_0 3; 8192 x 4096 + 2 x 1024, 545: 20; 5120 wide, 193: 12
    // (of 450 shared launches in 26 shapes and formats, those were 33 of the 49 that sharing made slower; in two rounds of ranges it takes 45 to 63 less)
    const bool in_ranges = ks_large > 1 && rounds == 1 && t_wide <= t_slim;
    const wide::TileShare sh(r8, (ntokens + 63) / 64, ncb);
    const uint32_t longest = sh.longest(), whole = (sh.rounds + (sh.rest ? 1u : 0u)) * ncb;
    const float t_share = 21.0f + 7.6f * (float)longest;
    if (may_share && !in_ranges && sh.mains <= 4 && 10 * longest <= 9 * whole && t_share < t_wide && t_share < t_slim) return WidePlan{WIDE_SHARE, 1};
    if (t_slim < t_wide) return WidePlan{eight ? WIDE_SLIM8 : WIDE_SLIM4, ks_slim};
    return wide ? WidePlan{WIDE_LARGE, ks_large} : WidePlan{WIDE_SMALL, ks_small};
}

}  // namespace slai
