// Activations of the wide prompt pass: f16 head + remainder pairs in the order the A operands of
// v_mfma_f32_32x32x16_f16 take them.
//
// Tokens in tiles of 32, columns in super-blocks of 256 of sixteen chunks.  Chunk c of super-block cb of token tile tt is
// 2048 bytes: [head | 2^11 remainder][columns 0-7 | 8-15 of the chunk][32 tokens][8 columns, in the order 0, 2, 1, 3, 4, 6, 5, 7],
// so that a lane (token = lane % 32, half = lane / 32) finds its operand at lane * 16.  Behind the sixteen chunks lie the sums of
// 32 consecutive activations as their pairs hold them, which the formats with an offset per sub-block multiply with their mins, divided
// by 32 (written only where such a format reads them): [head | 2^11 remainder][32 tokens][8 sub-blocks, same order], 1024 bytes.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define WIDE_HD __host__ __device__ __forceinline__
#else
#define WIDE_HD inline
#endif

namespace slai {
namespace wide {

constexpr uint32_t CHUNK_BYTES = 2048, SUMS_OFFSET = 16 * CHUNK_BYTES, SUPER_BYTES = SUMS_OFFSET + 1024;
constexpr uint32_t MAX_TOKENS = 1024;                          // of one pass

// where eight consecutive columns (c8 = column / 8) of token t start (heads; the remainders are 1024 bytes on)
WIDE_HD size_t pair_offset(uint32_t ncb, uint32_t t, uint32_t c8) {
    return (size_t)((t >> 5) * ncb + (c8 >> 5)) * SUPER_BYTES + ((c8 >> 1) & 15u) * CHUNK_BYTES + (c8 & 1u) * 512u + (t & 31u) * 16u;
}
// where the sums of super-block cb of token t start (heads; the remainders are 512 bytes on)
WIDE_HD size_t sums_offset(uint32_t ncb, uint32_t t, uint32_t cb) { return (size_t)((t >> 5) * ncb + cb) * SUPER_BYTES + SUMS_OFFSET + (t & 31u) * 16u; }
// place of element i of eight
WIDE_HD uint32_t wide_pos(uint32_t i) { return (i & 4u) | ((i & 1u) << 1) | ((i >> 1) & 1u); }
WIDE_HD size_t activation_bytes(uint32_t ncols, uint32_t ntokens) { return (size_t)((ntokens + 31) / 32) * ((ncols + 255) / 256) * SUPER_BYTES; }

// How tiles (512 rows x 64 tokens) that are no multiple of the compute units are shared out.  Workgroup i runs on die i mod 8; a die's 32
// workgroups take an eighth of the tiles in whole rounds, and of the `rest` tiles of the last, incomplete round one workgroup each takes super-blocks
// 0 .. cut and every other one the rests of `mains` of them (the last such may have fewer).  Everybody begins a tile at super-block 0
// or at cut, so that the workgroups of a die still read the same weights and activations at about the same time.  (Runs of equal length that begin
// anywhere read them each for itself: gate + up of the 7B shape at 255 tokens 238 us, 124 in plain rounds.)
constexpr uint32_t SHARE_DIES = 8, SHARE_RUNS = 32;
struct TileShare {
    uint32_t units, blocks, ncb, per_die, rounds, rest, mains, cut;
    WIDE_HD TileShare(uint32_t row_units, uint32_t token_blocks, uint32_t ncb_) : units(row_units), blocks(token_blocks), ncb(ncb_) {
        per_die = (units * blocks + SHARE_DIES - 1) / SHARE_DIES;
        rounds = per_die / SHARE_RUNS; rest = per_die % SHARE_RUNS;
        mains = (rest + SHARE_RUNS - rest - 1) / (SHARE_RUNS - rest);        // (0: no incomplete round)
        cut = (ncb * mains + mains) / (mains + 1);                           // at least as long as the rests of `mains` tiles
    }
    struct Part { uint32_t tile, c0, c1, place; bool any; };                 // place: of a shared tile among those of its die
    // part i of a workgroup; parts past the last are not `any`
    WIDE_HD Part part(uint32_t die, uint32_t run, uint32_t i) const {
        uint32_t j = i * SHARE_RUNS + run, c0 = 0, c1 = ncb;
        if (i >= rounds) {
            i -= rounds;
            const bool main = run < rest;
            const uint32_t at = main ? run : (run - rest) * mains + i;
            if (main ? i > 0 : i >= mains || at >= rest) return Part{0, 0, 0, 0, false};
            j = rounds * SHARE_RUNS + at;
            if (main) c1 = cut;
            else c0 = cut;
        }
        const uint32_t tile = die * per_die + j;
        return Part{tile, c0, c1, j - rounds * SHARE_RUNS, j < per_die && tile < units * blocks && c0 < c1};
    }
    WIDE_HD uint32_t token_block(uint32_t tile) const { return tile % blocks; }
    // the row unit of a tile: units 0, 8, 16 .. first (formats differ between the first units and the last, and every die is to have some of each)
    WIDE_HD uint32_t unit(uint32_t tile) const {
        const uint32_t p = tile / blocks, per = units / SHARE_DIES, more = units % SHARE_DIES, edge = more * (per + 1);
        return p < edge ? p / (per + 1) + SHARE_DIES * (p % (per + 1)) : more + (p - edge) / (per ? per : 1u) + SHARE_DIES * ((p - edge) % (per ? per : 1u));
    }
    // super-blocks of the workgroup with the most
    WIDE_HD uint32_t longest() const { return rounds * ncb + (rest ? cut : 0u); }
};

}  // namespace wide
}  // namespace slai
