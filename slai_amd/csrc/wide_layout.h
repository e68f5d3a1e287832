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

}  // namespace wide
}  // namespace slai
