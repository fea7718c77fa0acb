// Byte offsets of the FP8 prefill GEMMs' loads, for code on both sides (device kernels, host tests).
//
// A raw buffer load takes a vector offset (per lane) and a scalar one (per wave) and is out of range, returning nothing,
// where vector >= bytes - scalar. What that difference does below zero is not stated, so no scalar offset here is past the
// operand's end: a load that must not read is put out of range by its vector offset alone.
#pragma once

#if defined(__HIPCC__)
#define LQ_HOST_DEVICE __host__ __device__
#else
#define LQ_HOST_DEVICE
#endif

namespace lq {

constexpr unsigned kLoadNothing = 0x80000000u;  // operands are below 2^31 bytes

// Unit u (16 bytes; order of the tiled block: 16-byte pieces t of its first half, then of its second) of weight row n in
// K block 0 of a tiled FP8 matrix of KB blocks of 128: 16-row tiles of 2048 bytes per block.
LQ_HOST_DEVICE inline unsigned weight_unit_offset(int n, int u, int KB) {
  const int r = n & 15;
  return static_cast<unsigned>(n >> 4) * static_cast<unsigned>(KB) * 2048u +
         static_cast<unsigned>(((((r >> 3) * 2 + (u >> 2)) * 8 + (r & 7)) * 4 + (u & 3)) * 16);
}
// Unit u of activation row m in K block 0.
LQ_HOST_DEVICE inline unsigned activation_unit_offset(int m, int u, int K) {
  return static_cast<unsigned>(m) * static_cast<unsigned>(K) + static_cast<unsigned>(u * 16);
}
// Scalar offset of K block kb of `step` bytes a block; of the last of KB for one past it (whose vector offsets carry
// kLoadNothing).
LQ_HOST_DEVICE inline unsigned block_offset(int kb, int KB, int step) {
  return static_cast<unsigned>(kb < KB ? kb : KB - 1) * static_cast<unsigned>(step);
}
// The 256 x 256 tile issues its loads for all its rows, there or not: load i (0 .. 3) of a wave is 64 i rows on, by the scalar
// offset. For loads 0 to 2 that is within an operand of kWholeRows rows; load 3 of fewer than 193, which has no rows then,
// repeats load 0's (what such rows give is never stored). Weights have 256 rows or more.
constexpr int kWholeRows = 129;
LQ_HOST_DEVICE inline unsigned last_load_offset(int rows, unsigned step) { return rows > 192 ? 3u * step : 0u; }

}  // namespace lq
