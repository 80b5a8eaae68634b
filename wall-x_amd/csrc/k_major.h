// Byte arithmetic of an operand stored with K as its slow dimension ([k, cols] bf16 row-major: A under trans_a, B without
// trans_b), as the MFMA kernel loads it: one K step is 32 rows of K, four loading wavefronts take 8 rows each, and a load
// instruction fills 1 KiB of LDS.  No device code in here, so that the arithmetic can be checked at its bounds on the CPU.
#pragma once
#include <stdint.h>

namespace wx {

// Whether the arithmetic below is exact: the matrix and the 32 rows of a K step that may begin in its last row lie
// within 32-bit byte offsets.  (Beyond it rows past K would wrap round into the matrix in place of reading as zero.)
__host__ __device__ inline bool k_major_fits(int64_t k, int64_t cols) {
  return k * cols * 2 < (1ll << 32) && cols * 64 < (1ll << 32);
}

// Byte offset, from the K step's first row and the tile's first column, of the 16 bytes that `lane` loads in instruction
// `i` of loading wavefront `wave`; `tile_cols` is the tile's extent (256 or 128), `row_bytes` the matrix's pitch.
// Instruction i covers rows [rows i, + rows) of the wavefront's 8, rows = 1024 / (2 tile_cols); LDS position `lane` is
// chunk lane % chunks of row lane / chunks, and takes the matrix chunk whose 32-byte unit is XORed for the banks.
// (The pitch is any 32-bit number: a 24-bit product would be wrong from 2^23 columns on.  A row index of one or two bits
// costs a mask and an add per bit, where a 32-bit multiply takes four issue slots.)
__host__ __device__ inline uint32_t k_major_offset(int lane, int wave, int i, int tile_cols, uint32_t row_bytes) {
  const int chunks = tile_cols / 8, rows = 1024 / (tile_cols * 2);
  const int row = lane / chunks, chunk = (lane % chunks) ^ (row << 2) ^ (((rows * i) & 3) << 2) ^ ((wave & 1) << 1);
  uint32_t in_instruction = (0u - (static_cast<uint32_t>(row) & 1u)) & row_bytes;
  if (rows > 2) in_instruction += (0u - (static_cast<uint32_t>(row) >> 1)) & (2u * row_bytes);
  return in_instruction + static_cast<uint32_t>(chunk) * 16u + static_cast<uint32_t>(8 * wave + rows * i) * row_bytes;
}

// Bytes readable from the next K step's first row on, given those from this one's.
__host__ __device__ inline uint32_t k_major_left(uint32_t left, uint32_t step) { return left > step ? left - step : 0u; }

}  // namespace wx
