// Device code shared by the kernels that prepare the backward's operands: the
// bit transpose of packed signs and the 16-bit copies of scales.
#pragma once
#include "common.hpp"

namespace qste {

// Bit transpose of a packed sign matrix: in [rows][in_pitch] bytes (bit j of
// byte b is column 8b + j) -> out [cols][out_pitch] bytes (bit i of byte b is
// row 8b + i); bits for rows >= rows are zero.  One thread per 8 x 8 block:
// eight row bytes become one 64-bit word (byte = row, bit = column) whose
// transpose (three delta swaps) gives one byte per column.
__device__ __forceinline__ uint64_t transpose_8x8(uint64_t x) {
  uint64_t t;
  t = (x ^ (x >> 7)) & 0x00AA00AA00AA00AAull;
  x = x ^ t ^ (t << 7);
  t = (x ^ (x >> 14)) & 0x0000CCCC0000CCCCull;
  x = x ^ t ^ (t << 14);
  t = (x ^ (x >> 28)) & 0x00000000F0F0F0F0ull;
  x = x ^ t ^ (t << 28);
  return x;
}

// A workgroup transposes 128-row x 512-column tiles through LDS (walking
// row tiles by gridDim.y): the input rows arrive as 16-byte loads, a thread
// transposes the 8 x 8 blocks of one column byte over a 64-row group (eight
// row blocks at a time, so each of its 8 columns gathers 64 rows into one
// 8-byte LDS word), and every output column leaves as 16 contiguous bytes
// (8-byte stores by consecutive lanes).  Tiles of 128 rows give a
// 3072 x 768 sign matrix 48 workgroups (12 with 512-row tiles: 6.0 instead
// of 11.8 us).  out_pitch must be a multiple of 8.
constexpr int kTrRows = 128, kTrColBytes = 64;  // tile: 128 rows x 512 columns
constexpr int kTrGroups = kTrRows / 64;          // 64-row groups per tile
constexpr int kTrPad = 4;                        // bytes of padding per staged input row
struct TransposeLds {
  __attribute__((aligned(16))) uint8_t tile[kTrRows][kTrColBytes + kTrPad];
  uint64_t otile[8 * kTrColBytes][kTrGroups];  // [column][64-row group]
};

struct TransposeJob {
  const uint8_t* in;
  uint8_t* out;
  int64_t rows, cols, in_pitch, out_pitch, row_tiles;

  int64_t col_tiles() const { return (in_pitch + kTrColBytes - 1) / kTrColBytes; }
};

// row tiles cover every output byte (out_pitch * 8 rows, the padding
// included, which reads as zero)
inline TransposeJob transpose_job(const uint8_t* in, uint8_t* out, int64_t rows, int64_t cols, int64_t in_pitch,
                                  int64_t out_pitch) {
  return {in, out, rows, cols, in_pitch, out_pitch, (out_pitch * 8 + kTrRows - 1) / kTrRows};
}

// A workgroup of 256: tiles (bx, ty0), (bx, ty0 + step), ...
__device__ __forceinline__ void transpose_tiles(const TransposeJob& job, int64_t bx, int64_t ty0, int64_t step,
                                                TransposeLds& lds) {
  auto& tile = lds.tile;
  auto& otile = lds.otile;
  const uint8_t* const in = job.in;
  uint8_t* const out = job.out;
  const int64_t rows = job.rows, cols = job.cols, in_pitch = job.in_pitch, out_pitch = job.out_pitch;
  const int64_t cb0 = bx * kTrColBytes;
  const int tid = threadIdx.x;
  const bool vec = (in_pitch & 15) == 0 && (reinterpret_cast<uintptr_t>(in) & 15) == 0;
  for (int64_t ty = ty0; ty < job.row_tiles; ty += step) {
    const int64_t r0 = ty * kTrRows;
    // 128 rows x 64 bytes: load i of thread t is row (t >> 2) + 64 i, bytes
    // 16 (t & 3) .. + 15
#pragma unroll
    for (int i = 0; i < kTrGroups; ++i) {
      const int row = (tid >> 2) + 64 * i, part = tid & 3;
      const int64_t r = r0 + row;
      const int64_t cb = cb0 + 16 * part;
      uint32_t w[4] = {0u, 0u, 0u, 0u};
      if (r < rows) {
        if (vec && cb + 16 <= in_pitch) {
          const uint4 q = *reinterpret_cast<const uint4*>(in + r * in_pitch + cb);
          w[0] = q.x, w[1] = q.y, w[2] = q.z, w[3] = q.w;
        } else {
#pragma unroll
          for (int k = 0; k < 16; ++k)
            if (cb + k < in_pitch) w[k >> 2] |= static_cast<uint32_t>(in[r * in_pitch + cb + k]) << (8 * (k & 3));
        }
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) *reinterpret_cast<uint32_t*>(&tile[row][16 * part + 4 * d]) = w[d];
    }
    __syncthreads();
    if ((tid >> 6) < kTrGroups) {
      // column byte cbl of 64-row group g
      const int cbl = tid & 63, g = tid >> 6;
      uint64_t col[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const int rb = 8 * g + b;  // row block: rows 8 rb .. 8 rb + 7
        uint64_t x = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) x |= static_cast<uint64_t>(tile[8 * rb + i][cbl]) << (8 * i);
        x = transpose_8x8(x);  // byte j: column 8 cbl + j over the block's 8 rows
#pragma unroll
        for (int j = 0; j < 8; ++j) col[j] |= ((x >> (8 * j)) & 0xFFull) << (8 * b);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) otile[8 * cbl + j][g] = col[j];
    }
    __syncthreads();
    // 512 columns x 16 bytes: store i of thread t is column t / 2 + 128 i,
    // bytes 8 (t % 2) .. + 7
#pragma unroll
    for (int i = 0; i < 2 * kTrGroups; ++i) {
      const int cl = tid / kTrGroups + (256 / kTrGroups) * i, piece = tid % kTrGroups;
      const int64_t c = 8 * cb0 + cl;
      const int64_t ob = r0 / 8 + 8 * piece;
      if (c < cols && ob < out_pitch) *reinterpret_cast<uint64_t*>(out + c * out_pitch + ob) = otile[cl][piece];
    }
    __syncthreads();  // the next row tile reuses tile and otile
  }
}

// fp32 -> the 16-bit operand dtype, zero from n to padded
struct ScaleJob {
  const float* in;
  uint16_t* out;
  int64_t n, padded;
};

template <int DT>
__device__ __forceinline__ void scale_to_16(const ScaleJob& job, int64_t i) {
  if (i < job.padded) job.out[i] = i < job.n ? (DT == QSTE_F16 ? f32_to_f16(job.in[i]) : f32_to_bf16(job.in[i])) : 0;
}

}  // namespace qste
