// Row and column reductions of the backward pass.
//
//   row_inner   gs[r] = sum_c E[r, c] * sign[r, c]   (fallback.py:141-148)
//   colsums     v[r]  = sum_t dy[t, r] * offset[t]   (functional.py:139-144)
//               db[r] = sum_t dy[t, r]               (functional.py:193)
//
// Column sums run in two deterministic stages (chunk partials, then a fixed
// order sum) so results do not depend on scheduling; nothing uses atomics.
#include "common.hpp"
#include "prep.hpp"

namespace qste {

constexpr int kRowThreads = 256;
constexpr int kColChunk = 256;

__global__ __launch_bounds__(kRowThreads) void row_inner_kernel(const float* __restrict__ mat,
                                                                const uint8_t* __restrict__ packed,
                                                                float* __restrict__ out,
                                                                int64_t cols, int64_t stride) {
  __shared__ float red[kRowThreads / kWave];
  const int64_t r = blockIdx.x;
  const float* row = mat + r * cols;
  const uint8_t* bits = packed + r * stride;
  float acc = 0.0f;
  for (int64_t c = threadIdx.x; c < cols; c += kRowThreads) acc += row[c] * sign_of(bits, c);
  acc = block_sum(acc, red);
  if (threadIdx.x == 0) out[r] = acc;
}

// Sum of `parts` partial vectors [parts][n] into out[n], in order of p (the
// loads are issued 32 at a time, so a few rounds of memory latency cover
// the usual 16-64 parts; the additions stay sequential).
// Parts are `pitch` >= n apart.  Workgroups with blockIdx.y == 1 sum a second
// set of vectors (a bias gradient's beside the offset correction's): the
// launch, at 3.4 us, costs more than either sum.
__global__ void sum_partials_kernel(const float* __restrict__ partial0, int64_t parts, int64_t n, int64_t pitch,
                                    float* __restrict__ out0, const float* __restrict__ partial1,
                                    float* __restrict__ out1) {
  constexpr int kBatch = 32;
  const float* const partial = blockIdx.y ? partial1 : partial0;
  float* const out = blockIdx.y ? out1 : out0;
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i >= n) return;
  float s = 0.0f;
  int64_t p = 0;
  for (; p + kBatch <= parts; p += kBatch) {
    float v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) v[u] = partial[(p + u) * pitch + i];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) s += v[u];
  }
  for (; p + 8 <= parts; p += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = partial[(p + u) * pitch + i];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; p < parts; ++p) s += partial[p * pitch + i];
  out[i] = s;
}

template <int DT>
__global__ void colsum_partial_kernel(const typename Elem<DT>::T* __restrict__ dy,
                                      const float* __restrict__ offset, int64_t samples,
                                      int64_t rows, float* __restrict__ v_part,
                                      float* __restrict__ db_part) {
  const int64_t r = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (r >= rows) return;
  const int64_t t0 = static_cast<int64_t>(blockIdx.y) * kColChunk;
  const int64_t t1 = t0 + kColChunk < samples ? t0 + kColChunk : samples;
  float v = 0.0f, db = 0.0f;
  for (int64_t t = t0; t < t1; ++t) {
    const float g = Elem<DT>::load(dy, t * rows + r);
    v = fmaf(g, offset[t], v);
    db += g;
  }
  v_part[blockIdx.y * rows + r] = v;
  if (db_part) db_part[blockIdx.y * rows + r] = db;
}

// rows a multiple of NV, dy aligned to NV elements: each lane reduces NV
// adjacent columns (one load of up to 16 bytes per sample), so a wave covers
// 64 NV of them.  The chunk's kColChunk samples are split over the
// workgroup's kColWaves waves (a contiguous quarter each, UNROLL loads in
// flight), and the waves' sums are added in wave order through LDS: a fixed
// order, whatever NV is, so the result depends neither on scheduling nor on
// the width chosen (colsum_narrow).  At 16384 x 14336 four waves per chunk keep
// ~28 waves resident per CU, where one per chunk left the loads latency-bound.
constexpr int kColWaves = 4;
constexpr int kColThreads = kColWaves * kWave;

template <int NV>
constexpr int kColPad = NV == 1 ? 2 : 2 * NV + 1;  // 2 NV sums per lane, padded against bank conflicts
template <int NV>
constexpr int kColLds = kColWaves * kWave * kColPad<NV>;

template <int BYTES> struct ColVec;
template <> struct ColVec<16> { using T = uint4; };
template <> struct ColVec<4> { using T = uint32_t; };

template <int DT, int NV>
__device__ __forceinline__ void colsum_block(const typename Elem<DT>::T* __restrict__ dy,
                                             const float* __restrict__ offset, int64_t samples, int64_t rows,
                                             float* __restrict__ v_part, float* __restrict__ db_part, int64_t bx,
                                             int64_t by, float* red) {
  using T = typename Elem<DT>::T;
  using V = typename ColVec<NV * sizeof(T)>::T;
  constexpr int UNROLL = sizeof(V) == 16 ? 8 : 32;
  constexpr int kPad = kColPad<NV>;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // offset[t] in scalar registers
  const int64_t base = bx * (kWave * NV);
  const int64_t r = base + lane * NV;
  const int64_t c0 = by * kColChunk;
  const int64_t c1 = c0 + kColChunk < samples ? c0 + kColChunk : samples;
  constexpr int kPer = kColChunk / kColWaves;
  const int64_t t0 = c0 + wave * kPer < c1 ? c0 + wave * kPer : c1;
  const int64_t t1 = t0 + kPer < c1 ? t0 + kPer : c1;
  float v[NV], db[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = db[i] = 0.0f;
  if (r < rows) {
    const T* col = dy + r;
    auto take = [&](const V& q, float o) {
      const T* e = reinterpret_cast<const T*>(&q);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const float g = Elem<DT>::load(e, i);
        v[i] = fmaf(g, o, v[i]);
        db[i] += g;
      }
    };
    int64_t t = t0;
    for (; t + UNROLL <= t1; t += UNROLL) {
      V q[UNROLL];
      float o[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        q[u] = *reinterpret_cast<const V*>(col + (t + u) * rows);
        o[u] = offset[t + u];
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) take(q[u], o[u]);
    }
    for (; t < t1; ++t) take(*reinterpret_cast<const V*>(col + t * rows), offset[t]);
  }
  float* mine = red + (wave * kWave + lane) * kPad;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    mine[i] = v[i];
    mine[NV + i] = db[i];
  }
  __syncthreads();
  // 2 * 64 NV results per workgroup (its columns of v, then of db),
  // consecutive threads on consecutive columns; waves summed in order
  // 0..kColWaves-1.
  const int64_t part = by * rows;
#pragma unroll
  for (int j = threadIdx.x; j < 2 * kWave * NV; j += kColThreads) {
    const int which = j / (kWave * NV);
    const int c = j % (kWave * NV);
    const int64_t rc = base + c;
    const int slot = (c / NV) * kPad + which * NV + c % NV;
    float s = red[slot];
#pragma unroll
    for (int w = 1; w < kColWaves; ++w) s += red[w * kWave * kPad + slot];
    if (rc < rows) {
      if (which == 0) v_part[part + rc] = s;
      else if (db_part) db_part[part + rc] = s;
    }
  }
}

template <int DT, int NV>
__global__ __launch_bounds__(kColThreads) void colsum_partial_vec_kernel(
    const typename Elem<DT>::T* __restrict__ dy, const float* __restrict__ offset, int64_t samples, int64_t rows,
    float* __restrict__ v_part, float* __restrict__ db_part) {
  __shared__ float red[kColLds<NV>];
  colsum_block<DT, NV>(dy, offset, samples, rows, v_part, db_part, blockIdx.x, blockIdx.y, red);
}

// Columns per lane: 16-byte loads, or 4-byte ones (as many bytes in flight per
// wave) over four times the workgroups where the wide ones leave CUs idle.
// A layer's backward, wide / narrow: 2048 x 4096 (64 wide workgroups) 153.7 /
// 149.9 us, 4096 x 4096 (128) 247.7 / 243.0, 8184 x 3072 (192) 102.8 / 104.7.
template <int DT>
constexpr int kColWide = 16 / sizeof(typename Elem<DT>::T);
template <int DT>
constexpr int kColNarrow = 4 / sizeof(typename Elem<DT>::T);

inline bool colsum_narrow(int64_t rows, int64_t chunks, int wide) {
  return (rows + kWave * wide - 1) / (kWave * wide) * chunks < 160;
}

// What a 16-bit layer's backward reads besides dy itself, made in one launch:
// the column sums' chunk partials, the transposed signs of x and W and the
// 16-bit scales.  As five launches they took 27 us at 8192 samples of
// 4096 x 1024, of which 12 read dy; their workgroups side by side take 15.
struct PrepParams {
  const uint16_t* dy;
  const float* offset;
  int64_t samples, rows;
  float *v_part, *db_part;
  TransposeJob sign[2];
  ScaleJob scale[2];
  int64_t col_x;      // column-sum workgroups: col_x by chunks
  int64_t ends[5];    // running ends of the roles' workgroup ranges
};

template <int DT, int NV>
__global__ __launch_bounds__(kColThreads) void backward_prep_kernel(PrepParams p) {
  __shared__ union {
    float red[kColLds<NV>];
    TransposeLds tr;
  } lds;
  int64_t b = blockIdx.x;
  if (b < p.ends[0]) {
    colsum_block<DT, NV>(p.dy, p.offset, p.samples, p.rows, p.v_part, p.db_part, b % p.col_x, b / p.col_x, lds.red);
  } else if (b < p.ends[2]) {
    const int which = b >= p.ends[1];
    const TransposeJob& job = p.sign[which];
    b -= p.ends[which];
    transpose_tiles(job, b / job.row_tiles, b % job.row_tiles, job.row_tiles, lds.tr);
  } else {
    const int which = b >= p.ends[3];
    scale_to_16<DT>(p.scale[which], (b - p.ends[2 + which]) * kColThreads + threadIdx.x);
  }
}

// The column sums of 16-bit rows of any length, which also leave as rows of
// `padded` columns (a multiple of 64), zero behind the data: the copy that
// the matrix products of a ragged layer read, made in the pass that reads the
// gradient anyway (2046 x 50257 bf16: 115 us for both, where the scalar sums
// alone took 151).  The sums are those of colsum_partial_vec_kernel over the
// padded rows, [chunks][padded].
template <int DT>
__global__ __launch_bounds__(kColThreads) void colsum_pad_kernel(
    const uint16_t* __restrict__ dy, const float* __restrict__ offset, int64_t samples, int64_t rows, int64_t padded,
    uint16_t* __restrict__ out, float* __restrict__ v_part, float* __restrict__ db_part) {
  struct __attribute__((packed)) Unaligned {
    uint32_t w[4];
  };
  constexpr int NV = 8, UNROLL = 4, kPad = 2 * NV + 1;
  __shared__ float red[kColWaves * kWave * kPad];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (kWave * NV);
  const int64_t r = base + lane * NV;
  const int64_t c0 = static_cast<int64_t>(blockIdx.y) * kColChunk;
  const int64_t c1 = c0 + kColChunk < samples ? c0 + kColChunk : samples;
  constexpr int kPer = kColChunk / kColWaves;
  const int64_t t0 = c0 + wave * kPer < c1 ? c0 + wave * kPer : c1;
  const int64_t t1 = t0 + kPer < c1 ? t0 + kPer : c1;
  float v[NV], db[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = db[i] = 0.0f;
  auto load = [&](int64_t t) {
    const uint16_t* src = dy + t * rows + r;
    Unaligned q{{0u, 0u, 0u, 0u}};
    if (r + NV <= rows) {
      q = *reinterpret_cast<const Unaligned*>(src);
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (r + i < rows) q.w[i >> 1] |= static_cast<uint32_t>(src[i]) << (16 * (i & 1));
    }
    return q;
  };
  auto take = [&](int64_t t, const Unaligned& q) {
    *reinterpret_cast<uint4*>(out + t * padded + r) = make_uint4(q.w[0], q.w[1], q.w[2], q.w[3]);
    const float o = offset[t];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const uint16_t h = static_cast<uint16_t>(q.w[i >> 1] >> (16 * (i & 1)));
      const float g = DT == QSTE_F16 ? f16_to_f32(h) : bf16_to_f32(h);
      v[i] = fmaf(g, o, v[i]);
      db[i] += g;
    }
  };
  if (r < padded) {
    int64_t t = t0;
    for (; t + UNROLL <= t1; t += UNROLL) {
      Unaligned q[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) q[u] = load(t + u);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) take(t + u, q[u]);
    }
    for (; t < t1; ++t) take(t, load(t));
  }
  float* mine = red + (wave * kWave + lane) * kPad;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    mine[i] = v[i];
    mine[NV + i] = db[i];
  }
  __syncthreads();
  const int64_t part = static_cast<int64_t>(blockIdx.y) * padded;
#pragma unroll
  for (int j = threadIdx.x; j < 2 * kWave * NV; j += kColThreads) {
    const int which = j / (kWave * NV), c = j % (kWave * NV);
    const int slot = (c / NV) * kPad + which * NV + c % NV;
    float s = red[slot];
#pragma unroll
    for (int w = 1; w < kColWaves; ++w) s += red[w * kWave * kPad + slot];
    if (base + c < padded) {
      if (which == 0) v_part[part + base + c] = s;
      else if (db_part) db_part[part + base + c] = s;
    }
  }
}

int launch_row_inner(const float* mat, const uint8_t* packed, float* out, int64_t rows,
                     int64_t cols, hipStream_t stream) {
  if (rows == 0) return 0;
  row_inner_kernel<<<rows, kRowThreads, 0, stream>>>(mat, packed, out, cols, (cols + 7) / 8);
  return static_cast<int>(hipGetLastError());
}

static int launch_sums(const float* partial0, const float* partial1, int64_t parts, int64_t n, int64_t pitch,
                       float* out0, float* out1, hipStream_t stream) {
  // one wave per workgroup: a few thousand outputs still spread over most CUs
  const dim3 grid(ceil_div(n, kWave), out1 ? 2 : 1);
  sum_partials_kernel<<<grid, kWave, 0, stream>>>(partial0, parts, n, pitch, out0, partial1, out1);
  return static_cast<int>(hipGetLastError());
}

int launch_sum_partials(const float* partial, int64_t parts, int64_t n, float* out,
                        hipStream_t stream) {
  if (n == 0) return 0;
  return launch_sums(partial, nullptr, parts, n, n, out, nullptr, stream);
}

int colsum_chunks(int64_t samples) { return ceil_div(samples, kColChunk); }

// v_part / db_part: [colsum_chunks(samples)][rows] floats each.
int launch_colsums(const void* dy, int dtype, const float* offset, int64_t samples, int64_t rows,
                   float* v_part, float* db_part, float* v_out, float* db_out,
                   hipStream_t stream) {
  if (rows == 0) return 0;
  const int chunks = colsum_chunks(samples);
  const int nv = dtype == QSTE_F32 ? 4 : 8;  // columns per 16-byte vector
  const bool vec = (dtype == QSTE_BF16 || dtype == QSTE_F16 || dtype == QSTE_F32) && rows % nv == 0 &&
                   (reinterpret_cast<uintptr_t>(dy) & 15) == 0;
  if (chunks > 0 && vec) {
    const bool narrow = colsum_narrow(rows, chunks, nv);
    const dim3 grid(ceil_div(rows, kWave * (narrow ? nv / 4 : nv)), chunks);
#define QSTE_COLSUM(DT)                                                                                      \
  (narrow ? colsum_partial_vec_kernel<DT, kColNarrow<DT>> : colsum_partial_vec_kernel<DT, kColWide<DT>>)     \
      <<<grid, kColThreads, 0, stream>>>(static_cast<const Elem<DT>::T*>(dy), offset, samples, rows, v_part, \
                                         db_part)
    if (dtype == QSTE_BF16) QSTE_COLSUM(QSTE_BF16);
    else if (dtype == QSTE_F16) QSTE_COLSUM(QSTE_F16);
    else QSTE_COLSUM(QSTE_F32);
#undef QSTE_COLSUM
    int rc = static_cast<int>(hipGetLastError());
    if (rc) return rc;
  } else if (chunks > 0) {
    dim3 grid(ceil_div(rows, 256), chunks);
    switch (dtype) {
      case QSTE_F32:
        colsum_partial_kernel<QSTE_F32><<<grid, 256, 0, stream>>>(
            static_cast<const float*>(dy), offset, samples, rows, v_part, db_part);
        break;
      case QSTE_F16:
        colsum_partial_kernel<QSTE_F16><<<grid, 256, 0, stream>>>(
            static_cast<const uint16_t*>(dy), offset, samples, rows, v_part, db_part);
        break;
      case QSTE_BF16:
        colsum_partial_kernel<QSTE_BF16><<<grid, 256, 0, stream>>>(
            static_cast<const uint16_t*>(dy), offset, samples, rows, v_part, db_part);
        break;
      default:
        return QSTE_E_DTYPE;
    }
    int rc = static_cast<int>(hipGetLastError());
    if (rc) return rc;
  }
  return launch_sums(v_part, db_part, chunks, rows, rows, v_out, db_out, stream);
}

// Column sums as launch_colsums (bf16 / fp16) and the zero-padded copy of dy;
// v_part / db_part: [colsum_chunks(samples)][padded] floats each.
int launch_colsums_pad(const void* dy, int dtype, const float* offset, int64_t samples, int64_t rows, int64_t padded,
                       uint16_t* out, float* v_part, float* db_part, float* v_out, float* db_out,
                       hipStream_t stream) {
  const int chunks = colsum_chunks(samples);
  if (rows == 0 || chunks == 0) return 0;
  const dim3 grid(ceil_div(padded, kWave * 8), chunks);
  if (dtype == QSTE_F16)
    colsum_pad_kernel<QSTE_F16><<<grid, kColThreads, 0, stream>>>(static_cast<const uint16_t*>(dy), offset, samples,
                                                                  rows, padded, out, v_part, db_part);
  else
    colsum_pad_kernel<QSTE_BF16><<<grid, kColThreads, 0, stream>>>(static_cast<const uint16_t*>(dy), offset, samples,
                                                                   rows, padded, out, v_part, db_part);
  return launch_sums(v_part, db_part, chunks, rows, padded, v_out, db_out, stream);
}

// The operands of a 16-bit layer's backward in one launch, and the column
// sums' chunks added in a second.  dy: rows of a multiple of 8 on 16-byte
// boundaries, or null where the sums are not needed.  w: the signs and
// scales of W, or an empty job (out null) where no input gradient is taken.
int launch_backward_prep(const void* dy, int dtype, const float* offset, int64_t samples, int64_t rows, float* v_part,
                         float* db_part, float* v_out, float* db_out, const TransposeJob& x, const ScaleJob& xs,
                         const TransposeJob& w, const ScaleJob& ws, hipStream_t stream) {
  if (dtype != QSTE_BF16 && dtype != QSTE_F16) return QSTE_E_DTYPE;
  const int chunks = dy ? colsum_chunks(samples) : 0;
  const bool narrow = colsum_narrow(rows, chunks, 8);
  PrepParams p{static_cast<const uint16_t*>(dy), offset, samples, rows, v_part, db_part, {x, w}, {xs, ws}, 0, {}};
  p.col_x = ceil_div(rows, kWave * (narrow ? 2 : 8));
  int64_t end = 0, i = 0;
  for (int64_t n : {p.col_x * chunks, x.col_tiles() * x.row_tiles, w.out ? w.col_tiles() * w.row_tiles : 0,
                    static_cast<int64_t>(ceil_div(xs.padded, kColThreads)),
                    w.out ? static_cast<int64_t>(ceil_div(ws.padded, kColThreads)) : 0})
    p.ends[i++] = end += n;
  const dim3 grid(static_cast<unsigned>(end));
  if (dtype == QSTE_BF16)
    (narrow ? backward_prep_kernel<QSTE_BF16, 2> : backward_prep_kernel<QSTE_BF16, 8>)<<<grid, kColThreads, 0, stream>>>(p);
  else
    (narrow ? backward_prep_kernel<QSTE_F16, 2> : backward_prep_kernel<QSTE_F16, 8>)<<<grid, kColThreads, 0, stream>>>(p);
  const int rc = static_cast<int>(hipGetLastError());
  if (rc || !chunks) return rc;
  return launch_sums(v_part, db_part, chunks, rows, rows, v_out, db_out, stream);
}

}  // namespace qste
