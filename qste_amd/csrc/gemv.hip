// Skinny forward (decode and small batches): y[m, n] = (sum_k x[m, k]
// sign[n, k]) * scale[n] + bias[n] for up to 64 rows of bf16 / fp16 x, or up
// to 21 rows of fp32 x as three bf16 limbs each (fallback.py:95-108; the
// small-batch path of the reference GPU backend, cuda.py:198-501).
//
// The weight bits (N * K / 8 bytes) are the only large operand and each bit
// is used for a few rows only, so what the kernel spends per bit decides its
// time.  Expanding bits to +-1 operands costs the VALU one instruction per
// pair of weights at best (the matrix cores then wait for it).  Here the
// bits never become operand values:
//
// * Weights as the sparsity indexes of v_smfmac_f32_16x16x64.  That
//   instruction multiplies a 4:2 sparse A (its nonzero values and a 2-bit
//   index per value that says which element of its group of four it is)
//   with a dense B.  B holds every x twice, negated and plain, as the pair
//   (-x[k], x[k]); the two nonzeros of a group pick one element of each of
//   its two pairs.  All of A's values are 1.0, and the index of a value is
//   its weight bit (plus 2 for the second pair of the group): bit set picks
//   x[k], clear picks -x[k].  So 16 consecutive even (or odd) bits of a
//   weight dword, masked and OR-ed with the constant second-pair bits, are
//   the index operand as they are: 3 VALU instructions turn 32 weights of a
//   lane into the operands of 4 MFMAs, against 20 for bit expansion.  The
//   products are exact (x or -x), the sums the MFMA's fp32 sums.
// * x fragments (pairs) are formed once per 32 columns from LDS and used for
//   NBW blocks of 16 weight rows.
//
// MFMA layout: lane l holds A row l%16, nonzeros e = 0..7 of logical k
// 16(l/16) + 2e, + 2e + 1; B column l%16, values i = 0..7 at logical k
// 8(l/16) + i and i = 8..15 at 32 + 8(l/16) + i - 8; the accumulator's
// register j holds D[4(l/16) + j][l%16].  D's rows are weight rows and its
// columns rows of x, so each lane ends with four consecutive outputs of one
// row of y.  A lane group g's index dword covers columns 128g + 32j + 0..31
// of a 512-column chunk (j: which of its four dwords): the even bits are two
// MFMAs (the low half, then the high half of the index register), the odd
// bits two more.
//
// Work split: a workgroup of 8 waves owns 16 * NBW weight rows over one of
// `splits` ranges of K; its waves take the range's 512-column chunks in
// turn, each wave with x rows of its own in LDS (no barrier until the end),
// and the 8 partial accumulators are summed through LDS in wave order.  With
// splits > 1 the range sums go to a caller workspace and a second kernel adds
// them in range order: every workgroup reads all of x's rows over its range,
// so at many rows of x and few rows of weights x's traffic from L2 is what
// splitting K saves.
#include <type_traits>

#include "common.hpp"

namespace qste {
namespace gemv {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x8 __attribute__((ext_vector_type(8)));

constexpr int WAVES = 8;
constexpr int THREADS = 64 * WAVES;
constexpr int CHUNK_K = 512;  // columns per wave chunk (4 lane groups x 128)
constexpr uint32_t kRsrcWord3 = 0x00020000u;
constexpr uint32_t kOob = 0x80000000u;  // an offset past every buffer: reads zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
  const uint32_t n = bytes > 0x7FFFFFFFll ? 0x7FFFFFFFu : static_cast<uint32_t>(bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(n), kRsrcWord3);
}

__device__ __forceinline__ u32x4 ld128(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off), 0, 0));
}

// Per 16-bit type: the pair of ones and the sparse MFMA (H: which half of the
// index register).
template <int DT>
struct Op;

template <>
struct Op<QSTE_BF16> {
  static constexpr uint32_t ones = 0x3F803F80u;
  template <int H>
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x8 b, f32x4 c, uint32_t index) {
    return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                     __builtin_bit_cast(bf16x16_t, b), c, static_cast<int>(index), 0,
                                                     H);
  }
};

template <>
struct Op<QSTE_F16> {
  static constexpr uint32_t ones = 0x3C003C00u;
  template <int H>
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x8 b, f32x4 c, uint32_t index) {
    return __builtin_amdgcn_smfmac_f32_16x16x64_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x16_t, b),
                                                    c, static_cast<int>(index), 0, H);
  }
};

typedef __attribute__((address_space(3))) void lds_t;

// Wait until at most N of this wave's vector-memory loads are in flight.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  // s_waitcnt fields: vmcnt [3:0] and [15:14], expcnt [6:4] (7: none), lgkmcnt [11:8] (15: none)
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (((N >> 4) & 3) << 14) | 0xF70);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// What a launch is given besides the operands.
struct Args {
  const uint16_t* x;    // [xr, K] 16-bit rows (fp32: three limb rows per row)
  const uint8_t* bits;  // [N, K / 8]
  const float* scale;
  const float* bias;    // may be null
  void* y;              // [xr / limbs, N] (16-bit, or fp32 with limbs)
  float* partial;       // splits > 1: [splits][xr][N]
  const int* top;       // fp32: the largest exponent of each row of x (its limbs carry a power of two)
  int xr;               // rows of x
  int limbs;            // 1, or 3 (y in fp32, row m = rows 3m .. 3m + 2 of x)
  int splits;
  int chunks_per_split;
  int64_t N, K;
};

// Four outputs n .. n + 3 of row m from their sums.
template <int OUT>
__device__ __forceinline__ void finish4(const Args& p, int64_t m, int64_t n, f32x4 v, const float* sc,
                                        const float* bi, bool vec) {
  float r[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r[j] = v[j] * sc[j];
    r[j] = r[j] + bi[j];
  }
  const int64_t at = m * p.N + n;
  if constexpr (OUT == QSTE_F32) {
    float* y = static_cast<float*>(p.y);
    if (vec) {
      *reinterpret_cast<float4*>(y + at) = make_float4(r[0], r[1], r[2], r[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < p.N) y[at + j] = r[j];
    }
  } else {
    uint16_t* y = static_cast<uint16_t*>(p.y);
    uint16_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = OUT == QSTE_F16 ? f32_to_f16(r[j]) : f32_to_bf16(r[j]);
    if (vec) {
      *reinterpret_cast<uint2*>(y + at) = make_uint2(h[0] | (static_cast<uint32_t>(h[1]) << 16),
                                                     h[2] | (static_cast<uint32_t>(h[3]) << 16));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < p.N) y[at + j] = h[j];
    }
  }
}

// XR rows of x are staged (>= p.xr: 4 or a multiple of 16; rows past p.xr
// are left as they are, their outputs are never stored), NBW blocks of 16
// weight rows per workgroup.  STAGED: x arrives in four stages a chunk, as it
// has to past 16 rows; up to 16 rows that is for fp32, whose rows then share
// one order of sums whatever their number.
template <int XR, int NBW, bool STAGED>
struct Cfg {
  static_assert(STAGED || XR <= 16, "whole chunks of more rows do not fit");
  // A chunk's fragments of one tile of x are all formed first and the blocks
  // streamed past them: pays from three blocks on (28672 x 8192, M = 1: 10.3
  // against 12.7 us; 4096 x 4096, one block: 3.9 both ways; 4096 x 14336: 7.7
  // against 7.2)
  static constexpr bool RESIDENT = !STAGED && NBW >= 3;
  static constexpr int MT = (XR + 15) / 16;                     // MFMA columns / 16
  static constexpr int STAGES = STAGED ? 4 : 1;                 // x stages per chunk
  static constexpr int JS = 4 / STAGES;
  // one stage: whole chunks of a row (1 KB and a pad: the 16 rows of a
  // fragment read cover all banks), or 256 bytes of a row (16-byte piece i of
  // row r at slot i ^ (r % 16))
  static constexpr int PITCH = STAGES == 1 ? 1040 : 256;
  // chunks of x in LDS at a time: below 16 rows there is room for two, which
  // takes x's latency out of a wave's chain of chunks
  static constexpr int XBUF = XR < 16 && !RESIDENT ? 2 : 1;
  static constexpr int x_bytes = XBUF * XR * PITCH;             // per wave
  static constexpr int red_bytes = WAVES * NBW * MT * 64 * 16;
  static constexpr int bytes = WAVES * x_bytes > red_bytes ? WAVES * x_bytes : red_bytes;
  // weight loads in flight: a chunk's, or two where blocks are streamed (the
  // CUs' streams stay interleaved; 4 in flight: 4-6% slower at M = 1)
  static constexpr int D = RESIDENT ? 2 : NBW;
};

template <int DT, int XR, int NBW, bool STAGED>
__global__ __launch_bounds__(THREADS, 1) void skinny_kernel(Args p) {
  using C = Cfg<XR, NBW, STAGED>;
  constexpr int MT = C::MT, JS = C::JS, D = C::D;
  __shared__ __attribute__((aligned(16))) uint8_t smem[C::bytes];
  __shared__ float epi[2][16 * NBW];
  constexpr bool kLimbs = DT == QSTE_BF16 && STAGED;  // what fp32 rows run on
  __shared__ int back[kLimbs ? XR / 3 : 1];           // fp32: the power of two to undo, per row of y
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l16 = lane & 15, q = lane >> 4;
  const int64_t K = p.K, pb = K / 8;
  // consecutive workgroups land on different XCDs: with the range as the
  // fastest index, an XCD's workgroups read few ranges of x
  const int range = static_cast<int>(blockIdx.x) % p.splits;
  const int64_t n0 = static_cast<int64_t>(static_cast<int>(blockIdx.x) / p.splits) * (16 * NBW);
  const int c_first = range * p.chunks_per_split;
  const int c_all = static_cast<int>((K + CHUNK_K - 1) / CHUNK_K);
  const int c_last = min(c_first + p.chunks_per_split, c_all);

  // rows past N read zero through the buffer bounds
  const __amdgpu_buffer_rsrc_t rb = rsrc(p.bits, p.N * pb);
  const __amdgpu_buffer_rsrc_t rx = rsrc(p.x, static_cast<int64_t>(p.xr) * K * 2);
  uint32_t boff[NBW];
#pragma unroll
  for (int b = 0; b < NBW; ++b) boff[b] = static_cast<uint32_t>((n0 + 16 * b + l16) * pb + 16 * q);

  uint8_t* xs = smem + wave * C::x_bytes;
  auto issue_x = [&](int c, int stage, int buf = 0) {
    // columns past K (a last chunk that K ends inside) read zero
    if constexpr (C::STAGES == 1) {
      const uint32_t off =
          c < c_last && CHUNK_K * c + 8 * lane < K ? 1024u * static_cast<uint32_t>(c) + 16u * lane : kOob;
      auto row = [&](int r, uint32_t at) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_t*)(xs + (buf * XR + r) * C::PITCH), 16,
                                                 static_cast<int>(at), static_cast<int>(r * K * 2), 0, 0);
      };
      if constexpr (C::XBUF > 1) {  // always XR loads: the waits below count them
#pragma unroll
        for (int r = 0; r < XR; ++r) row(r, r < p.xr ? off : kOob);
      } else {
        for (int r = 0; r < p.xr; ++r) row(r, off);
      }
    } else {
      const int col = CHUNK_K * c + 128 * stage;
#pragma unroll
      for (int r = 0; r < XR; r += 4) {
        if (r >= p.xr) break;
        const int row = r + (lane >> 4), piece = (lane & 15) ^ (row & 15);
        const uint32_t off = col + 8 * piece < K ? static_cast<uint32_t>((lane >> 4) * K * 2 + 16 * piece) : kOob;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_t*)(xs + r * C::PITCH), 16, static_cast<int>(off),
                                                 static_cast<int>(r * K * 2 + 2 * static_cast<int64_t>(col)), 0, 0);
      }
    }
  };
  // The weights of a lane group g cover columns 128g + 32j of the chunk with
  // dword j where a stage holds whole chunks, and 128j + 32g (the 4 x 4
  // transpose of groups and dwords, by_stage below) where stage j holds
  // columns 128j .. + 127.  This lane's x of dword j, tile mt, half-dword H
  // and logical k half h: 8 columns at 16H + 8(q%2) of the 32 columns of
  // group 2h + q/2.
  auto read_x = [&](int j, int mt, int H, int h, int buf = 0) {
    const int g = 2 * h + (q >> 1);
    if constexpr (C::STAGES == 1) {
      const int row = buf * XR + (XR >= 16 ? l16 : l16 % XR);
      return *reinterpret_cast<const u32x4*>(xs + row * C::PITCH + 256 * g + 64 * j + 32 * H + 16 * (q & 1));
    } else {
      const int row = 16 * mt + l16, piece = (4 * g + 2 * H + (q & 1)) ^ l16;
      return *reinterpret_cast<const u32x4*>(xs + row * C::PITCH + 16 * piece);
    }
  };
  auto by_stage = [&](u32x4 w) {
    if constexpr (C::STAGES == 1) return w;
    const auto a = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
    const auto e = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
    const auto o = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    return u32x4{e[0], o[0], e[1], o[1]};
  };

  u32x4 W[NBW];
  auto issue_w1 = [&](int c, int b) { return ld128(rb, c < c_last ? boff[b] + 64u * static_cast<uint32_t>(c) : kOob); };

  f32x4 acc[NBW][MT];
#pragma unroll
  for (int b = 0; b < NBW; ++b)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[b][mt] = f32x4{};
  const u32x4 ones = {Op<DT>::ones, Op<DT>::ones, Op<DT>::ones, Op<DT>::ones};
  auto pairs = [&](uint32_t v, int odd) {  // (-x, x) of the even or the odd one of two columns
    return __builtin_amdgcn_perm(v, v ^ 0x80008000u, odd ? 0x07060302u : 0x05040100u);
  };
  auto even_index = [](uint32_t w) { return (w & 0x55555555u) | 0x88888888u; };
  auto odd_index = [](uint32_t w) { return ((w >> 1) & 0x55555555u) | 0x88888888u; };

  int c = c_first + wave;
  if (c < c_last) {
    issue_x(c, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < D; ++b) W[b] = issue_w1(c, b);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (C::XBUF > 1) issue_x(c + WAVES, 0, 1);
    __builtin_amdgcn_sched_barrier(0);
  }
  // the epilogue's row scale, bias and powers of two, fetched while the first loads fly
  float out_scale = 0.0f, out_bias = 0.0f;
  if (tid < 16 * NBW && n0 + tid < p.N) {
    out_scale = p.scale[n0 + tid];
    out_bias = p.bias ? p.bias[n0 + tid] : 0.0f;
  }
  int out_top = 0;
  if (kLimbs && p.limbs == 3 && tid < p.xr / 3) out_top = p.top[tid];
  if constexpr (C::RESIDENT) {
    for (; c < c_last; c += WAVES) {
      wait_vm<D>();  // all but the newest loads, the weights in flight: x is in LDS
      u32x8 f[4][2][2];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int H = 0; H < 2; ++H) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const u32x4 v = read_x(j, 0, H, h);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int o = 0; o < 2; ++o) f[j][H][o][4 * h + i] = pairs(v[i], o);
          }
          asm volatile("" : "+v"(f[j][H][0]), "+v"(f[j][H][1]));
        }
      // the x rows are in registers from here on: the next chunk's may land
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
      if (c + WAVES < c_last) issue_x(c + WAVES, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < NBW; ++b) {
        const u32x4 w = W[b];
        // the load D blocks ahead
        if (b + D < NBW) W[b + D] = issue_w1(c, b + D);
        else W[b + D - NBW] = issue_w1(c + WAVES, b + D - NBW);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t e = even_index(w[j]), o = odd_index(w[j]);
          acc[b][0] = Op<DT>::template mma<0>(ones, f[j][0][0], acc[b][0], e);
          acc[b][0] = Op<DT>::template mma<0>(ones, f[j][0][1], acc[b][0], o);
          acc[b][0] = Op<DT>::template mma<1>(ones, f[j][1][0], acc[b][0], e);
          acc[b][0] = Op<DT>::template mma<1>(ones, f[j][1][1], acc[b][0], o);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    u32x4 Wn[NBW];
    for (int buf = 0; c < c_last; c += WAVES, buf ^= C::XBUF - 1) {
      const int cn = c + WAVES;
      if constexpr (C::STAGES > 1) {
        wait_vm<0>();
#pragma unroll
        for (int b = 0; b < NBW; ++b) W[b] = by_stage(W[b]);
      }
#pragma unroll
      for (int st = 0; st < C::STAGES; ++st) {
        // the next chunk's weights go out behind this chunk's last x stage
        // (loads complete in order: x must not wait for weights not needed yet)
        if (st == C::STAGES - 1) {
#pragma unroll
          for (int b = 0; b < NBW; ++b) Wn[b] = issue_w1(cn, b);
          // all but the loads just issued (and the x of the chunk after
          // this one, issued before them): the stage is in LDS
          wait_vm<NBW + (C::XBUF - 1) * XR>();
        } else {
          wait_vm<0>();
        }
#pragma unroll
        for (int jj = 0; jj < JS; ++jj) {
          const int j = JS * st + jj;
          u32x4 raw[MT][2][2];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int H = 0; H < 2; ++H)
#pragma unroll
              for (int h = 0; h < 2; ++h) raw[mt][H][h] = read_x(j, mt, H, h, buf);
          if (jj == JS - 1) {
            // the stage is in registers from here on: the next one's direct
            // loads may overwrite it
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int H = 0; H < 2; ++H)
#pragma unroll
                for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(raw[mt][H][h]));
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            __builtin_amdgcn_sched_barrier(0);
            if (st + 1 < C::STAGES) issue_x(c, st + 1);
            else if (C::XBUF > 1) issue_x(cn + WAVES, 0, buf);
            else if (cn < c_last) issue_x(cn, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
          uint32_t index[NBW][2];
#pragma unroll
          for (int b = 0; b < NBW; ++b) {
            index[b][0] = even_index(W[b][j]);
            index[b][1] = odd_index(W[b][j]);
          }
          auto half = [&](auto half_index) {
            constexpr int H = decltype(half_index)::value;
            u32x8 f[MT][2];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int o = 0; o < 2; ++o) f[mt][o][i] = pairs(raw[mt][H][i >> 2][i & 3], o);
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
              for (int b = 0; b < NBW; ++b)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                  acc[b][mt] = Op<DT>::template mma<H>(ones, f[mt][o], acc[b][mt], index[b][o]);
          };
          half(std::integral_constant<int, 0>{});
          half(std::integral_constant<int, 1>{});
        }
      }
#pragma unroll
      for (int b = 0; b < NBW; ++b) W[b] = Wn[b];
    }
  }

  // partial sums of the 8 waves, added in wave order, in the LDS the x rows
  // were staged in: two chunks in LDS leave loads past the last chunk in
  // flight (they land as zeros), and the barrier alone does not wait for them
  if constexpr (C::XBUF > 1) wait_vm<0>();
  if (tid < 16 * NBW) {
    epi[0][tid] = out_scale;
    epi[1][tid] = out_bias;
  }
  if (kLimbs && p.limbs == 3 && tid < p.xr / 3) back[tid] = -limb_shift(out_top);
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [WAVES][NBW * MT][64]
#pragma unroll
  for (int b = 0; b < NBW; ++b)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * NBW * MT + b * MT + mt) * 64 + lane] = acc[b][mt];
  __syncthreads();
  auto total = [&](int b, int row, int g) {  // x row `row`, weight rows 16b + 4g + 0..3
    const int at = (b * MT + (row >> 4)) * 64 + 16 * g + (row & 15);
    f32x4 v = red[at];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += red[w * NBW * MT * 64 + at];
    return v;
  };
  const bool full = (p.N & 3) == 0;
  if (p.splits > 1) {
    float* part = p.partial + static_cast<int64_t>(range) * p.xr * p.N;
    for (int i = tid; i < NBW * p.xr * 4; i += THREADS) {
      const int g = i & 3, b = (i >> 2) % NBW, row = (i >> 2) / NBW;
      const int64_t n = n0 + 16 * b + 4 * g;
      if (n >= p.N) continue;
      const f32x4 v = total(b, row, g);
      float* d = part + static_cast<int64_t>(row) * p.N + n;
      if (full) {
        *reinterpret_cast<f32x4*>(d) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < p.N) d[j] = v[j];
      }
    }
    return;
  }
  const int rows = p.xr / p.limbs;
  const int align = p.limbs == 3 ? 15 : 7;
  const bool vec = full && (reinterpret_cast<uintptr_t>(p.y) & align) == 0;
  for (int i = tid; i < NBW * rows * 4; i += THREADS) {
    const int g = i & 3, b = (i >> 2) % NBW, m = (i >> 2) / NBW;
    const int64_t n = n0 + 16 * b + 4 * g;
    if (n >= p.N) continue;
    const float* sc = &epi[0][16 * b + 4 * g];
    const float* bi = &epi[1][16 * b + 4 * g];
    if constexpr (kLimbs) {
      if (p.limbs == 3) {
        f32x4 v = (total(b, 3 * m + 2, g) + total(b, 3 * m + 1, g)) + total(b, 3 * m, g);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ldexpf(v[j], back[m]);
        finish4<QSTE_F32>(p, m, n, v, sc, bi, vec);
        continue;
      }
    }
    finish4<DT>(p, m, n, total(b, m, g), sc, bi, vec);
  }
}

// splits > 1 (16-bit x): the range sums added in range order, then scale, bias
// and one rounding; four outputs a thread.
template <int DT>
__global__ __launch_bounds__(256) void combine_kernel(Args p) {
  const int64_t quads = (p.N + 3) / 4;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= p.xr * quads) return;
  const int64_t m = i / quads, n = 4 * (i - m * quads);
  const bool full = (p.N & 3) == 0;
  float sc[4], bi[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sc[j] = n + j < p.N ? p.scale[n + j] : 0.0f;
    bi[j] = n + j < p.N && p.bias ? p.bias[n + j] : 0.0f;
  }
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s = 0; s < p.splits; ++s) {
    const float* d = p.partial + (static_cast<int64_t>(s) * p.xr + m) * p.N + n;
    if (full) {
      v += *reinterpret_cast<const f32x4*>(d);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < p.N) v[j] += d[j];
    }
  }
  const bool vec = full && (reinterpret_cast<uintptr_t>(p.y) & 7) == 0;
  finish4<DT>(p, m, n, v, sc, bi, vec);
}

// Weight blocks per workgroup at most: what the waves' accumulators and their
// image in LDS at the end have room for.
constexpr int most_blocks(int xr) { return xr <= 32 ? 8 : (xr <= 48 ? 6 : 4); }

template <int DT, int XR, bool STAGED, int NBW = 1>
void launch_nbw(int nbw, const Args& p, hipStream_t stream) {
  if constexpr (NBW < most_blocks(XR)) {
    if (nbw > NBW) return launch_nbw<DT, XR, STAGED, NBW + 1>(nbw, p, stream);
  }
  const int groups = static_cast<int>((p.N + 16 * NBW - 1) / (16 * NBW));
  skinny_kernel<DT, XR, NBW, STAGED><<<groups * p.splits, THREADS, 0, stream>>>(p);
}

template <int DT>
void launch_xr(int nbw, const Args& p, hipStream_t stream) {
  if constexpr (DT == QSTE_BF16) {
    if (p.limbs == 3 && p.xr <= 16) return launch_nbw<DT, 16, true>(nbw, p, stream);
  }
  if (p.xr <= 4) launch_nbw<DT, 4, false>(nbw, p, stream);
  else if (p.xr <= 16) launch_nbw<DT, 16, false>(nbw, p, stream);
  else if (p.xr <= 32) launch_nbw<DT, 32, true>(nbw, p, stream);
  else if (p.xr <= 48) launch_nbw<DT, 48, true>(nbw, p, stream);
  else launch_nbw<DT, 64, true>(nbw, p, stream);
}

// Rows of x a launch takes: four tiles of 16, or 21 rows of three limbs.
constexpr int64_t kRows16 = 64, kRows32 = 21;

// Blocks of weights a plan that splits K has at most (two per CU).
constexpr int64_t kSplitBlocks = 2 * 256;

struct Plan {
  int nbw, splits, chunks_per_split;
};

// Weight blocks per workgroup and ranges of K for xr rows of x.
//
// Blocks: the workgroups of one round over the 256 CUs as even as the most
// blocks a workgroup can hold allows.  Ranges: with 1 to 2 blocks per
// workgroup, forming fragments from x (0.087 us per chunk and tile of 16
// rows: 192 VALU instructions) and x's reads from L2 (0.0085 us per chunk and
// row) bound the kernel, not the weights; S ranges cut both S-fold, and cost
// a second launch and the sums' round trip, a little more for more ranges.
// Measured, one range against the best split: 8192 x 28672, M = 40: 40.6 / 31.9
// us; 4096 x 14336, M = 24: 14.4 / 13.0; three
// blocks and more (14336 x 4096, M = 40: 11.8 / 20.8) are never split.
//
// A row's sums are in an order of its own K alone, not of how many other rows
// the call brings: up to 16 rows are never cut (8192 x 28672, M = 16: 14.5 us cut in
// two, 16.1 whole), nor are fp32 rows, and past 16 the line is drawn for the
// instance's last row (32, 48, 64), so only those steps change a row's bits.
Plan plan_of(int64_t xr, int64_t rows, int64_t cols, bool may_split) {
  const int64_t blocks = (rows + 15) / 16, chunks = (cols + CHUNK_K - 1) / CHUNK_K;
  const int64_t most = most_blocks(static_cast<int>(xr)), tiles = (xr + 15) / 16;
  int64_t splits = 1, per = chunks;
  if (may_split && xr > 16 && blocks <= kSplitBlocks) {
    double best = 0.0;
    for (int64_t s = 2; s <= 4 && 2 * s <= chunks; s *= 2) {
      const int64_t cps = (chunks + s - 1) / s, ns = (chunks + cps - 1) / cps;
      if ((blocks * ns + 255) / 256 > most) continue;  // a second round
      const double saved = static_cast<double>(chunks - cps) * tiles * (0.087 + 16 * 0.0085);
      const double cost = 4.5 + 1.3 * static_cast<double>(ns - 2) + static_cast<double>(ns * 16 * tiles * rows) * 8.0 / 4e6;
      if (saved - cost > best) {
        best = saved - cost;
        splits = ns;
        per = cps;
      }
    }
  }
  const int64_t work = blocks * splits, rounds = (work + 256 * most - 1) / (256 * most);
  int64_t nbw = (work + 256 * rounds - 1) / (256 * rounds);
  return Plan{static_cast<int>(nbw < 1 ? 1 : nbw), static_cast<int>(splits), static_cast<int>(per)};
}

// Time of a call in us with xr rows of x, fitted to 1000 measured products (300
// to 128256 rows of weights over 128 to 28672 columns): 90% of the times are
// within 13% of it.  A round of workgroups takes a fixed time, the sums and
// outputs of its blocks (first two terms), and per chunk x's reads, the MFMAs
// and a wave's chain.
double estimate(int64_t xr, const Plan& plan, int64_t rows, bool staged) {
  struct Rates {
    double call, round, block, read, mma, chain;
  };
  const Rates t = staged ? Rates{1.6, 0.87, 0.317, 0.0055, 0.0255, 1.42} : Rates{1.4, 1.16, 0.172, 0.0064, 0.007, 0.84};
  const double tiles = static_cast<double>((xr + 15) / 16), per = static_cast<double>(plan.chunks_per_split);
  const int64_t groups = (rows + 16 * plan.nbw - 1) / (16 * plan.nbw) * plan.splits;
  const double combine = plan.splits > 1 ? 3.0 + static_cast<double>(plan.splits * xr * rows) * 8.0 / 3.3e6 : 0.0;
  return t.call + combine +
         static_cast<double>((groups + 255) / 256) *
             (t.round + plan.nbw * tiles * (t.block + t.mma * per) + t.read * per * static_cast<double>(xr) +
              t.chain * static_cast<double>((plan.chunks_per_split + WAVES - 1) / WAVES));
}

// Rows of 16-bit x that m rows make (three limbs for an fp32 row), 0 when
// the product is not for this path.
int64_t x_rows(int dtype, int64_t m, int64_t rows, int64_t cols) {
  const int64_t most = dtype == QSTE_F32 ? kRows32 : kRows16;
  if (m < 1 || m > most || rows < 1 || cols < 128 || cols % 128 != 0) return 0;
  const int64_t xr = dtype == QSTE_F32 ? 3 * m : m;
  // 32-bit buffer offsets, with room for the padded last block and the
  // out-of-range marker
  return (rows + 128) * (cols / 8) < (int64_t{1} << 31) && xr * cols * 2 < (int64_t{1} << 31) ? xr : 0;
}

template <int DT>
int run(const Args& p, const Plan& plan, hipStream_t stream) {
  launch_xr<DT>(plan.nbw, p, stream);
  int rc = static_cast<int>(hipGetLastError());
  if (rc || p.splits == 1) return rc;
  const int64_t items = p.xr * ((p.N + 3) / 4);
  combine_kernel<DT><<<static_cast<int>((items + 255) / 256), 256, 0, stream>>>(p);
  return static_cast<int>(hipGetLastError());
}

size_t up256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }

}  // namespace gemv

int launch_limbs(const float*, int64_t, int64_t, uint16_t*, int*, hipStream_t);

// Time of a product on this path in us, negative when its sizes are not for it.
// It is the time of the instance's last row (16, 32, 48 or 64; 21 in fp32): a
// choice made by it does not change with the rows a call brings along.
double gemv_forward_us(int64_t m, int64_t rows, int64_t cols, int dtype) {
  const int64_t xr = gemv::x_rows(dtype, m, rows, cols);
  if (xr == 0) return -1.0;
  const bool fp32 = dtype == QSTE_F32;
  const int64_t top = fp32 ? 3 * gemv::kRows32 : (xr + 15) / 16 * 16;
  // (fp32: the limbs of x are a launch of their own)
  return gemv::estimate(top, gemv::plan_of(top, rows, cols, !fp32), rows, fp32 || top > 16) + (fp32 ? 2.7 : 0.0);
}

// Workspace of a product on this path: fp32 x's limbs and their exponents, or the range sums of
// the plan (past 16 rows two ranges wherever the blocks are few enough for any
// plan to split, so that the size does not depend on where the plan's line
// lies); 0 where none is needed or the product is not for this path.
size_t gemv_forward_workspace(int64_t m, int64_t rows, int64_t cols, int dtype) {
  const int64_t xr = gemv::x_rows(dtype, m, rows, cols);
  if (xr == 0) return 0;
  const bool fp32 = dtype == QSTE_F32;
  const gemv::Plan plan = gemv::plan_of(xr, rows, cols, !fp32);
  int64_t ranges = plan.splits > 1 ? plan.splits : 0;
  if (!fp32 && m > 16 && ranges < 2 && (rows + 15) / 16 <= gemv::kSplitBlocks) ranges = 2;
  return (fp32 ? gemv::up256(static_cast<size_t>(xr * cols) * 2) + gemv::up256(static_cast<size_t>(m) * sizeof(int)) : 0) +
         static_cast<size_t>(ranges * xr * rows) * sizeof(float);
}

// Returns 1 when the call is not for this path (fp32 needs its workspace; 16
// bit runs in one range without one).
int gemv_linear_forward(const void* x, int dtype, const uint8_t* packed, const float* scale, const float* bias,
                        void* y, int64_t m, int64_t rows, int64_t cols, void* workspace, size_t workspace_bytes,
                        hipStream_t stream) {
  const int64_t xr = gemv::x_rows(dtype, m, rows, cols);
  const bool fp32 = dtype == QSTE_F32;
  if (xr == 0 || (reinterpret_cast<uintptr_t>(x) & 15) ||
      (reinterpret_cast<uintptr_t>(packed) & 15))
    return 1;
  const bool room = workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 &&
                    workspace_bytes >= gemv_forward_workspace(m, rows, cols, dtype);
  if (fp32 && !room) return 1;
  const gemv::Plan plan = gemv::plan_of(xr, rows, cols, room && !fp32);
  gemv::Args p{};
  p.x = static_cast<const uint16_t*>(x);
  p.bits = packed;
  p.scale = scale;
  p.bias = bias;
  p.y = y;
  p.xr = static_cast<int>(xr);
  p.limbs = fp32 ? 3 : 1;
  p.splits = plan.splits;
  p.chunks_per_split = plan.chunks_per_split;
  p.N = rows;
  p.K = cols;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  if (fp32) {
    uint16_t* xl = reinterpret_cast<uint16_t*>(ws);
    int* top = reinterpret_cast<int*>(ws + gemv::up256(static_cast<size_t>(p.xr * cols) * 2));
    const int rc = launch_limbs(static_cast<const float*>(x), m, cols, xl, top, stream);
    if (rc) return rc;
    p.x = xl;
    p.top = top;
  }
  p.partial = reinterpret_cast<float*>(ws);
  return dtype == QSTE_F16 ? gemv::run<QSTE_F16>(p, plan, stream) : gemv::run<QSTE_BF16>(p, plan, stream);
}

}  // namespace qste
