// The learned per-row scale of a binary layer and its gradient
// (src/qste/surface.py:84-85):
//
//   e = exp(log_scale),  s = clamp(e, lo, hi)
//   d log_scale = (lo <= e <= hi ? ds : 0) * e
//
// torch evaluates the forward as two launches (exp, clamp) and its autograd
// as six (a zero fill, two comparisons, their logical and, the where, the
// product with exp's result); here each direction is one launch over the
// rows.  Values are rounded as torch rounds them: exp is the device
// library's expf, the function torch's exp kernels call (for bf16 / fp16
// tensors on the fp32 value, rounded once to the dtype); clamp keeps a NaN
// and is min(max(e, lo), hi) otherwise, rounded to the dtype; the
// backward's comparisons are against the bounds rounded to the dtype, as
// torch compares a tensor with a Python float; its product is fp32, rounded
// to the dtype.  The forward also writes e, which the backward reads (torch's
// exp backward reads its saved result, not log_scale, so an in-place update
// of log_scale between forward and backward changes neither).
#include "common.hpp"

namespace qste {
namespace rowscale {

constexpr int kThreads = 256;

template <int DT>
__global__ __launch_bounds__(kThreads) void forward_kernel(const typename Elem<DT>::T* __restrict__ log_scale,
                                                           typename Elem<DT>::T* __restrict__ scale,
                                                           typename Elem<DT>::T* __restrict__ e_out, int64_t n,
                                                           float lo, float hi) {
  using E = Elem<DT>;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n) return;
  const float e = E::round(expf(E::load(log_scale, i)));
  E::store(e_out, i, e);
  E::store(scale, i, e != e ? e : fminf(fmaxf(e, lo), hi));
}

template <int DT>
__global__ __launch_bounds__(kThreads) void backward_kernel(const typename Elem<DT>::T* __restrict__ e_in,
                                                            const typename Elem<DT>::T* __restrict__ grad,
                                                            typename Elem<DT>::T* __restrict__ grad_log, int64_t n,
                                                            float lo, float hi) {
  using E = Elem<DT>;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n) return;
  const float e = E::load(e_in, i);
  // torch compares a tensor with a Python float in the tensor's dtype: the
  // bounds rounded to it
  const float pass = (e >= E::round(lo) && e <= E::round(hi)) ? E::load(grad, i) : 0.0f;
  E::store(grad_log, i, pass * e);
}

}  // namespace rowscale

#define QSTE_SCALE_DT_SWITCH(dtype, ...)                                  \
  switch (dtype) {                                                       \
    case QSTE_F32: { constexpr int DT = QSTE_F32; __VA_ARGS__; } break;  \
    case QSTE_F16: { constexpr int DT = QSTE_F16; __VA_ARGS__; } break;  \
    case QSTE_BF16: { constexpr int DT = QSTE_BF16; __VA_ARGS__; } break; \
    default: return QSTE_E_DTYPE;                                        \
  }

int launch_row_scale(const void* log_scale, int dtype, void* scale, void* e, int64_t n, float lo, float hi,
                     hipStream_t stream) {
  if (n == 0) return 0;
  QSTE_SCALE_DT_SWITCH(dtype, {
    using T = typename Elem<DT>::T;
    rowscale::forward_kernel<DT><<<ceil_div(n, rowscale::kThreads), rowscale::kThreads, 0, stream>>>(
        static_cast<const T*>(log_scale), static_cast<T*>(scale), static_cast<T*>(e), n, lo, hi);
  });
  return static_cast<int>(hipGetLastError());
}

int launch_row_scale_backward(const void* e, const void* grad, int dtype, void* grad_log, int64_t n, float lo,
                              float hi, hipStream_t stream) {
  if (n == 0) return 0;
  QSTE_SCALE_DT_SWITCH(dtype, {
    using T = typename Elem<DT>::T;
    rowscale::backward_kernel<DT><<<ceil_div(n, rowscale::kThreads), rowscale::kThreads, 0, stream>>>(
        static_cast<const T*>(e), static_cast<const T*>(grad), static_cast<T*>(grad_log), n, lo, hi);
  });
  return static_cast<int>(hipGetLastError());
}
#undef QSTE_SCALE_DT_SWITCH

// The end of an optimizer step in one launch: every surface's log-scales
// clamped in place (torch's clamp: NaN stays) and the surfaces' flip counts
// added up.  Bound by the launch: a clamp per surface, a stack and a sum took
// 10 launches for eight surfaces, 40 us of host time; this takes 6.
namespace finish {

constexpr int kMost = 64;  // surfaces per launch
constexpr int kThreads = 256;

struct Args {
  float* log_scale[kMost];
  int64_t n[kMost];
  const int64_t* flips[kMost];
  int64_t* total;
  float lo, hi;
  int nflips, first;
};

__global__ __launch_bounds__(kThreads) void finish_kernel(Args a) {
  float* const x = a.log_scale[blockIdx.y];
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x; i < a.n[blockIdx.y];
       i += static_cast<int64_t>(gridDim.x) * kThreads) {
    const float v = x[i];
    x[i] = v != v ? v : fminf(fmaxf(v, a.lo), a.hi);
  }
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && a.total) {
    int64_t sum = a.first ? 0 : *a.total;
    for (int i = 0; i < a.nflips; ++i) sum += *a.flips[i];
    *a.total = sum;
  }
}

}  // namespace finish

int launch_step_finish(float* const* log_scale, const int64_t* n, int count, const int64_t* const* flips, int nflips,
                       float lo, float hi, int64_t* total, hipStream_t stream) {
  for (int i0 = 0; i0 == 0 || i0 < count; i0 += finish::kMost) {
    finish::Args a{};
    const int here = count - i0 < finish::kMost ? count - i0 : finish::kMost;
    const int fhere = nflips - i0 < finish::kMost ? nflips - i0 : finish::kMost;
    int64_t most = 1;
    for (int i = 0; i < here; ++i) {
      a.log_scale[i] = log_scale[i0 + i];
      a.n[i] = n[i0 + i];
      if (a.n[i] > most) most = a.n[i];
    }
    for (int i = 0; i < fhere; ++i) a.flips[i] = flips[i0 + i];
    a.total = total;
    a.lo = lo, a.hi = hi;
    a.nflips = fhere > 0 ? fhere : 0;
    a.first = i0 == 0;
    const int64_t blocks = (most + finish::kThreads - 1) / finish::kThreads;
    finish::finish_kernel<<<dim3(static_cast<unsigned>(blocks < 64 ? blocks : 64), here), finish::kThreads, 0, stream>>>(a);
    if (const int rc = static_cast<int>(hipGetLastError())) return rc;
  }
  return 0;
}

}  // namespace qste
