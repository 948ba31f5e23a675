// Linear layers of the smallest decode steps (skinny.h), M <= 4 rows:
//   skinny_linear  out = x W^T (+ bias)
//   skinny_swiglu  out = silu(x Wg^T) * (x Wu^T), W = [Wg | Wu] stacked
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

namespace {

constexpr int NW = 4;

// GLU: the wave's two rows are a gate row and its up row (N apart)
template <int M, int R, bool GLU>
__global__ __launch_bounds__(NW * 64) void skinny_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const int64_t x_stride, const short* __restrict__ w,
    const short* __restrict__ bias, const int N, const int K) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * NW + wave) * (GLU ? 1 : R);
  if (n0 >= N) return;
  const short* wp[R];
  float acc[M][R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    wp[r] = w + (int64_t)(GLU ? r * N + n0 : min(n0 + r, N - 1)) * K;
#pragma unroll
    for (int m = 0; m < M; m++) acc[m][r] = 0.f;
  }
  skinny::stream_rows<M, R>(acc, wp, x, x_stride, K, lane);
#pragma unroll
  for (int m = 0; m < M; m++) {
#pragma unroll
    for (int r = 0; r < R; r++) acc[m][r] = wave_reduce_sum(acc[m][r]);
    if constexpr (GLU) {
      if (lane == 0)
        out[(int64_t)m * N + n0] =
            f32_to_bf16(skinny::silu(acc[m][0]) * acc[m][1]);
    } else {
#pragma unroll
      for (int r = 0; r < R; r++)
        if (lane == 0 && n0 + r < N)
          out[(int64_t)m * N + n0 + r] = f32_to_bf16(
              acc[m][r] + (bias ? bf16_to_f32(bias[n0 + r]) : 0.f));
    }
  }
}

void check(const at::Tensor& out, const at::Tensor& x, const at::Tensor& w,
           int64_t N) {
  for (const auto& t : {out, x, w})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 && t.dim() == 2 &&
                t.stride(1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(w.is_contiguous() && out.is_contiguous() &&
              x.size(1) == w.size(1) && out.size(0) == x.size(0) &&
              out.size(1) == N);
  TORCH_CHECK(x.size(0) >= 1 && x.size(0) <= 4 && w.size(1) % 8 == 0 &&
              w.size(1) > 0 && (x.size(0) == 1 || x.stride(0) % 8 == 0) &&
              w.size(0) < (1ll << 31) && w.size(1) < (1ll << 31));
}

}  // namespace

void skinny_linear(at::Tensor out, at::Tensor x, at::Tensor w,
                   at::Tensor bias) {
  const int64_t N = w.size(0);
  check(out, x, w, N);
  const bool has_bias = bias.numel() > 0;
  TORCH_CHECK(!has_bias || (bias.is_cuda() && bias.is_contiguous() &&
                            bias.dtype() == at::kBFloat16 &&
                            bias.numel() == N));
  if (N == 0) return;
  // one row per wave keeps most waves under way for a single x row (N =
  // 4096, K = 4096: 6.6 us against 6.8 with two); with more, two rows share
  // the x loads (M = 4, N = 28672: 48 us)
#define SL_LAUNCH(M_, R_)                                                     \
  hipLaunchKernelGGL((skinny_linear_kernel<M_, R_, false>),                   \
      dim3((N + NW * R_ - 1) / (NW * R_)), dim3(NW * 64), 0,                  \
      at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),                 \
      (const short*)x.data_ptr(), x.stride(0), (const short*)w.data_ptr(),    \
      has_bias ? (const short*)bias.data_ptr() : nullptr, (int)N,             \
      (int)w.size(1))
  switch (x.size(0)) {
    case 1: SL_LAUNCH(1, 1); break;
    case 2: SL_LAUNCH(2, 2); break;
    case 3: SL_LAUNCH(3, 2); break;
    default: SL_LAUNCH(4, 2); break;
  }
#undef SL_LAUNCH
}

void skinny_swiglu(at::Tensor out, at::Tensor x, at::Tensor w) {
  TORCH_CHECK(w.size(0) % 2 == 0);
  const int64_t N = w.size(0) / 2;
  check(out, x, w, N);
  if (N == 0) return;
#define SG_LAUNCH(M_)                                                         \
  hipLaunchKernelGGL((skinny_linear_kernel<M_, 2, true>),                     \
      dim3((N + NW - 1) / NW), dim3(NW * 64), 0,                              \
      at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),                 \
      (const short*)x.data_ptr(), x.stride(0), (const short*)w.data_ptr(),    \
      nullptr, (int)N, (int)w.size(1))
  switch (x.size(0)) {
    case 1: SG_LAUNCH(1); break;
    case 2: SG_LAUNCH(2); break;
    case 3: SG_LAUNCH(3); break;
    default: SG_LAUNCH(4); break;
  }
#undef SG_LAUNCH
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("skinny_linear(Tensor(a!) out, Tensor x, Tensor w, Tensor bias) -> ()");
  m.def("skinny_swiglu(Tensor(a!) out, Tensor x, Tensor w) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("skinny_linear", &kaito::skinny_linear);
  m.impl("skinny_swiglu", &kaito::skinny_swiglu);
}
