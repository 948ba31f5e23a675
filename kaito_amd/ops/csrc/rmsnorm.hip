// Fused RMSNorm kernels for gfx950.
//
// Replaces the fused CUDA norm ops the reference delegates to vLLM
// (invoked via presets/workspace/inference/vllm/inference_api.py -> vLLM).
//
// Memory-bound: target is HBM BW. All bf16 traffic is vectorized as
// short8 (16 B/lane). One workgroup per token row; grid-stride over rows.
#include "common.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

// out[row] = x[row] / rms(x[row]) * w      (x: bf16 [T, H], w: bf16 [H])
// If RESIDUAL: residual += x first (both updated in place semantics:
// residual_out = x + residual; out = norm(residual_out) * w).
template <bool RESIDUAL>
__global__ void rms_norm_kernel(
    short* __restrict__ out,            // [T, H] bf16
    const short* __restrict__ x,        // [T, H] bf16
    short* __restrict__ residual,       // [T, H] bf16 or nullptr
    const short* __restrict__ w,        // [H]
    const float eps, const int H, const int T) {
  __shared__ float red[16];
  const int VEC = 8;
  const int nvec = H / VEC;

  for (int row = blockIdx.x; row < T; row += gridDim.x) {
    const short8_t* xv = reinterpret_cast<const short8_t*>(x + (int64_t)row * H);
    short8_t* rv = RESIDUAL ? reinterpret_cast<short8_t*>(residual + (int64_t)row * H) : nullptr;
    float ss = 0.f;
    // pass 1: (optionally add residual), accumulate sum of squares.
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = xv[i];
      if (RESIDUAL) {
        short8_t r = rv[i];
#pragma unroll
        for (int j = 0; j < VEC; j++) {
          float f = bf16_to_f32(v[j]) + bf16_to_f32(r[j]);
          v[j] = f32_to_bf16(f);
        }
        rv[i] = v;  // residual stream updated in bf16
      }
#pragma unroll
      for (int j = 0; j < VEC; j++) {
        float f = bf16_to_f32(v[j]);
        ss += f * f;
      }
    }
    ss = block_reduce_sum(ss, red);
    // broadcast via LDS (block_reduce leaves full sum in every lane of wave0
    // only when nwaves<=64; we re-broadcast explicitly for safety)
    __shared__ float s_inv;
    if (threadIdx.x == 0) s_inv = rsqrtf(ss / (float)H + eps);
    __syncthreads();
    const float inv = s_inv;

    const short8_t* src = RESIDUAL ? reinterpret_cast<const short8_t*>(residual + (int64_t)row * H) : xv;
    const short8_t* wv = reinterpret_cast<const short8_t*>(w);
    short8_t* ov = reinterpret_cast<short8_t*>(out + (int64_t)row * H);
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = src[i];
      short8_t g = wv[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < VEC; j++)
        o[j] = f32_to_bf16(bf16_to_f32(v[j]) * inv * bf16_to_f32(g[j]));
      ov[i] = o;
    }
    __syncthreads();
  }
}

// The same for rows of up to 2048 ITER, which stay in registers: the residual is
// not read back, and one barrier less stands in the chain that bounds small steps.
// 1 row of 4096 with the residual 3.2 -> 2.9 us with the launch, 256 4.0 -> 3.6, 9200
// 47.1 -> 45.2; 9200 of 8192 without it 64.8 -> 52.0. The same bits.
template <bool RESIDUAL, int ITER>
__global__ __launch_bounds__(256) void rms_norm_reg_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    short* __restrict__ residual, const short* __restrict__ w,
    const float eps, const int H, const int T) {
  __shared__ float red[2][4];
  const int at = threadIdx.x * 8;
  short8_t g[ITER];
#pragma unroll
  for (int i = 0; i < ITER; i++)
    if (i * 2048 + at < H)
      g[i] = *reinterpret_cast<const short8_t*>(w + i * 2048 + at);
  int par = 0;
  for (int64_t row = blockIdx.x; row < T; row += gridDim.x, par ^= 1) {
    short8_t v[ITER];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < ITER; i++) {
      const int c = i * 2048 + at;
      if (c >= H) break;
      v[i] = *reinterpret_cast<const short8_t*>(x + row * H + c);
      if constexpr (RESIDUAL) {
        short8_t* r = reinterpret_cast<short8_t*>(residual + row * H + c);
        const short8_t u = *r;
#pragma unroll
        for (int j = 0; j < 8; j++)
          v[i][j] = f32_to_bf16(bf16_to_f32(v[i][j]) + bf16_to_f32(u[j]));
        *r = v[i];
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float f = bf16_to_f32(v[i][j]);
        ss += f * f;
      }
    }
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & 63) == 0) red[par][threadIdx.x >> 6] = ss;
    __syncthreads();                // the other half is free once all are here
    ss = (red[par][0] + red[par][1]) + (red[par][2] + red[par][3]);
    const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
    for (int i = 0; i < ITER; i++) {
      const int c = i * 2048 + at;
      if (c >= H) break;
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; j++)
        o[j] = f32_to_bf16(bf16_to_f32(v[i][j]) * inv * bf16_to_f32(g[i][j]));
      *reinterpret_cast<short8_t*>(out + row * H + c) = o;
    }
  }
}

// rms_norm_reg_kernel<true> of rows that a product split over K left in parts, summed
// here in their order and rounded to bf16 as by the launch that would else have done
// it: the same bits, a launch and a pass less. With
// the product, us, by way of its sum and now: 4096 x 14336 28.3, 27.3 at 16 rows, 33.1,
// 31.6 at 64, 53.7, 51.3 at 250, 7168 x 18432 104.3, 100.4 at 250, 4096 x 4096 17.9,
// 16.5 at 64.
template <int ITER>
__global__ __launch_bounds__(256) void rms_norm_parts_kernel(
    short* __restrict__ out, const float* __restrict__ part, const int splits,
    short* __restrict__ residual, const short* __restrict__ w,
    const float eps, const int H, const int T) {
  __shared__ float red[4];
  const int at = threadIdx.x * 8;
  const int64_t row = blockIdx.x, total = (int64_t)T * H;
  short8_t g[ITER], v[ITER];
  float f[ITER][8];
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = i * 2048 + at;
#pragma unroll
    for (int j = 0; j < 8; j++) f[i][j] = -0.f;
    if (c >= H) break;
    g[i] = *reinterpret_cast<const short8_t*>(w + c);
    v[i] = *reinterpret_cast<const short8_t*>(residual + row * H + c);
  }
#pragma unroll 4
  for (int s = 0; s < splits; s++) {
#pragma unroll
    for (int i = 0; i < ITER; i++) {
      const int c = i * 2048 + at;
      if (c >= H) break;
      const f32x4* p =
          reinterpret_cast<const f32x4*>(part + s * total + row * H + c);
      const f32x4 a = p[0], b = p[1];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        f[i][j] += a[j];
        f[i][j + 4] += b[j];
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = i * 2048 + at;
    if (c >= H) break;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      v[i][j] = f32_to_bf16(bf16_to_f32(f32_to_bf16(f[i][j])) +
                            bf16_to_f32(v[i][j]));
      const float e = bf16_to_f32(v[i][j]);
      ss += e * e;
    }
    *reinterpret_cast<short8_t*>(residual + row * H + c) = v[i];
  }
  ss = wave_reduce_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = i * 2048 + at;
    if (c >= H) break;
    short8_t o;
#pragma unroll
    for (int j = 0; j < 8; j++)
      o[j] = f32_to_bf16(bf16_to_f32(v[i][j]) * inv * bf16_to_f32(g[i][j]));
    *reinterpret_cast<short8_t*>(out + row * H + c) = o;
  }
}

// LayerNorm (+optional bias, +optional residual add) — phi-2 / falcon
// norm layers. Same vectorized one-workgroup-per-row structure.
template <bool RESIDUAL>
__global__ void layer_norm_kernel(
    short* __restrict__ out,            // [T, H] bf16
    const short* __restrict__ x,        // [T, H] bf16
    short* __restrict__ residual,       // [T, H] bf16 or nullptr
    const short* __restrict__ w,        // [H]
    const short* __restrict__ b,        // [H] or nullptr
    const float eps, const int H, const int T) {
  __shared__ float red[16];
  const int VEC = 8;
  const int nvec = H / VEC;
  for (int row = blockIdx.x; row < T; row += gridDim.x) {
    const short8_t* xv =
        reinterpret_cast<const short8_t*>(x + (int64_t)row * H);
    short8_t* rv = RESIDUAL
        ? reinterpret_cast<short8_t*>(residual + (int64_t)row * H) : nullptr;
    float sum = 0.f, ssq = 0.f;
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = xv[i];
      if (RESIDUAL) {
        short8_t r = rv[i];
#pragma unroll
        for (int j = 0; j < VEC; j++)
          v[j] = f32_to_bf16(bf16_to_f32(v[j]) + bf16_to_f32(r[j]));
        rv[i] = v;
      }
#pragma unroll
      for (int j = 0; j < VEC; j++) {
        const float f = bf16_to_f32(v[j]);
        sum += f;
        ssq += f * f;
      }
    }
    sum = block_reduce_sum(sum, red);
    __syncthreads();          // red[] reused by the second reduction
    ssq = block_reduce_sum(ssq, red);
    __shared__ float s_mu, s_inv;
    if (threadIdx.x == 0) {
      const float mu = sum / (float)H;
      s_mu = mu;
      s_inv = rsqrtf(ssq / (float)H - mu * mu + eps);
    }
    __syncthreads();
    const float mu = s_mu, inv = s_inv;
    const short8_t* src = RESIDUAL
        ? reinterpret_cast<const short8_t*>(residual + (int64_t)row * H) : xv;
    short8_t* ov = reinterpret_cast<short8_t*>(out + (int64_t)row * H);
    const short8_t* wv = reinterpret_cast<const short8_t*>(w);
    const short8_t* bv = reinterpret_cast<const short8_t*>(b);
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = src[i];
      short8_t g = wv[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < VEC; j++) {
        float f = (bf16_to_f32(v[j]) - mu) * inv * bf16_to_f32(g[j]);
        if (b != nullptr) f += bf16_to_f32(bv[i][j]);
        o[j] = f32_to_bf16(f);
      }
      ov[i] = o;
    }
    __syncthreads();
  }
}

void layer_norm(at::Tensor out, at::Tensor input, at::Tensor weight,
                at::Tensor bias, double eps) {
  TORCH_CHECK(input.is_cuda() && input.dtype() == at::kBFloat16);
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous());
  const int H = input.size(-1);
  const int64_t T = input.numel() / H;
  TORCH_CHECK(H % 8 == 0);
  const int block = 256;
  const int grid = (int)std::min<int64_t>(T, 2048);
  auto stream = at::hip::getCurrentHIPStream();
  const short* b = bias.numel() > 0 ? (const short*)bias.data_ptr() : nullptr;
  hipLaunchKernelGGL((layer_norm_kernel<false>), dim3(grid), dim3(block), 0,
      stream, (short*)out.data_ptr(), (const short*)input.data_ptr(), nullptr,
      (const short*)weight.data_ptr(), b, (float)eps, H, (int)T);
}

void fused_add_layer_norm(at::Tensor out, at::Tensor input,
                          at::Tensor residual, at::Tensor weight,
                          at::Tensor bias, double eps) {
  TORCH_CHECK(input.is_cuda() && input.dtype() == at::kBFloat16);
  TORCH_CHECK(input.is_contiguous() && residual.is_contiguous() &&
              out.is_contiguous());
  const int H = input.size(-1);
  const int64_t T = input.numel() / H;
  TORCH_CHECK(H % 8 == 0);
  const int block = 256;
  const int grid = (int)std::min<int64_t>(T, 2048);
  auto stream = at::hip::getCurrentHIPStream();
  const short* b = bias.numel() > 0 ? (const short*)bias.data_ptr() : nullptr;
  hipLaunchKernelGGL((layer_norm_kernel<true>), dim3(grid), dim3(block), 0,
      stream, (short*)out.data_ptr(), (const short*)input.data_ptr(),
      (short*)residual.data_ptr(), (const short*)weight.data_ptr(), b,
      (float)eps, H, (int)T);
}

namespace {

template <bool RESIDUAL>
void launch_rms(const at::Tensor& out, const at::Tensor& input,
                short* residual, const at::Tensor& weight, double eps) {
  const int H = input.size(-1);
  const int64_t T = input.numel() / H;
  TORCH_CHECK(H % 8 == 0, "hidden size must be multiple of 8");
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((int)std::min<int64_t>(T, 2048)),
        dim3(256), 0, at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),
        (const short*)input.data_ptr(), residual,
        (const short*)weight.data_ptr(), (float)eps, H, (int)T);
  };
  if (H <= 2048) launch(&rms_norm_reg_kernel<RESIDUAL, 1>);
  else if (H <= 4096) launch(&rms_norm_reg_kernel<RESIDUAL, 2>);
  else if (H <= 8192) launch(&rms_norm_reg_kernel<RESIDUAL, 4>);
  else launch(&rms_norm_kernel<RESIDUAL>);
}

}  // namespace

void rms_norm(at::Tensor out, at::Tensor input, at::Tensor weight, double eps) {
  TORCH_CHECK(input.is_cuda() && input.dtype() == at::kBFloat16, "rms_norm: bf16 GPU only");
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous());
  launch_rms<false>(out, input, nullptr, weight, eps);
}

void fused_add_rms_norm(at::Tensor out, at::Tensor input, at::Tensor residual,
                        at::Tensor weight, double eps) {
  TORCH_CHECK(input.is_cuda() && input.dtype() == at::kBFloat16, "fused_add_rms_norm: bf16 GPU only");
  TORCH_CHECK(input.is_contiguous() && residual.is_contiguous() && out.is_contiguous());
  launch_rms<true>(out, input, (short*)residual.data_ptr(), weight, eps);
}

// fused_add_rms_norm of the sum of part [splits, T, H] f32
void add_rms_norm_parts(at::Tensor out, at::Tensor part, at::Tensor residual,
                        at::Tensor weight, double eps) {
  TORCH_CHECK(part.is_cuda() && part.dim() == 3 && part.is_contiguous() &&
              part.dtype() == at::kFloat);
  const int64_t S = part.size(0), T = part.size(1), H = part.size(2);
  for (const auto& t : {out, residual})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dim() == 2 &&
                t.dtype() == at::kBFloat16 && t.size(0) == T && t.size(1) == H &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(weight.is_cuda() && weight.is_contiguous() &&
              weight.numel() == H && weight.dtype() == at::kBFloat16 &&
              (uintptr_t)weight.data_ptr() % 16 == 0);
  TORCH_CHECK(S >= 1 && S <= 64 && T <= 65535 && H % 8 == 0 && H <= 8192);
  if (T == 0 || H == 0) return;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(T), dim3(256), 0,
        at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),
        part.data_ptr<float>(), (int)S, (short*)residual.data_ptr(),
        (const short*)weight.data_ptr(), (float)eps, (int)H, (int)T);
  };
  if (H <= 2048) launch(&rms_norm_parts_kernel<1>);
  else if (H <= 4096) launch(&rms_norm_parts_kernel<2>);
  else launch(&rms_norm_parts_kernel<4>);
}

}  // namespace kaito
