// Rotary position embedding (neox / llama "rotate-half" style), in-place
// on Q and K. gfx950: trig tables are precomputed on device once (host-side
// cache tensor) — on-device sinf/cosf per element turns a memory-bound op
// VALU-bound (guide Appendix B).
//
// cos_sin_cache: [max_pos, rot_dim] f32 laid out as [cos(rot_dim/2) | sin(rot_dim/2)].
#include "common.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

// q: [T, QH*D], k: [T, KH*D] (contiguous rows); positions: [T] int32/64.
// rotate-half: out[i]       = x[i]*cos[i] - x[i+R/2]*sin[i]
//              out[i+R/2]   = x[i+R/2]*cos[i] + x[i]*sin[i]      (i < R/2)
__global__ void rope_kernel(
    short* __restrict__ q, short* __restrict__ k,
    const int64_t* __restrict__ positions,
    const float* __restrict__ cos_sin,  // [max_pos, R]
    const int T, const int QH, const int KH, const int D, const int R,
    const int64_t q_stride, const int64_t k_stride) {
  const int token = blockIdx.x;
  if (token >= T) return;
  const int64_t pos = positions[token];
  const float* cs = cos_sin + pos * R;
  const int half = R / 2;
  const int total_heads = QH + KH;

  // Each thread handles one (head, i<half) pair; vectorize by 2 along i.
  for (int idx = threadIdx.x; idx < total_heads * half / 2; idx += blockDim.x) {
    const int pair = idx * 2;               // i offset within half, step 2
    const int h = pair / half;
    const int i = pair % half;
    short* base = (h < QH)
        ? q + (int64_t)token * q_stride + (int64_t)h * D
        : k + (int64_t)token * k_stride + (int64_t)(h - QH) * D;
    // load x[i..i+1] and x[i+half..i+half+1]
    short2 xa = *reinterpret_cast<short2*>(base + i);
    short2 xb = *reinterpret_cast<short2*>(base + i + half);
    float2 c = *reinterpret_cast<const float2*>(cs + i);
    float2 s = *reinterpret_cast<const float2*>(cs + half + i);
    float a0 = bf16_to_f32(xa.x), a1 = bf16_to_f32(xa.y);
    float b0 = bf16_to_f32(xb.x), b1 = bf16_to_f32(xb.y);
    short2 oa, ob;
    oa.x = f32_to_bf16(a0 * c.x - b0 * s.x);
    oa.y = f32_to_bf16(a1 * c.y - b1 * s.y);
    ob.x = f32_to_bf16(b0 * c.x + a0 * s.x);
    ob.y = f32_to_bf16(b1 * c.y + a1 * s.y);
    *reinterpret_cast<short2*>(base + i) = oa;
    *reinterpret_cast<short2*>(base + i + half) = ob;
  }
}

void rotary_embedding(at::Tensor positions, at::Tensor q, at::Tensor k,
                      int64_t head_dim, at::Tensor cos_sin_cache) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == at::kBFloat16);
  TORCH_CHECK(positions.dtype() == at::kLong);
  TORCH_CHECK(q.stride(-1) == 1 && k.stride(-1) == 1,
              "rope: innermost dim must be contiguous");
  const int T = positions.size(0);
  const int R = cos_sin_cache.size(1);
  const int D = (int)head_dim;
  const int QH = (int)(q.size(-1) / D) * (q.dim() == 3 ? (int)q.size(1) : 1);
  const int KH = (int)(k.size(-1) / D) * (k.dim() == 3 ? (int)k.size(1) : 1);
  TORCH_CHECK(R <= D && R % 4 == 0, "rot_dim must be <= head_dim, mult of 4");
  auto stream = at::hip::getCurrentHIPStream();
  const int block = 256;
  hipLaunchKernelGGL(rope_kernel, dim3(T), dim3(block), 0, stream,
      (short*)q.data_ptr(), (short*)k.data_ptr(),
      positions.data_ptr<int64_t>(), cos_sin_cache.data_ptr<float>(),
      T, QH, KH, D, R, q.stride(0), k.stride(0));
}

namespace {

// The rotation and the scatter of k and v into the paged cache (cache.hip) in
// one pass, 16 bytes at a time. Decode steps are bound by the launches (two
// of about 4 us before, one now), prompts by memory (k was read twice).
// Same arithmetic and rounding as the two.
template <bool FP8>
__global__ __launch_bounds__(256)
void rope_cache_kernel(
    short* __restrict__ q, short* __restrict__ k, const short* __restrict__ v,
    const int64_t q_stride, const int64_t k_stride, const int64_t v_stride,
    const int64_t* __restrict__ positions,
    const float* __restrict__ cos_sin,      // [max_pos, R]
    void* __restrict__ k_cache,             // [B, KH, BS, D] bf16 | e4m3
    void* __restrict__ v_cache, const int64_t* __restrict__ slots,
    const int QH, const int KH, const int D, const int R, const int BS) {
  const int64_t t = blockIdx.x, slot = slots[t];
  const float* cs = cos_sin + positions[t] * R;
  const int64_t page = slot / BS * KH;      // head h: row (page + h) * BS + off
  const int off = (int)(slot % BS), half = R / 2;
  auto put = [&](void* cache, const int h, const int d, const short8_t x) {
    if (slot < 0) return;
    const int64_t at = (((page + h) * BS + off) * D + d) / 8;
    if constexpr (FP8) {
      u8x8_t o;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t w = f32x2_to_fp8x2(bf16_to_f32(x[2 * j]),
                                          bf16_to_f32(x[2 * j + 1]));
        o[2 * j] = w & 0xFF;
        o[2 * j + 1] = (w >> 8) & 0xFF;
      }
      reinterpret_cast<u8x8_t*>(cache)[at] = o;
    } else {
      reinterpret_cast<short8_t*>(cache)[at] = x;
    }
  };
  // (head, 8 pairs) | v chunks | k chunks that are not rotated
  const int pairs = half / 8, rot = (QH + KH) * pairs, vc = KH * D / 8;
  const int rest = (D - R) / 8, total = rot + vc + KH * rest;
  for (int i = threadIdx.x; i < total; i += 256) {
    if (i < rot) {
      const int h = i / pairs, d = i % pairs * 8;
      short* x = h < QH ? q + t * q_stride + (int64_t)h * D
                        : k + t * k_stride + (int64_t)(h - QH) * D;
      const short8_t xa = *reinterpret_cast<const short8_t*>(x + d);
      const short8_t xb = *reinterpret_cast<const short8_t*>(x + half + d);
      short8_t oa, ob;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float c = cs[d + j], s = cs[half + d + j];
        const float a = bf16_to_f32(xa[j]), b = bf16_to_f32(xb[j]);
        oa[j] = f32_to_bf16(a * c - b * s);
        ob[j] = f32_to_bf16(b * c + a * s);
      }
      *reinterpret_cast<short8_t*>(x + d) = oa;
      *reinterpret_cast<short8_t*>(x + half + d) = ob;
      if (h >= QH) {
        put(k_cache, h - QH, d, oa);
        put(k_cache, h - QH, half + d, ob);
      }
    } else if (i < rot + vc) {
      const int c = (i - rot) * 8;
      put(v_cache, c / D, c % D,
          *reinterpret_cast<const short8_t*>(v + t * v_stride + c));
    } else {
      const int c = i - rot - vc, h = c / rest, d = R + c % rest * 8;
      put(k_cache, h, d,
          *reinterpret_cast<const short8_t*>(k + t * k_stride +
                                             (int64_t)h * D + d));
    }
  }
}

}  // namespace

// q [T, QH * D], k and v [T, KH * D] rows of any stride; k_cache's last dim
// is D
void rope_and_cache(at::Tensor positions, at::Tensor q, at::Tensor k,
                    at::Tensor v, at::Tensor cos_sin, at::Tensor k_cache,
                    at::Tensor v_cache, at::Tensor slots) {
  auto ok = [](const at::Tensor& t) {
    return t.is_cuda() && t.dtype() == at::kBFloat16 && t.dim() == 2 &&
           t.stride(1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0 &&
           (t.size(0) == 1 || t.stride(0) % 8 == 0);
  };
  TORCH_CHECK(ok(q) && ok(k) && ok(v));
  const int64_t T = q.size(0);
  const int R = cos_sin.size(1), KH = k_cache.size(1), BS = k_cache.size(2);
  const int D = k_cache.size(3);
  TORCH_CHECK(D % 8 == 0 && R % 16 == 0 && R <= D && q.size(1) % D == 0 &&
              k.size(1) == (int64_t)KH * D && v.size(1) == k.size(1) &&
              k.size(0) == T && v.size(0) == T);
  TORCH_CHECK(positions.dtype() == at::kLong && positions.numel() == T &&
              positions.is_contiguous() && slots.dtype() == at::kLong &&
              slots.numel() == T && slots.is_contiguous());
  TORCH_CHECK(cos_sin.dtype() == at::kFloat && cos_sin.is_contiguous() &&
              k_cache.is_contiguous() && v_cache.is_contiguous() &&
              k_cache.dtype() == v_cache.dtype() &&
              k_cache.sizes() == v_cache.sizes());
  if (T == 0) return;
  const bool fp8 = k_cache.dtype() == at::kByte;
  TORCH_CHECK(fp8 || k_cache.dtype() == at::kBFloat16);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(T), dim3(256), 0,
        at::hip::getCurrentHIPStream(), (short*)q.data_ptr(),
        (short*)k.data_ptr(), (const short*)v.data_ptr(), q.stride(0),
        k.stride(0), v.stride(0), positions.data_ptr<int64_t>(),
        cos_sin.data_ptr<float>(), k_cache.data_ptr(), v_cache.data_ptr(),
        slots.data_ptr<int64_t>(), (int)(q.size(1) / D), KH, D, R, BS);
  };
  if (fp8) launch(&rope_cache_kernel<true>);
  else launch(&rope_cache_kernel<false>);
}

}  // namespace kaito
