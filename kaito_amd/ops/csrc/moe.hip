// MoE feed-forward of decode-sized steps for gfx950: few rows per expert, so
// both products stream the weights once (skinny.h stream_tile) and are bound
// by that. Everything is device-side and static-shaped, so that MoE decode
// steps capture into hipGraphs:
//
//   * tokens are sorted by expert on the GPU (moe_route.hip) and the kernels
//     get `sorted_ids` (token per sorted row) and `offsets` ([E+1] exclusive
//     prefix sums, by global expert);
//   * moe_gate_silu: act[s] = silu(x[tok] Wg^T) * (x[tok] Wu^T), the rows
//     gathered through sorted_ids (ungated experts, act_mode 2: relu(.)^2). A
//     workgroup's 16 weight rows are 8 gate rows and their 8 up rows;
//   * moe_down_rows: y[s] = act[s] Wd^T in f32, summed per token by
//     moe_combine.
//
// One workgroup per (16 weight rows, expert); an expert with more rows than 16
// MT is walked in passes, whose weights come back from the caches. Measured
// on one MI355X (32 tokens, 8 experts of 2048 x 2048, top 2) against 64 x 128
// tiles with both operands staged behind barriers, on 128 workgroups:
// 89 us for both products, now 47 (201 MB of weights: 4.3 TB/s). 32 experts
// of 2880 x 2880 (K in stages of 64), top 4, whole layer: 8 tokens 491 -> 178,
// 64 tokens 440 -> 297.
//
// Expert parallelism: callers pass `e_base` and the LOCAL weights; TP shards
// the expert intermediate dim. Both use these kernels unchanged.
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

namespace {

struct StreamArgs {
  const short* x;                   // up: [T, K]; down: [TK, K]
  const short* w;                   // [E local, rows, K]
  const short* bias;                // [E local, rows] or nullptr
  const int* rows;                  // token of a sorted row
  const int* offsets;               // [global E + 1]
  int e_base, N, K;
  int act_mode;
  float limit;
  short* act;                       // up: [TK, N]
  float* y;                         // down: [TK, N]
};

enum Kind { UP_GATED, UP_PLAIN, DOWN };

// act_mode 1: clamped swiglu — gate=min(g,limit), up=clamp(u,±limit),
// (up+1) * gate*sigmoid(1.702*gate); gpt-oss uses limit 7
KAITO_DEV float moe_act_f(int mode, float g, float u, float limit) {
  if (mode == 1) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    const float glu = g / (1.f + __expf(-1.702f * g));
    return (u + 1.f) * glu;
  }
  return skinny::silu(g) * u;
}

template <int MT, int KS, int KIND>
__global__ __launch_bounds__(256, 2) void moe_stream_kernel(const StreamArgs a) {
  constexpr int NI = skinny::tile_loads<KS>();
  constexpr bool GATED = KIND == UP_GATED;
  __shared__ __attribute__((aligned(128))) short ring[4][2][16 * KS];
  static_assert(sizeof(ring) >= 4 * MT * 64 * sizeof(f32x4), "fold");
  const int le = blockIdx.y;
  const int begin = a.offsets[a.e_base + le], end = a.offsets[a.e_base + le + 1];
  if (begin >= end) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (GATED ? 8 : 16);
  const int64_t wrows = GATED ? 2 * a.N : a.N;
  const short* src[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int r = skinny::tile_row<KS>(j, lane);
    const int64_t n = GATED ? n0 + r % 8 + (r >= 8 ? a.N : 0) : n0 + r;
    src[j] = a.w + (le * wrows + n) * a.K + skinny::tile_col<KS>(j, lane);
  }
  f32x4* red = reinterpret_cast<f32x4*>(&ring[0][0][0]);
  const int slot = threadIdx.x, l = slot & 63, c = l & 15;
  const bool mine = slot < MT * 64 && !(GATED && c >= 8);
  const short* be = a.bias ? a.bias + le * wrows + n0 + c : nullptr;
  for (int m0 = begin; m0 < end; m0 += 16 * MT) {
    const short* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const int m = min(m0 + mt * 16 + (lane & 15), end - 1);
      const int64_t row = KIND == DOWN ? m : a.rows[m];
      xp[mt] = a.x + row * a.K + (lane >> 4) * 8;
    }
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    skinny::stream_tile<MT, KS>(acc, src, xp, ring[wave][0], a.K, wave, lane);
    __syncthreads();                // every wave is done with its stages
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
      red[(wave * MT + mt) * 64 + lane] = acc[mt];
    __syncthreads();
    if (mine) {
      f32x4 v = skinny::fold<MT, 4>(red, slot), u{0.f, 0.f, 0.f, 0.f};
      if constexpr (GATED) u = skinny::fold<MT, 4>(red, slot + 8);
      if (be) {
        v += bf16_to_f32(be[0]);
        if constexpr (GATED) u += bf16_to_f32(be[a.N]);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = m0 + (slot >> 6) * 16 + (l >> 4) * 4 + r;
        if (m >= end) break;
        if constexpr (KIND == UP_GATED) {
          a.act[(int64_t)m * a.N + n0 + c] =
              f32_to_bf16(moe_act_f(a.act_mode, v[r], u[r], a.limit));
        } else if constexpr (KIND == UP_PLAIN) {
          const float p = fmaxf(v[r], 0.f);
          a.act[(int64_t)m * a.N + n0 + c] = f32_to_bf16(p * p);
        } else {
          a.y[(int64_t)m * a.N + n0 + c] = v[r];
        }
      }
    }
    __syncthreads();                // sums read before the next pass's stages
  }
}

// pairs: (token, expert) pairs of the step, over all E experts
template <int KIND>
void launch_stream(const StreamArgs& a, int64_t E_local, int64_t pairs,
                   int64_t E) {
  const dim3 grid(a.N / (KIND == UP_GATED ? 8 : 16), E_local), block(256);
  auto stream = at::hip::getCurrentHIPStream();
  // two row tiles once most experts have more than one
  const bool two = pairs > 12 * E;
#define MS_LAUNCH(MT_, KS_)                                                   \
  hipLaunchKernelGGL((moe_stream_kernel<MT_, KS_, KIND>), grid, block, 0,     \
                     stream, a)
  if (a.K % 256 == 0) {
    if (two) MS_LAUNCH(2, 256); else MS_LAUNCH(1, 256);
  } else {
    if (two) MS_LAUNCH(2, 64); else MS_LAUNCH(1, 64);
  }
#undef MS_LAUNCH
}

void check16(const at::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 &&
              t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0);
}

}  // namespace

void moe_gate_silu(at::Tensor act, at::Tensor x, at::Tensor w_gate_up,
                   at::Tensor sorted_ids, at::Tensor offsets,
                   at::Tensor bias, int64_t act_mode,
                   int64_t e_base, int64_t n_local_experts,
                   double act_limit) {
  check16(act); check16(x); check16(w_gate_up);
  TORCH_CHECK(sorted_ids.dtype() == at::kInt && offsets.dtype() == at::kInt);
  const bool gated = act_mode != 2;
  StreamArgs a{};
  a.N = act.size(1); a.K = x.size(1);
  TORCH_CHECK(a.K % 64 == 0 && a.N % 64 == 0,
              "H/IE must be multiples of 64 for the fused MoE path");
  TORCH_CHECK(w_gate_up.size(1) == (gated ? 2 : 1) * (int64_t)a.N &&
              w_gate_up.size(2) == a.K &&
              w_gate_up.size(0) >= n_local_experts &&
              offsets.numel() > e_base + n_local_experts &&
              act.size(0) >= sorted_ids.numel());
  if (bias.numel() > 0) {
    TORCH_CHECK(bias.dtype() == at::kBFloat16 && bias.is_contiguous() &&
                bias.numel() == w_gate_up.size(0) * 2 * a.N);
    a.bias = (const short*)bias.data_ptr();
  }
  TORCH_CHECK(gated || a.bias == nullptr, "ungated experts take no bias");
  if (sorted_ids.numel() == 0 || n_local_experts == 0 || a.N == 0) return;
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w_gate_up.data_ptr();
  a.rows = sorted_ids.data_ptr<int>();
  a.offsets = offsets.data_ptr<int>();
  a.e_base = (int)e_base;
  a.act_mode = (int)act_mode;
  a.limit = (float)act_limit;
  a.act = (short*)act.data_ptr();
  const int64_t pairs = sorted_ids.numel(), E = offsets.numel() - 1;
  if (gated) launch_stream<UP_GATED>(a, n_local_experts, pairs, E);
  else launch_stream<UP_PLAIN>(a, n_local_experts, pairs, E);
}

void moe_down_rows(at::Tensor y, at::Tensor act, at::Tensor w_down,
                   at::Tensor offsets, at::Tensor bias, int64_t e_base,
                   int64_t n_local_experts) {
  TORCH_CHECK(y.is_cuda() && y.dtype() == at::kFloat && y.is_contiguous() &&
              offsets.dtype() == at::kInt);
  check16(act); check16(w_down);
  StreamArgs a{};
  a.N = y.size(1); a.K = act.size(1);
  TORCH_CHECK(a.N % 64 == 0 && a.K % 64 == 0);
  TORCH_CHECK(w_down.size(1) == a.N && w_down.size(2) == a.K &&
              w_down.size(0) >= n_local_experts &&
              offsets.numel() > e_base + n_local_experts &&
              act.size(0) >= y.size(0));
  if (bias.numel() > 0) {
    TORCH_CHECK(bias.dtype() == at::kBFloat16 && bias.is_contiguous() &&
                bias.numel() == w_down.size(0) * a.N);
    a.bias = (const short*)bias.data_ptr();
  }
  if (y.size(0) == 0 || n_local_experts == 0 || a.N == 0) return;
  a.x = (const short*)act.data_ptr();
  a.w = (const short*)w_down.data_ptr();
  a.offsets = offsets.data_ptr<int>();
  a.e_base = (int)e_base;
  a.y = y.data_ptr<float>();
  launch_stream<DOWN>(a, n_local_experts, y.size(0), offsets.numel() - 1);
}

}  // namespace kaito
