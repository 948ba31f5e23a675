// Products of 9 to 256 rows with a large weight matrix, out[M, N] = x[M, K] W^T:
// linear layers of batched decode steps and short prompts, whose bytes are W's
// (out = silu(x Wg^T) * (x Wu^T) for a stacked pair).
//
// A workgroup of 8 waves takes all M rows of x and 64 or 128 rows of W over one of
// `splits` parts of K; the parts' f32 sums are added, in order, by a second launch.
// Both operands arrive by direct LDS loads, three to eight K steps under way
// (16-byte chunk c of row r at c ^ (r & 7)), a barrier a step, transposed products
// (a lane holds 4 neighbouring outputs of a row of x).
//
// What bounds it: a CU takes 126 B/ns from L2 into LDS, but only 52 to 60 while
// misses are among the loads, whatever the number of steps under way: data return
// in order and some 400 lines can be asked for, so that all of them move at the pace
// of HBM's latency. x comes through that path once per workgroup, so time goes by
// (rows + columns) x K of a workgroup, and more columns with more parts of K pay for
// the parts' sums (plan_for). Interleaving W's loads in bursts of 8 steps gave 74
// B/ns alone, at the price of the LDS that holds them; touching W's lines ahead
// nothing.
//
// One MI355X, weights out of the caches, us, hipBLASLt and here (sums included):
// 4096 x 14336: 33 rows 33.3 and 26.7, 64 36.2 and 30.0, 128 49.4 and 38.5, 256 59.1
// and 47.3; 7168 x 18432 at 256 208 and 88; 28672 x 4096 as a pair: 64 60.2 and 49,
// 256 79.8 and 75; 4096 x 4096 at 64 14.2 and 15.0, at 256 20.7 and 26. At 256 rows
// of 28672 x 4096 the matrix cores' 41 us (1.45 PFLOP/s), 43 us of HBM and 52 of
// staging do not overlap fully.
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <cmath>

namespace kaito {

namespace {

using skinny::hbf16x8;
using skinny::load_x;
using skinny::mfma16;

constexpr int THREADS = 512;        // 8 waves
constexpr int LDS_BYTES = 160 * 1024;

struct BatchArgs {
  short* out;                       // [M, N]
  float* part;                      // [splits, M, N] or nullptr
  const short* x;
  int64_t x_stride;
  const short* w;                   // [N, K]; GLU [2 N, K]
  const short* bias;                // [N] or nullptr
  int M, N, K, splits;
};

enum Out { BF16, PARTIAL, GLU };

// BM = 16 WM MT rows of x, BN = 16 WN NT of w (WN = 8 / WM)
template <int WM, int MT, int NT, int BK>
struct Tile {
  static constexpr int WN = 8 / WM, BM = 16 * WM * MT, BN = 16 * WN * NT;
  static constexpr int STAGE = (BM + BN) * BK;
  static constexpr int FIT = LDS_BYTES / (STAGE * 2);
  static constexpr int NST = FIT < 8 ? FIT : 8;
};

template <int WM, int MT, int NT, int BK, int OUT>
KAITO_DEV void batch_tile(const BatchArgs& a, short* lds) {
  using T = Tile<WM, MT, NT, BK>;
  constexpr int WN = T::WN, BM = T::BM, BN = T::BN, CH = BK / 8;
  constexpr int STAGE = T::STAGE, NST = T::NST;
  constexpr int LX = (BM * CH + THREADS - 1) / THREADS, LW = BN * CH / THREADS;
  static_assert(BN * CH % THREADS == 0 && NST >= 3 &&
                (BM * CH % THREADS == 0 || THREADS % (BM * CH) == 0), "stage");
  static_assert(OUT != GLU || NT % 2 == 0, "pairs");
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int split = blockIdx.x % a.splits, tile = blockIdx.x / a.splits;
  constexpr int COLS = OUT == GLU ? BN / 2 : BN;
  const int n0 = tile * COLS;
  const int steps = a.K / BK;
  const int first = (int)((int64_t)steps * split / a.splits);
  const int last = (int)((int64_t)steps * (split + 1) / a.splits);

  const auto xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<short*>(a.x), 0, 0xffffffff, 0x27000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<short*>(a.w + (int64_t)n0 * a.K), 0, 0xffffffff, 0x27000);
  uint32_t xs[LX], ws[LW];
  int xd[LX];
#pragma unroll
  for (int j = 0; j < LX; j++) {
    const int s = (j * THREADS + threadIdx.x) % (BM * CH);
    const int row = s / CH, c = (s % CH) ^ (row & 7);
    xs[j] = (uint32_t)(min(row, a.M - 1) * a.x_stride + c * 8) * 2;
    xd[j] = (j * THREADS + wave * 64) % (BM * CH) * 8;
  }
#pragma unroll
  for (int j = 0; j < LW; j++) {
    const int s = j * THREADS + threadIdx.x, row = s / CH;
    const int c = (s % CH) ^ (row & 7);
    // GLU: every 32 tile rows are 16 gate rows, then their up rows
    const uint32_t n = OUT == GLU
        ? min(row / 32 * 16 + row % 16, a.N - 1 - n0) +
              (row % 32 >= 16 ? a.N : 0)
        : min(row, a.N - 1 - n0);
    ws[j] = (n * a.K + c * 8) * 2;
  }
  auto fetch = [&](const int s, const int slot) {
    short* p = lds + slot * STAGE;
    const int at = s * BK * 2;
#pragma unroll
    for (int j = 0; j < LW; j++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          wr,
          (__attribute__((address_space(3))) void*)(p + BM * BK +
                                                    (j * THREADS + wave * 64) *
                                                        8),
          16, ws[j], at, 0, 2 /* non-temporal */);
#pragma unroll
    for (int j = 0; j < LX; j++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xr, (__attribute__((address_space(3))) void*)(p + xd[j]), 16, xs[j],
          at, 0, 0);
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Fragments of 32 k are read one step ahead of their products, the first of
  // the next stage beside the last products of this one: the barrier that frees
  // this stage stands between its last read and its last products.
  constexpr int KK = BK / 32;
  hbf16x8 wf[2][NT], xf[2][MT];
  auto read = [&](const int slot, const int kk) {
    const int c = ((kk * 4 + hi) ^ (lo & 7)) * 8, f = kk & 1;
    const short* xb = lds + slot * STAGE + (wm * MT * 16 + lo) * BK + c;
    const short* wb = lds + slot * STAGE + (BM + wn * NT * 16 + lo) * BK + c;
#pragma unroll
    for (int i = 0; i < NT; i++) wf[f][i] = load_x(wb + i * 16 * BK);
#pragma unroll
    for (int j = 0; j < MT; j++) xf[f][j] = load_x(xb + j * 16 * BK);
  };
  auto multiply = [&](const int kk) {
    const int f = kk & 1;
    __builtin_amdgcn_sched_barrier(0);      // the next reads are under way
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int i = 0; i < NT; i++)
        acc[i][j] = mfma16(wf[f][i], xf[f][j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // own reads done and own loads landed but for the newest LATER stages: all's
  auto meet = [&](const bool later) {
    constexpr int N = (NST - 2) * (LX + LW);
    if (later)
      __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    else
      __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (first < last) {
#pragma unroll
    for (int i = 0; i < NST - 1; i++)
      if (first + i < last) fetch(first + i, i);
    meet(first + NST - 2 < last);
    if (first + NST - 1 < last) fetch(first + NST - 1, NST - 1);
    read(0, 0);
    int slot = 0;
    for (int s = first; s < last; s++) {
#pragma unroll
      for (int kk = 0; kk < KK - 1; kk++) {
        read(slot, kk + 1);
        multiply(kk);
      }
      meet(s + NST - 1 < last);
      if (s + NST < last) fetch(s + NST, slot);
      slot = slot == NST - 1 ? 0 : slot + 1;
      if (s + 1 < last) read(slot, 0);
      multiply(KK - 1);
    }
  }
  // lane: row lo of tile j, columns 4 hi .. of tile i
#pragma unroll
  for (int j = 0; j < MT; j++) {
    const int m = (wm * MT + j) * 16 + lo;
    if (m >= a.M) continue;
    if constexpr (OUT == GLU) {
#pragma unroll
      for (int i = 0; i < NT; i += 2) {
        const int n = n0 + (wn * NT + i) * 8 + hi * 4;
        if (n >= a.N) continue;
        short4_t o;
#pragma unroll
        for (int r = 0; r < 4; r++)
          o[r] = f32_to_bf16(skinny::silu(acc[i][j][r]) * acc[i + 1][j][r]);
        *reinterpret_cast<short4_t*>(a.out + (int64_t)m * a.N + n) = o;
      }
    } else {
#pragma unroll
      for (int i = 0; i < NT; i++) {
        const int n = n0 + (wn * NT + i) * 16 + hi * 4;
        if (n >= a.N) continue;
        if constexpr (OUT == PARTIAL) {
          *reinterpret_cast<f32x4*>(
              a.part + ((int64_t)split * a.M + m) * a.N + n) = acc[i][j];
        } else {
          short4_t o;
#pragma unroll
          for (int r = 0; r < 4; r++)
            o[r] = f32_to_bf16(acc[i][j][r] +
                               (a.bias ? bf16_to_f32(a.bias[n + r]) : 0.f));
          *reinterpret_cast<short4_t*>(a.out + (int64_t)m * a.N + n) = o;
        }
      }
    }
  }
}

template <int WM, int MT, int NT, int BK, int OUT>
__global__ __launch_bounds__(THREADS, 2) void batch_linear_kernel(
    const BatchArgs a) {
  using T = Tile<WM, MT, NT, BK>;
  __shared__ __attribute__((aligned(128))) short lds[T::NST * T::STAGE];
  batch_tile<WM, MT, NT, BK, OUT>(a, lds);
}

// out = the splits' sum, in order (+ bias)
__global__ __launch_bounds__(256) void batch_sum_kernel(
    short* __restrict__ out, const float* __restrict__ part,
    const short* __restrict__ bias, const int splits, const int64_t total,
    const int N) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(part + i);
  for (int s = 1; s < splits; s++)
    v += *reinterpret_cast<const f32x4*>(part + s * total + i);
  short4_t o;
#pragma unroll
  for (int r = 0; r < 4; r++)
    o[r] = f32_to_bf16(v[r] + (bias ? bf16_to_f32(bias[i % N + r]) : 0.f));
  *reinterpret_cast<short4_t*>(out + i) = o;
}

// Calls go(kernel, its columns) with the kernel for M rows and `cols` columns
template <int OUT, typename Go>
void with_kernel(int M, int K, int cols, const Go& go) {
  const bool wide = K % 128 == 0;   // K steps of 128 for few rows
  if (cols == 64) {
    if constexpr (OUT != GLU)
      if (M <= 32 && wide) return go(batch_linear_kernel<2, 1, 1, 128, OUT>);
    if (M <= 64) return go(batch_linear_kernel<4, 1, 2, 64, OUT>);
    if (M <= 128) return go(batch_linear_kernel<4, 2, 2, 64, OUT>);
    if (M <= 192) return go(batch_linear_kernel<4, 3, 2, 64, OUT>);
    return go(batch_linear_kernel<4, 4, 2, 64, OUT>);
  }
  if constexpr (OUT != GLU)
    if (M <= 16 && wide) return go(batch_linear_kernel<1, 1, 1, 128, OUT>);
  if (M <= 32 && wide) return go(batch_linear_kernel<2, 1, 2, 128, OUT>);
  if (M <= 64) return go(batch_linear_kernel<4, 1, 4, 64, OUT>);
  if (M <= 128) return go(batch_linear_kernel<4, 2, 4, 64, OUT>);
  if (M <= 192) return go(batch_linear_kernel<4, 3, 4, 64, OUT>);
  return go(batch_linear_kernel<4, 4, 4, 64, OUT>);
}

struct Plan {
  int cols, splits;
};

// The plan with the least time by what was measured: staging at 52 B/ns per CU (one
// workgroup each), W at 5.5 TB/s over the chip, the two overlapping in part, 4 us
// per round of workgroups, 3 for the second launch, whose sums move at 4 TB/s. Up to
// 32 rows count as 32 also where the tile holds 64: rows past the last are one
// line's reads (with 64 of them 4096 x 2880 at 17 rows would take 128 x 8, 12.1 us
// where 64 x 4 takes 10.8). Against the best of cols 64 and 128 with 1 to 16 splits,
// 22 sizes of 9 to 256 rows: within 8 % but for 65 rows, which count as 128 (to
// 25 %), 2048 x 11008 below 17 rows (17 %) and 8192 x 2880 and 8192 x 7232 at 17 (29
// and 10 %). 4096 x 14336: 128 x 8 at 64 rows 30.0 us, 64 x 4 28.7; at 256 rows 47.3.
Plan plan_for(int64_t M, int64_t N, int64_t K, bool glu) {
  const int64_t steps = K / 64;
  Plan best{64, 1};
  double least = 1e30;
  for (int cols = 64; cols <= 128; cols += 64) {
    const int64_t rows = M <= 16 && cols == 128 && !glu ? 16
        : M <= 32 ? 32 : (M + 63) / 64 * 64;
    const int64_t own = glu ? cols / 2 : cols, tiles = (N + own - 1) / own;
    const int64_t most = glu ? 1 : std::min<int64_t>(16, steps / 4);
    for (int64_t s = 1; s == 1 || (s <= most && tiles * s <= 512); s++) {
      const int64_t rounds = (tiles * s + 255) / 256;
      const double staged =
          rounds * ((steps + s - 1) / s) * (rows + cols) * 128 / 52e3;
      const double streamed = (glu ? 2. : 1.) * N * K * 2 / 5.5e6;
      const double us = std::sqrt(staged * staged + streamed * streamed) +
          4 * rounds + (s > 1 ? 3 + s * M * N * 8 / 4e6 : 0);
      if (us < least) {
        least = us;
        best = {cols, (int)s};
      }
    }
  }
  return best;
}

template <int OUT>
void launch(const BatchArgs& a, int cols) {
  const int per = OUT == GLU ? cols / 2 : cols;
  with_kernel<OUT>(a.M, a.K, cols, [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((a.N + per - 1) / per * a.splits),
                       dim3(THREADS), 0, at::hip::getCurrentHIPStream(), a);
  });
}

}  // namespace

static BatchArgs batch_args(const at::Tensor& x, const at::Tensor& w, bool glu) {
  for (const auto& t : {x, w})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 && t.dim() == 2 &&
                t.stride(1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0);
  BatchArgs a{};
  TORCH_CHECK(w.size(0) % (glu ? 2 : 1) == 0 && w.size(0) < (1ll << 31) &&
              x.size(0) >= 1 && x.size(0) <= 256 && w.size(1) < (1ll << 31));
  a.M = (int)x.size(0);
  a.N = (int)(w.size(0) / (glu ? 2 : 1));
  a.K = (int)w.size(1);
  a.x_stride = x.stride(0);
  TORCH_CHECK(w.is_contiguous() && x.size(1) == a.K &&
              (a.M == 1 || a.x_stride % 8 == 0) && a.K % 64 == 0 && a.K > 0 &&
              a.N % 16 == 0 && (int64_t)a.M * a.x_stride < (1ll << 31) &&
              ((glu ? a.N : 0) + 128ll) * a.K < (1ll << 31));
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  return a;
}

void batch_linear(at::Tensor out, at::Tensor x, at::Tensor w, at::Tensor bias,
                  int64_t cols, int64_t splits, bool glu) {
  BatchArgs a = batch_args(x, w, glu);
  TORCH_CHECK(out.is_cuda() && out.dtype() == at::kBFloat16 && out.dim() == 2 &&
              out.is_contiguous() && (uintptr_t)out.data_ptr() % 16 == 0 &&
              out.size(0) == a.M && out.size(1) == a.N);
  const bool has_bias = bias.numel() > 0;
  TORCH_CHECK(!has_bias || (!glu && bias.is_cuda() && bias.is_contiguous() &&
                            bias.dtype() == at::kBFloat16 &&
                            bias.numel() == a.N));
  if (a.N == 0) return;
  if (cols == 0) {
    const Plan p = plan_for(a.M, a.N, a.K, glu);
    cols = p.cols;
    splits = p.splits;
  }
  TORCH_CHECK((cols == 64 || cols == 128) && splits >= 1 &&
              splits <= a.K / 64 && !(glu && splits > 1));
  a.out = (short*)out.data_ptr();
  a.bias = has_bias ? (const short*)bias.data_ptr() : nullptr;
  a.splits = (int)splits;
  if (glu) return launch<GLU>(a, cols);
  if (splits == 1) return launch<BF16>(a, cols);
  const at::Tensor part = at::empty({splits, a.M, a.N},
                                    out.options().dtype(at::kFloat));
  a.part = part.data_ptr<float>();
  launch<PARTIAL>(a, cols);
  const int64_t total = (int64_t)a.M * a.N;
  hipLaunchKernelGGL(batch_sum_kernel, dim3((total + 1023) / 1024), dim3(256),
                     0, at::hip::getCurrentHIPStream(), a.out, a.part, a.bias,
                     a.splits, total, a.N);
}

// The splits' sums [splits, M, N] f32 of batch_linear's plan; empty if it has one
at::Tensor batch_parts(at::Tensor x, at::Tensor w) {
  BatchArgs a = batch_args(x, w, false);
  const Plan p = plan_for(a.M, a.N, a.K, false);
  const auto f32 = x.options().dtype(at::kFloat);
  if (a.N == 0 || p.splits == 1) return at::empty({0}, f32);
  const at::Tensor part = at::empty({p.splits, a.M, a.N}, f32);
  a.part = part.data_ptr<float>();
  a.splits = p.splits;
  launch<PARTIAL>(a, p.cols);
  return part;
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("batch_parts(Tensor x, Tensor w) -> Tensor");
  m.def("batch_linear(Tensor(a!) out, Tensor x, Tensor w, Tensor bias, int cols, int splits, bool glu) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("batch_parts", &kaito::batch_parts);
  m.impl("batch_linear", &kaito::batch_linear);
}
