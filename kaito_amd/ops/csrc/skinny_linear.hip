// Linear layers of decode steps (skinny.h), M <= 32 rows:
//   skinny_linear  out = x W^T (+ bias)
//   skinny_swiglu  out = silu(x Wg^T) * (x Wu^T), W = [Wg | Wu] stacked
//   skinny_norm    either of them of the RMS norm of x + residual
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <type_traits>

namespace kaito {

namespace {

constexpr int NW = 4;

// One product; two of the same K and rows of x (of one x or of two) share a
// launch, the second's workgroups behind the first's.
struct Part {
  short* out;                       // [M, N]
  const short* x;
  int64_t x_stride;
  const short* w;                   // [N, K]; GLU [2 N, K]
  const short* bias;                // [N] or nullptr
  int N;
};
struct Parts {
  Part part[2];
  int first;                        // workgroups (staying ones: tiles) of part 0
  int M, K;
};

// GLU: the wave's two rows are a gate row and its up row (N apart)
template <int M, int R, bool GLU>
KAITO_DEV void linear_rows(short* __restrict__ out,
                           const short* __restrict__ x, const int64_t x_stride,
                           const short* __restrict__ w,
                           const short* __restrict__ bias, const int N,
                           const int K, const int block) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (block * NW + wave) * (GLU ? 1 : R);
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

// A product alone has a kernel of its own: chosen from two by the workgroup it took
// (us) 4.9 where it takes 4.6 (576 x 8192, one row), 15.9 and 14.9 (4096 x 8192, four),
// 6.3 and 6.0 (28672 x 64).
template <int M, int R, bool GLU>
__global__ __launch_bounds__(NW * 64) void skinny_linear_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const int64_t x_stride, const short* __restrict__ w,
    const short* __restrict__ bias, const int, const int N, const int K) {
  linear_rows<M, R, GLU>(out, x, x_stride, w, bias, N, K, blockIdx.x);
}

template <int M, int R>
__global__ __launch_bounds__(NW * 64) void skinny_linear_pair_kernel(
    const Parts a) {
  const int second = (int)blockIdx.x >= a.first;
  const Part p = second ? a.part[1] : a.part[0];
  linear_rows<M, R, false>(p.out, p.x, p.x_stride, p.w, p.bias, p.N, a.K,
                           blockIdx.x - second * a.first);
}

// The products of rms(x + residual) * g, with the sum left for later layers. Each
// workgroup norms the rows for itself, on top of its first weights' way: they are
// asked for behind x and nothing waits for them before the norm is in LDS, and a
// launch of its own, with nothing under way, is saved. Bit for bit what the norm's
// kernel and skinny_linear_kernel leave.
// With the norm's launch, us, two and one (weights out of the caches): 6144 x 4096
// 11.9, 10.5 for one row and 13.6, 11.4 for two, silu * up of 2 x 14336 x 4096 39.3,
// 37.7 and 40.9, 39.0, of 2 x 28672 x 8192 143, 140 and 153, 145, 7680 x 5120 18.0,
// 16.4 and 19.2, 17.3, 1024 x 512 4.6, 2.9 and 5.0, 3.4.
struct NormArgs {
  short* out;                       // [M, N]
  short* sum;                       // [M, K], x + residual
  const short *x, *residual;        // [M, K]
  const short* g;                   // [K]
  const short* w;                   // [N, K]; GLU [2 N, K]
  const short* bias;                // [N] or nullptr
  float eps;
  int N, K;                         // K: 512 n, at most 2048 ITER; WHOLE: that
};

// until this wave's reads and writes of LDS are done, and those of all waves;
// loads stay under way
KAITO_DEV void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int M, int R, int ITER, bool WHOLE, bool GLU>
__global__ __launch_bounds__(NW * 64) void skinny_norm_kernel(
    const NormArgs a) {
  using skinny::hbf16x8;
  constexpr int U = 4;              // loads of a row under way, 2048 k
  __shared__ __attribute__((aligned(16))) short xs[M][ITER * 2048];
  __shared__ float red[M][NW];
  const int N = a.N, K = WHOLE ? ITER * 2048 : a.K, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * NW + wave) * (GLU ? 1 : R);
  const int at = threadIdx.x * 8;
  short8_t v[M][ITER], u[M][ITER], g[ITER];
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = min(i * 2048 + at, K - 8);
#pragma unroll
    for (int m = 0; m < M; m++) {
      v[m][i] = *reinterpret_cast<const short8_t*>(a.x + m * K + c);
      u[m][i] = *reinterpret_cast<const short8_t*>(a.residual + m * K + c);
    }
    g[i] = *reinterpret_cast<const short8_t*>(a.g + c);
  }
  __builtin_amdgcn_sched_barrier(0);
  const short* wp[R];
  float acc[M][R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    wp[r] = a.w + (int64_t)(GLU ? r * N + min(n0, N - 1)
                                : min(n0 + r, N - 1)) * K + lane * 8;
#pragma unroll
    for (int m = 0; m < M; m++) acc[m][r] = 0.f;
  }
  hbf16x8 w[2][U][R];
  auto fetch = [&](const int k0, const int b) {
#pragma unroll
    for (int j = 0; j < U; j++)
#pragma unroll
      for (int r = 0; r < R; r++)
        if (k0 + j * 512 < K)       // uniform
          w[b][j][r] = skinny::load_stream<hbf16x8>(wp[r] + k0 + j * 512);
  };
  fetch(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  float ss[M];
#pragma unroll
  for (int m = 0; m < M; m++) {
    ss[m] = 0.f;
#pragma unroll
    for (int i = 0; i < ITER; i++) {
      if (i * 2048 + at >= K) break;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        v[m][i][j] = f32_to_bf16(bf16_to_f32(v[m][i][j]) +
                                 bf16_to_f32(u[m][i][j]));
        const float f = bf16_to_f32(v[m][i][j]);
        ss[m] += f * f;
      }
    }
    ss[m] = wave_reduce_sum(ss[m]);
    if (lane == 0) red[m][wave] = ss[m];
  }
  lds_barrier();
#pragma unroll
  for (int m = 0; m < M; m++) {
    const float s = (red[m][0] + red[m][1]) + (red[m][2] + red[m][3]);
    const float inv = rsqrtf(s / (float)K + a.eps);
#pragma unroll
    for (int i = 0; i < ITER; i++) {
      const int c = i * 2048 + at;
      if (c >= K) break;
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; j++)
        o[j] = f32_to_bf16(bf16_to_f32(v[m][i][j]) * inv * bf16_to_f32(g[i][j]));
      *reinterpret_cast<short8_t*>(&xs[m][c]) = o;
      if (blockIdx.x == 0)
        *reinterpret_cast<short8_t*>(a.sum + m * K + c) = v[m][i];
    }
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int k0 = i * 2048;
    if (k0 >= K) break;             // uniform
    if (i + 1 < ITER) fetch(k0 + 2048, (i + 1) & 1);
#pragma unroll
    for (int j = 0; j < U; j++) {
      if (k0 + j * 512 >= K) break;
#pragma unroll
      for (int m = 0; m < M; m++) {
        const hbf16x8 xv = skinny::load_x(&xs[m][k0 + j * 512 + lane * 8]);
#pragma unroll
        for (int r = 0; r < R; r++)
          acc[m][r] = skinny::dot8(w[i & 1][j][r], xv, acc[m][r]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < M; m++) {
#pragma unroll
    for (int r = 0; r < R; r++) acc[m][r] = wave_reduce_sum(acc[m][r]);
    if constexpr (GLU) {
      if (lane == 0 && n0 < N)
        a.out[(int64_t)m * N + n0] =
            f32_to_bf16(skinny::silu(acc[m][0]) * acc[m][1]);
    } else {
#pragma unroll
      for (int r = 0; r < R; r++)
        if (lane == 0 && n0 + r < N)
          a.out[(int64_t)m * N + n0 + r] = f32_to_bf16(
              acc[m][r] + (a.bias ? bf16_to_f32(a.bias[n0 + r]) : 0.f));
    }
  }
}

// M <= 16 MT rows; N is a multiple of 16 (GLU: of 8, the workgroup's 16 rows
// are 8 gate rows and their up rows, N apart), K of the stage
template <int MT, int KS, bool GLU>
KAITO_DEV void linear_tile(short* __restrict__ out,
                           const short* __restrict__ x, const int64_t x_stride,
                           const short* __restrict__ w,
                           const short* __restrict__ bias, const int M,
                           const int N, const int K, const int block) {
  constexpr int NI = skinny::tile_loads<KS>();
  __shared__ __attribute__((aligned(128))) short ring[4][2][16 * KS];
  static_assert(sizeof(ring) >= 4 * MT * 64 * sizeof(f32x4), "fold");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = block * (GLU ? 8 : 16);
  const short *src[NI], *xp[MT];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int r = skinny::tile_row<KS>(j, lane);
    const int64_t n = GLU ? n0 + r % 8 + (r >= 8 ? N : 0) : n0 + r;
    src[j] = w + n * K + skinny::tile_col<KS>(j, lane);
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
    xp[mt] = x + min(mt * 16 + (lane & 15), M - 1) * x_stride +
        (lane >> 4) * 8;
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  skinny::stream_tile<MT, KS>(acc, src, xp, ring[wave][0], K, wave, lane);
  __syncthreads();                  // every wave is done with its stages
  f32x4* red = reinterpret_cast<f32x4*>(&ring[0][0][0]);
#pragma unroll
  for (int mt = 0; mt < MT; mt++) red[(wave * MT + mt) * 64 + lane] = acc[mt];
  __syncthreads();
  // slot: tile mt, lane l: rows 16 mt + 4 (l >> 4) .. of column l & 15
  if (threadIdx.x >= MT * 64) return;
  const int slot = threadIdx.x, l = slot & 63, c = l & 15;
  if (GLU && c >= 8) return;
  f32x4 v = skinny::fold<MT, 4>(red, slot);
  if constexpr (GLU) {
    const f32x4 u = skinny::fold<MT, 4>(red, slot + 8);
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = skinny::silu(v[r]) * u[r];
  } else if (bias) {
    v += bf16_to_f32(bias[n0 + c]);
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int m = (slot >> 6) * 16 + (l >> 4) * 4 + r;
    if (m < M) out[(int64_t)m * N + n0 + c] = f32_to_bf16(v[r]);
  }
}

template <int MT, int KS, bool GLU>
__global__ __launch_bounds__(256, 2) void skinny_tile_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const int64_t x_stride, const short* __restrict__ w,
    const short* __restrict__ bias, const int M, const int N, const int K) {
  linear_tile<MT, KS, GLU>(out, x, x_stride, w, bias, M, N, K, blockIdx.x);
}

template <int MT, int KS>
__global__ __launch_bounds__(256, 2) void skinny_tile_pair_kernel(
    const Parts a) {
  const int second = (int)blockIdx.x >= a.first;
  const Part p = second ? a.part[1] : a.part[0];
  linear_tile<MT, KS, false>(p.out, p.x, p.x_stride, p.w, p.bias, a.M, p.N,
                             a.K, blockIdx.x - second * a.first);
}

// K = 1024 S: see skinny::stream_tiles. gridDim.x workgroups share the tiles of
// both parts, which have one x.
template <int MT, int S, bool GLU, bool TWO>
__global__ __launch_bounds__(256, 2) void skinny_tiles_kernel(const Parts a) {
  constexpr int KS = skinny::TILES_KS, TW = skinny::TILE_NW;
  constexpr int COLS = GLU ? 8 : 16;
  __shared__ __attribute__((aligned(128))) short ring[TW][2][16 * KS];
  __shared__ f32x4 red[2][TW][MT * 64];
  const Part p = a.part[0], p2 = a.part[TWO];
  const int M = a.M, K = a.K, first = a.first;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = threadIdx.x, l = slot & 63, c = l & 15;
  const bool mine = slot < MT * 64 && !(GLU && c >= 8);
  skinny::stream_tiles<MT, S, TWO>(
      p.w, p2.w, first,
      [&](const int j) {
        const int r = skinny::tile_row<KS>(j, lane);
        const uint32_t n = GLU ? r % 8 + (r >= 8 ? p.N : 0) : r;
        return (n * K + skinny::tile_col<KS>(j, lane)) * 2;
      },
      COLS * K * 2, blockIdx.x, gridDim.x, first + (TWO ? p2.N / COLS : 0),
      [&](const short* (&xp)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          xp[mt] = p.x + min(mt * 16 + (lane & 15), M - 1) * p.x_stride +
              (lane >> 4) * 8;
      },
      ring[wave][0], &red[0][0][0], wave, lane,
      [&](const int t, const f32x4* sums) {
        if (!mine) return;
        const bool second = TWO && t >= first;
        const int N = second ? p2.N : p.N;
        const short* bias = second ? p2.bias : p.bias;
        short* out = second ? p2.out : p.out;
        const int n = (second ? t - first : t) * COLS + c;
        f32x4 v = skinny::fold<MT, TW>(sums, slot);
        if constexpr (GLU) {
          const f32x4 u = skinny::fold<MT, TW>(sums, slot + 8);
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] = skinny::silu(v[r]) * u[r];
        } else if (bias) {
          v += bf16_to_f32(bias[n]);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int m = (slot >> 6) * 16 + (l >> 4) * 4 + r;
          if (m < M) out[(int64_t)m * N + n] = f32_to_bf16(v[r]);
        }
      });
}

constexpr int MAX_M = 32;

// Rows of W streamed whole, or tiles of 16 through LDS? Beyond 4 rows of x
// tiles. 3 and 4 rows are about even while W is small and tile counts go
// unevenly on 256 CUs (5120 x 5120 at 4 rows: 13.6 us, 14.5 in tiles; 4096 x
// 4096 9.2, 8.7); beyond 2^25 weights the row kernel's sums are the bound
// (28672 x 4096: 49.4, 41.7; 128256 x 4096: 217, 164).
bool in_tiles(int64_t M, int64_t N, int64_t K, int64_t cols, int64_t weights) {
  return M > 4 || (M > 2 && weights > (1ll << 25) && K % 64 == 0 &&
                   N % cols == 0);
}

// Tiles handed to workgroups that stay, a CU each, or to one workgroup per tile?
// From three tiles per CU on (us, per tile and staying; 2048 columns: 448 tiles
// 8.9 and 9.2, 512 of a pair 8.9 and 9.5, 768 13.1 and 12.6 at M = 5, 15.5 and
// 13.6 at 16, 19.4 and 15.9 at 32, 2000 44.1 and 29.6 at 32; 4096 columns: 384
// 13.8 and 14.0, 1792 of a pair 40.2 and 39.3 at 5, 48.5 and 41.8 at 16, 8016
// 209 and 168 at 16). Beyond 16 rows, whose x costs twice as much to bring, as
// soon as a tile per CU is not enough (M = 32: 256 tiles 8.9 and 9.6, 322 13.3
// and 11.4, 384 13.6 and 11.9, 512 14.5 and 12.8; M = 17: 322 11.0 and 10.4). Two
// workgroups per CU are no faster (1792 of a pair 42.8).
constexpr int WORKGROUPS = 256;

bool many_tiles(int M, int64_t tiles, int64_t weights, int64_t K) {
  return tiles >= (M > 16 ? WORKGROUPS + 64 : 3 * WORKGROUPS) &&
         weights < (1ll << 31) && (K == 2048 || (K == 4096 && M <= 16));
}

void check(const at::Tensor& out, const at::Tensor& x, const at::Tensor& w,
           int64_t N, int64_t cols) {
  for (const auto& t : {out, x, w})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 && t.dim() == 2 &&
                t.stride(1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(w.is_contiguous() && out.is_contiguous() &&
              x.size(1) == w.size(1) && out.size(0) == x.size(0) &&
              out.size(1) == N);
  const int64_t M = x.size(0), K = w.size(1);
  TORCH_CHECK(M >= 1 && M <= MAX_M && K % 8 == 0 && K > 0 &&
              (M == 1 || x.stride(0) % 8 == 0) && w.size(0) < (1ll << 31) &&
              K < (1ll << 31));
  TORCH_CHECK(M <= 4 || (K % 64 == 0 && N % cols == 0),
              "more than 4 rows: K in whole stages, N in whole tiles");
}

template <int V> using Int = std::integral_constant<int, V>;

template <typename Kernel>
void launch(Kernel kernel, int64_t workgroups, const Parts& a) {
  hipLaunchKernelGGL(kernel, dim3(workgroups),
                     dim3(256), 0, at::hip::getCurrentHIPStream(), a);
}

// a product alone
template <typename Kernel>
void launch_one(Kernel kernel, int64_t workgroups, const Parts& a) {
  const Part& p = a.part[0];
  hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), p.out, p.x, p.x_stride,
                     p.w, p.bias, a.M, p.N, a.K);
}

// `cols` output columns of a tile or, GLU, half of its 16 rows of W
template <bool GLU>
void run(Parts a, bool shared_x) {
  constexpr int cols = GLU ? 8 : 16;
  const int64_t K = a.K, N0 = a.part[0].N, N1 = a.part[1].N, N = N0 + N1;
  const int64_t weights = (GLU ? 2 : 1) * N * K;
  const int M = a.M;
  if (in_tiles(M, N0 % cols ? N0 : N, K, cols, weights)) {
    a.first = (int)(N0 / cols);
    if (shared_x && many_tiles(M, N / cols, weights, K)) {
      auto stay = [&](auto two) {
        constexpr bool TWO = decltype(two)::value;
        if (K == 4096)
          launch(&skinny_tiles_kernel<1, 4, GLU, TWO>, WORKGROUPS, a);
        else if (M > 16)
          launch(&skinny_tiles_kernel<2, 2, GLU, TWO>, WORKGROUPS, a);
        else
          launch(&skinny_tiles_kernel<1, 2, GLU, TWO>, WORKGROUPS, a);
      };
      if (GLU || N1 == 0) stay(std::false_type{});
      else stay(std::bool_constant<!GLU>{});
      return;
    }
    auto tile = [&](auto mt, auto ks) {
      constexpr int MT = decltype(mt)::value, KS = decltype(ks)::value;
      if constexpr (!GLU)
        if (N1 > 0)
          return launch(&skinny_tile_pair_kernel<MT, KS>, N / cols, a);
      launch_one(&skinny_tile_kernel<MT, KS, GLU>, N / cols, a);
    };
    if (M > 16) {
      if (K % 256 == 0) tile(Int<2>{}, Int<256>{});
      else tile(Int<2>{}, Int<64>{});
    } else {
      if (K % 256 == 0) tile(Int<1>{}, Int<256>{});
      else tile(Int<1>{}, Int<64>{});
    }
    return;
  }
  // one row per wave keeps most waves under way for a single x row (N =
  // 4096, K = 4096: 6.6 us against 6.8 with two); with more, two rows share
  // the x loads (M = 4, N = 28672: 48 us)
  const int64_t per = NW * (GLU || M == 1 ? 1 : 2);
  a.first = (int)((N0 + per - 1) / per);
  auto rows = [&](auto m, auto r) {
    constexpr int MM = decltype(m)::value, R = decltype(r)::value;
    if constexpr (!GLU)
      if (N1 > 0)
        return launch(&skinny_linear_pair_kernel<MM, R>,
                      a.first + (N1 + per - 1) / per, a);
    launch_one(&skinny_linear_kernel<MM, R, GLU>, a.first, a);
  };
  switch (M) {
    case 1: rows(Int<1>{}, Int<GLU ? 2 : 1>{}); break;
    case 2: rows(Int<2>{}, Int<2>{}); break;
    case 3: rows(Int<3>{}, Int<2>{}); break;
    default: rows(Int<4>{}, Int<2>{}); break;
  }
}

Part part_of(const at::Tensor& out, const at::Tensor& x, const at::Tensor& w,
             int64_t N) {
  return {(short*)out.data_ptr(), (const short*)x.data_ptr(), x.stride(0),
          (const short*)w.data_ptr(), nullptr, (int)N};
}

Part part_of(const at::Tensor& out, const at::Tensor& x, const at::Tensor& w,
             const at::Tensor& bias) {
  const int64_t N = w.size(0);
  Part p = part_of(out, x, w, N);
  if (bias.numel() > 0) {
    TORCH_CHECK(bias.is_cuda() && bias.is_contiguous() &&
                bias.dtype() == at::kBFloat16 && bias.numel() == N);
    p.bias = (const short*)bias.data_ptr();
  }
  return p;
}

}  // namespace

void skinny_linear(at::Tensor out, at::Tensor x, at::Tensor w,
                   at::Tensor bias) {
  const int64_t N = w.size(0);
  check(out, x, w, N, 16);
  if (N == 0) return;
  Parts a{};
  a.part[0] = part_of(out, x, w, bias);
  a.M = (int)x.size(0);
  a.K = (int)w.size(1);
  run<false>(a, true);
}

// two products of as many rows and the same K in one launch
void skinny_linear_pair(at::Tensor out, at::Tensor x, at::Tensor w,
                        at::Tensor bias, at::Tensor out2, at::Tensor x2,
                        at::Tensor w2, at::Tensor bias2) {
  const int64_t N = w.size(0), N2 = w2.size(0);
  check(out, x, w, N, 16);
  check(out2, x2, w2, N2, 16);
  TORCH_CHECK(x2.size(0) == x.size(0) && w2.size(1) == w.size(1) &&
              N % 16 == 0 && N2 % 16 == 0 && N > 0 && N2 > 0 &&
              N + N2 < (1ll << 31));
  Parts a{};
  a.part[0] = part_of(out, x, w, bias);
  a.part[1] = part_of(out2, x2, w2, bias2);
  a.M = (int)x.size(0);
  a.K = (int)w.size(1);
  run<false>(a, x.data_ptr() == x2.data_ptr() && x.stride(0) == x2.stride(0));
}

// of rms(x + residual) * g; sum: x + residual, not one of the others
void skinny_norm(at::Tensor out, at::Tensor sum, at::Tensor x,
                 at::Tensor residual, at::Tensor g, double eps, at::Tensor w,
                 at::Tensor bias, bool glu) {
  TORCH_CHECK(!glu || (w.dim() == 2 && w.size(0) % 2 == 0 && bias.numel() == 0));
  const int64_t N = glu ? w.size(0) / 2 : w.size(0);
  check(out, x, w, N, 1);
  const int64_t M = x.size(0), K = w.size(1);
  for (const auto& t : {x, residual, sum})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.sizes() == x.sizes() &&
                t.dtype() == at::kBFloat16 && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(g.is_cuda() && g.is_contiguous() && g.numel() == K &&
              g.dtype() == at::kBFloat16 && (uintptr_t)g.data_ptr() % 16 == 0);
  TORCH_CHECK(M <= 2 && K % 512 == 0 && K <= 8192 &&
              sum.data_ptr() != residual.data_ptr() &&
              sum.data_ptr() != x.data_ptr());
  if (N == 0) return;
  const Part p = part_of(out, x, w, bias);
  const NormArgs a = {p.out, (short*)sum.data_ptr(), p.x,
                      (const short*)residual.data_ptr(),
                      (const short*)g.data_ptr(), p.w, p.bias, (float)eps,
                      (int)N, (int)K};
  auto run_norm = [&](auto m, auto r, auto is_glu) {
    constexpr int MM = decltype(m)::value, R = decltype(r)::value;
    constexpr bool GLU = decltype(is_glu)::value;
    const int64_t per = NW * (GLU ? 1 : R);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((N + per - 1) / per), dim3(NW * 64), 0,
                         at::hip::getCurrentHIPStream(), a);
    };
    auto iter = [&](auto whole) {
      constexpr bool WHOLE = decltype(whole)::value;
      if (K <= 2048) go(&skinny_norm_kernel<MM, R, 1, WHOLE, GLU>);
      else if (K <= 4096) go(&skinny_norm_kernel<MM, R, 2, WHOLE, GLU>);
      else if (K <= 6144) go(&skinny_norm_kernel<MM, R, 3, WHOLE, GLU>);
      else go(&skinny_norm_kernel<MM, R, 4, WHOLE, GLU>);
    };
    if (K % 2048) iter(std::false_type{});
    else iter(std::true_type{});
  };
  using std::integral_constant;
  const integral_constant<int, 1> one;
  const integral_constant<int, 2> two;
  if (glu) {
    if (M == 1) run_norm(one, two, std::true_type{});
    else run_norm(two, two, std::true_type{});
  } else {
    if (M == 1) run_norm(one, one, std::false_type{});
    else run_norm(two, two, std::false_type{});
  }
}

void skinny_swiglu(at::Tensor out, at::Tensor x, at::Tensor w) {
  TORCH_CHECK(w.size(0) % 2 == 0);
  const int64_t N = w.size(0) / 2;
  check(out, x, w, N, 8);
  if (N == 0) return;
  Parts a{};
  a.part[0] = part_of(out, x, w, N);
  a.M = (int)x.size(0);
  a.K = (int)w.size(1);
  run<true>(a, true);
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("skinny_linear(Tensor(a!) out, Tensor x, Tensor w, Tensor bias) -> ()");
  m.def("skinny_linear_pair(Tensor(a!) out, Tensor x, Tensor w, Tensor bias, Tensor(b!) out2, Tensor x2, Tensor w2, Tensor bias2) -> ()");
  m.def("skinny_norm(Tensor(a!) out, Tensor(b!) sum, Tensor x, Tensor residual, Tensor g, float eps, Tensor w, Tensor bias, bool glu) -> ()");
  m.def("skinny_swiglu(Tensor(a!) out, Tensor x, Tensor w) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("skinny_linear", &kaito::skinny_linear);
  m.impl("skinny_linear_pair", &kaito::skinny_linear_pair);
  m.impl("skinny_norm", &kaito::skinny_norm);
  m.impl("skinny_swiglu", &kaito::skinny_swiglu);
}
