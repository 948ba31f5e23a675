// W4A16 group-quantized linear kernels (AWQ/GPTQ-class presets; the catalog
// carries qwen3-8b-awq etc.).
//
// Native layout (loaders repack AWQ checkpoints into this):
//   qweight: uint32 [N, K/8]   8 consecutive K nibbles per word, row-major
//   scales:  float  [N, K/G]   group size G (typ. 128), w = s*q - z
//   zeros:   float  [N, K/G]   z folded as s*zq at repack time
//
// Two paths:
//   w4a16_gemv    : M <= 32 decode shapes. Memory-bound on the 4-bit
//                   weights (N*K/2 bytes vs 2*N*K for bf16 -> ~4x less
//                   traffic than a bf16 GEMM at small M); skinny.h.
//   w4a16_dequant : tile dequant to bf16 scratch; large-M callers then run
//                   the scratch through hipBLASLt MFMA (dequant is
//                   O(N*K) against the GEMM's O(M*N*K) -> noise at M>=128).
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <algorithm>

namespace kaito {

// ---------------------------------------------------------------- gemv
// M <= 4: a wave streams whole rows of packed weights, two or four of them
// against the same x. One row of x: 14.9 us for N = 28672, K = 4096 (66 MB
// with the scales: 4.4 TB/s), 10.6 for 4096 x 14336, 4.3 for 4096 x 4096; with
// more rows the vector unit is the bound (M = 2: 18.9, 13.2, 5.5 us). Lanes
// with 64 k of one row that turned nibbles into f32 one by one took 36.2,
// 19.1, 6.6 and 62.6, 32.0, 10.3 us; nibbles as bf16 128 + q, which cost the
// sums 4 bits, 16.3, 11.3, 4.5 and 25.0, 16.6, 6.3.
template <int M, int R>
__global__ __launch_bounds__(256) void w4a16_stream_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const uint32_t* __restrict__ qw, const float* __restrict__ scales,
    const float* __restrict__ zeros, int N, int K, int group) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * 4 + wave) * R;
  if (n0 >= N) return;
  const uint32_t* wp[R];
  const float *sc[R], *ze[R];
  float acc[M][R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int64_t n = min(n0 + r, N - 1);
    wp[r] = qw + n * (K >> 3);
    sc[r] = scales + n * (K / group);
    ze[r] = zeros + n * (K / group);
#pragma unroll
    for (int m = 0; m < M; m++) acc[m][r] = 0.f;
  }
  skinny::stream_rows_w4<M, R>(acc, wp, sc, ze, x, K, K, group, lane);
#pragma unroll
  for (int m = 0; m < M; m++)
#pragma unroll
    for (int r = 0; r < R; r++) {
      const float v = wave_reduce_sum(acc[m][r]);
      if (lane == 0 && n0 + r < N) out[(int64_t)m * N + n0 + r] = f32_to_bf16(v);
    }
}

// 5 <= M <= 32: the same weights as MFMA operands, 16 rows per workgroup,
// the waves over K
template <int MT, int NT, int WORDS>
__global__ __launch_bounds__(256) void w4a16_mfma_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const uint32_t* __restrict__ qw, const float* __restrict__ scales,
    const float* __restrict__ zeros, int M, int N, int K, int group) {
  constexpr int TILES = MT * NT, NW = 4;
  __shared__ f32x4 red[NW * TILES * 64];
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * NT;
  const uint32_t* wp[NT];
  const float *sc[NT], *ze[NT];
  const short* xp[MT];
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const int64_t n = min(n0 + j * 16 + lo, N - 1);
    wp[j] = qw + n * (K >> 3) + hi * WORDS;
    sc[j] = scales + n * (K / group);
    ze[j] = zeros + n * (K / group);
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
    xp[mt] = x + (int64_t)min(mt * 16 + lo, M - 1) * K + hi * 8 * WORDS;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  skinny::accumulate_w4<MT, NT, WORDS>(acc, wp, sc, ze, xp, K, group, wave,
                                       NW);
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int j = 0; j < NT; j++)
      red[(wave * TILES + j * MT + mt) * 64 + lane] = acc[mt][j];
  __syncthreads();
  for (int slot = threadIdx.x; slot < TILES * 64; slot += NW * 64) {
    const f32x4 v = skinny::fold<TILES, NW>(red, slot);
    const int tile = slot / 64, l = slot % 64, mt = tile % MT;
    const int n = n0 + tile / MT * 16 + (l & 15);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = mt * 16 + (l >> 4) * 4 + r;
      if (m < M && n < N) out[(int64_t)m * N + n] = f32_to_bf16(v[r]);
    }
  }
}

// ---------------------------------------------------------------- tiles
// Few rows of x, kept in LDS: a workgroup per CU that goes from tile to tile of
// 16 rows of W, its eight waves over K, each with a ring of its own through which
// 512 k of a tile (4 KB of nibbles, 256 contiguous bytes of a row, and the rows'
// scales and zeros) arrive by direct loads, up to DEPTH stages under way. A lane's
// 16 bytes are 32 k of one group, four operands of v_mfma_f32_16x16x32_bf16, so
// that a nibble is unpacked once and multiplied with every row of x on the matrix
// unit. x lies in the unpacked nibbles' order, beside its sums over the groups.
// Bound by the chain of a tile, with two waves per SIMD to cover it: wait, unpack
// (232 vector instructions per stage), multiply, meet at a barrier, sum. 28672 x
// 4096, 2 rows: vector unit busy 31 %, matrix cores 9, LDS 16, 3.8 TB/s; of the
// waves' time 38 % waits for loads and barriers, 30 for issue. Hence, from 512 tiles
// on, two workgroups of four waves per CU, whose barriers do not meet: 12288 x 4096,
// 2 rows, 10.4 -> 9.2 us, 28672 x 2560 13.2 -> 11.5, as a pair 28672 x 4096 15.9 ->
// 14.8, with the norm 16.8 -> 15.6 (57344 x 8192 44.6 both; fewer tiles the same or
// slower). x is asked for ahead of the weights, behind which its loads would end:
// 4096 x 14336 11.2 -> 9.7, 28672 x 4096 as a pair, 5 rows, 17.3 -> 16.0. Little of it
// is not: 8 loads of a thread, most of them of nothing new, hold the weights up for
// longer than x behind them takes (2 rows, pairs, x ahead and behind, 2048 x 2048 4.9
// and 4.5, 4096 x 1024 4.9 and 4.5, 7168 x 2048 6.4 and 6.1, one row of 4096 x 4096 5.7
// and 5.4, 16 of 4096 x 512 5.3 and 4.9, but 16 of 4096 x 2048 6.6 and 6.9, 6144 x 4096
// 7.4 and 7.8; asked for only where there is some: 5.1, 4.7, and 5.9 -> 6.2 of 8704 x
// 2048, as the waits count for either). The wave
// that sums by turns: no change. The time hardly grows
// with the rows. us, rows streamed (5 rows and more: MFMA from global memory) and
// tiles before these two, at 1, 2, 3, 4, 8 rows: 28672 x 4096 15.8 19.7 23.6 33.2 37.7 and 16.7 17.4
// 17.4 17.5 18.3; 4096 x 14336 11.4 13.8 and 11.7 11.7 (more rows do not fit); 4096 x
// 4096 4.6 5.7 7.9 8.8 8.7 and 5.9 6.1 6.6 7.0 7.9. Four waves: 20.5 at 2 rows; sums
// of two tiles at a time: no change.
namespace {

constexpr int W4_K = 512;           // k of a stage
constexpr int W4_STAGE = 16 * W4_K / 2 + 2 * 256;
constexpr int W4_LDS = 160 * 1024;  // for 8 waves; for 4 half of it

// bytes behind the rings: sums over the waves (twice), sums of x, x
__host__ __device__ constexpr int w4_red(int waves, int mr) {
  return waves * mr * 4 * 16;
}
inline bool w4_fits(int waves, int depth, int mr, int64_t M, int64_t K) {
  return waves * depth * W4_STAGE + 2 * w4_red(waves, mr) + K / 128 * mr * 4 +
         M * (K * 2 + 16) <= W4_LDS * waves / 8;
}

KAITO_DEV __amdgpu_buffer_rsrc_t w4_buffer(const void* p,
                                           const uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x27000);
}

// The rows are rms(x + residual) * g, with the sum left for later layers: up to 2
// of them, K up to 2048 W4_NORM
struct W4Norm {
  short* sum;                       // [M, K]
  const short *residual, *g;        // [M, K], [K]
  float eps;
};
constexpr int W4_NORM = 4;
constexpr int W4_AHEAD = 8;         // 16-byte parts of x that a thread asks for first

// MR: rows of x that have a place (4 or 16); GLU: N gate rows, then N up rows.
// NORM: four waves norm a row each workgroup for itself, as the norm's kernel does
// and to the same bits, while the first weights are on the way; its launch is
// saved: us, two launches and one, 28672 x 4096 20.1, 17.7 for two rows, 22016 x
// 5120 21.4, 19.1 for one and 22.2, 19.6, 57344 x 8192 48.2, 44.3 and 53.9, 47.0.
template <int NW, int MR, int DEPTH, bool GLU, bool NORM, int AHEAD = W4_AHEAD>
__global__ __launch_bounds__(64 * NW, 2) void w4a16_tiles_kernel(
    short* __restrict__ out, const short* __restrict__ x,
    const uint32_t* __restrict__ qw, const float* __restrict__ scales,
    const float* __restrict__ zeros, const int M, const int N, const int K,
    const W4Norm norm) {
  using skinny::hbf16x8;
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int COLS = GLU ? 8 : 16, LOADS = 6, USED = MR * 4;
  __shared__ __attribute__((aligned(128))) char lds[W4_LDS * NW / 8];
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* ring = lds + wave * DEPTH * W4_STAGE;
  f32x4* red = reinterpret_cast<f32x4*>(lds + NW * DEPTH * W4_STAGE);
  float* xs = reinterpret_cast<float*>(
      lds + NW * DEPTH * W4_STAGE + 2 * w4_red(NW, MR));     // [K / 128][MR]
  short* xl = reinterpret_cast<short*>(xs + K / 128 * MR);  // [M][K + 8]
  const int ntiles = N / COLS, nst = K / W4_K;
  const int spt = (nst + NW - 1) / NW;  // stages of a wave and tile
  if ((int)blockIdx.x >= ntiles) return;

  auto n_of = [&](const int r) {    // row of W of row r of tile 0
    return (uint32_t)(GLU ? r % 8 + (r >= 8 ? N : 0) : r);
  };
  uint32_t wo[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int r = j * 4 + lane / 16;
    wo[j] = n_of(r) * (K / 2) + ((lane % 16) ^ r) * 16;
  }
  const uint32_t so = n_of(lane / 4) * (K / 128) * 4 + lane % 4 * 4;
  int ft = blockIdx.x, fs = 0;      // the next stage to ask for
  auto fetch = [&](const int slot) {
    // past the last stage: loads of nothing, so that the waits stay counts
    const uint32_t all = __builtin_amdgcn_readfirstlane(
        ft < ntiles && fs * NW + wave < nst ? 0xffffffff : 0);
    const auto wr = w4_buffer(qw, all), sr = w4_buffer(scales, all),
               zr = w4_buffer(zeros, all);
    const int k = (fs * NW + wave) * W4_K;
    const uint32_t row = ft * COLS;
    const uint32_t at = __builtin_amdgcn_readfirstlane(row * (K / 2) + k / 2);
    const uint32_t sat =
        __builtin_amdgcn_readfirstlane(row * (K / 128) * 4 + k / 128 * 4);
    char* p = ring + slot * W4_STAGE;
#define W4_COPY(R_, P_, SIZE_, OFF_, AT_, AUX_)                               \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(                                 \
        R_, (__attribute__((address_space(3))) void*)(P_), SIZE_, OFF_, AT_,  \
        0, AUX_)
#pragma unroll
    for (int j = 0; j < 4; j++)
      W4_COPY(wr, p + j * 1024, 16, wo[j], at, 2 /* non-temporal */);
    W4_COPY(sr, p + 4096, 4, so, sat, 0);
    W4_COPY(zr, p + 4352, 4, so, sat, 0);
#undef W4_COPY
    if (++fs == spt) {
      fs = 0;
      ft += gridDim.x;
    }
  };
  // four waves norm a row, of four waves both rows one behind the other
  constexpr int NR = NORM ? 8 / NW : 1;
  const int nm = wave / 4 * NR, nat = (threadIdx.x & 255) * 8;  // row, first k
  short8_t nv[NR][NORM ? W4_NORM : 1], nr[NR][NORM ? W4_NORM : 1],
      ng[NORM ? W4_NORM : 1];
  hbf16x8 xv[NORM || !AHEAD ? 1 : AHEAD];
  // x ahead of the weights: loads end in order
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < W4_NORM; i++) {
      const int k = i * 2048 + nat;
      if (k >= K) break;            // uniform in a wave: K is whole stages
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const int64_t row = (int64_t)min(nm + r, M - 1) * K;
        nv[r][i] = *reinterpret_cast<const short8_t*>(x + row + k);
        nr[r][i] =
            *reinterpret_cast<const short8_t*>(norm.residual + row + k);
      }
      ng[i] = *reinterpret_cast<const short8_t*>(norm.g + k);
    }
  } else {
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      xv[i] = skinny::load_x(
          x + min(i * 64 * NW + (int)threadIdx.x, M * K / 8 - 1) * 8);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < DEPTH; i++) fetch(i);

  // ---- x and its sums over the groups; 16 threads have a group
  if constexpr (NORM) {
    float* const rn = reinterpret_cast<float*>(red);
#pragma unroll
    for (int r = 0; r < NR; r++) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < W4_NORM; i++) {
        if (i * 2048 + nat >= K) break;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          nv[r][i][e] = f32_to_bf16(bf16_to_f32(nv[r][i][e]) +
                                    bf16_to_f32(nr[r][i][e]));
          const float f = bf16_to_f32(nv[r][i][e]);
          ss += f * f;
        }
      }
      ss = wave_reduce_sum(ss);
      if (lane == 0) rn[(nm + r) * 4 + wave % 4] = ss;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);       // weights stay under way
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int m = nm + r;
      const float* s = rn + m * 4;
      const float inv =
          rsqrtf(((s[0] + s[1]) + (s[2] + s[3])) / (float)K + norm.eps);
#pragma unroll
      for (int i = 0; i < W4_NORM; i++) {
        const int k = i * 2048 + nat;
        if (m >= M || k >= K) break;          // uniform in a wave
        hbf16x8 v;
        float sum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          v[e] =
              (__bf16)(bf16_to_f32(nv[r][i][e]) * inv * bf16_to_f32(ng[i][e]));
          sum += (float)v[e];
        }
        sum = group_reduce_sum<16>(sum);
        *reinterpret_cast<hbf16x8*>(xl + m * (K + 8) + k) =
            skinny::nibble_order(v);
        if (nat % 128 == 0) xs[k / 128 * MR + m] = sum;
        if (blockIdx.x == 0)
          *reinterpret_cast<short8_t*>(norm.sum + (int64_t)m * K + k) =
              nv[r][i];
      }
    }
  } else {
    auto place = [&](const int c, const hbf16x8 v) {
      const int m = c / (K / 8), k = c % (K / 8) * 8;
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++) sum += (float)v[e];
      sum = group_reduce_sum<16>(sum);
      *reinterpret_cast<hbf16x8*>(xl + m * (K + 8) + k) =
          skinny::nibble_order(v);
      if (c % 16 == 0) xs[k / 128 * MR + m] = sum;
    };
    int c = threadIdx.x;
#pragma unroll
    for (int i = 0; i < AHEAD; i++, c += 64 * NW)
      if (c < M * K / 8) place(c, xv[i]);     // uniform in 16 lanes
    for (; c < M * K / 8; c += 64 * NW)
      place(c, skinny::load_x(x + (int64_t)c * 8));
  }
  skinny::wait_loads<0>();
  __syncthreads();

  const short* xr = xl + min(lo, M - 1) * (K + 8) + hi * 32;
  // rows past M of a lane's four are not stored
  const float* xsr = xs + (MR == 16 ? 4 * hi : 0);
  int slot = 0, par = 0;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    f32x4 acc{0.f, 0.f, 0.f, 0.f};
    for (int st = 0; st < spt; st++) {
      skinny::wait_loads<(DEPTH - 1) * LOADS>();
      const int k = (st * NW + wave) * W4_K;
      if (k < K) {
        const char* p = ring + slot * W4_STAGE;
        const f32x4 sc = *reinterpret_cast<const f32x4*>(p + 4096 + lo * 16);
        const f32x4 ze = *reinterpret_cast<const f32x4*>(p + 4352 + lo * 16);
        u32x4 w[4];
#pragma unroll
        for (int g = 0; g < 4; g++)
          w[g] = *reinterpret_cast<const u32x4*>(
              p + lo * 256 + ((g * 4 + hi) ^ lo) * 16);
        f32x4 dot[4];
#pragma unroll
        for (int g = 0; g < 4; g++) dot[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int g = 0; g < 4; g++)
            dot[g] = skinny::mfma16(
                skinny::load_x(xr + k + g * 128 + j * 8),
                skinny::nibbles(w[g][j]), dot[g]);
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const f32x4 s =
              *reinterpret_cast<const f32x4*>(xsr + (k / 128 + g) * MR);
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[r] += sc[g] * skinny::NIBBLE * dot[g][r] - ze[g] * s[r];
        }
      }
      // its reads are done before it is overwritten
      __builtin_amdgcn_s_waitcnt(0xc07f);
      asm volatile("" ::: "memory");
      fetch(slot);
      slot = slot == DEPTH - 1 ? 0 : slot + 1;
    }
    f32x4* sums = red + par * NW * USED;
    if (lane < USED) sums[wave * USED + lane] = acc;
    // own sums written, the next weights still under way; the other half of
    // red is free once all are here
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wave == 0 && lane < USED && !(GLU && lo >= 8)) {
      f32x4 v = sums[lane];
#pragma unroll
      for (int w = 1; w < NW; w++) v += sums[w * USED + lane];
      if constexpr (GLU) {
        f32x4 u = sums[lane + 8];
#pragma unroll
        for (int w = 1; w < NW; w++) u += sums[w * USED + lane + 8];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = skinny::silu(v[r]) * u[r];
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = 4 * hi + r;
        if (m < M) out[(int64_t)m * N + t * COLS + lo] = f32_to_bf16(v[r]);
      }
    }
    par ^= 1;
  }
  skinny::wait_loads<0>();          // no copy to LDS outlives the workgroup's
}

// 0, or the stages of a ring with which the sizes fit
int w4_tiles_depth(int64_t M, int64_t rows, int64_t K, int64_t group) {
  if (M < 1 || M > 16 || group != 128 || K % W4_K || rows % 16 ||
      rows * (K / 2) >= 1LL << 32)
    return 0;
  const int mr = M <= 4 ? 4 : 16;
  return w4_fits(8, 3, mr, M, K) ? 3 : w4_fits(8, 2, mr, M, K) ? 2 : 0;
}

// Whether they are faster than the row streams (from 5 rows of x on: MFMA from
// global memory), us, streams and tiles. K = 512 S keeps S of the eight waves
// busy.
//   Alone: one row never; two with many weights, 4096 x 14336 13.8 and 9.7,
// 8192 x 4096 8.1 and 7.7, 4096 x 8192 8.5 and 8.2, but 6144 x 4096 7.1 and 7.4,
// 12288 x 2048 6.4 and 6.6, 16384 x 2048 6.9 and 7.6. Three or four of a narrow K with 4096 rows of W (2048 x 2048 4.4 and 4.7,
// 11008 .84). More, from K of 2048 on (4096 x 1024 3.8 and 4.6 at 5, 57344 x 512 9.7
// and 20.2), beyond 8 rows at 2048 with 6144 of W (4096: 6.1 and 6.7 at 16).
//   A pair saves a launch. One row: but for some 400 tiles, which are neither two
// rounds of one workgroup per CU nor enough for two (6144 x 2048 5.5 and 5.7, x 4096
// 7.0 and 7.2, x 8192 10.5 and 10.4; 4096 x 4096 6.5 and 5.4, 5120 x 2048 5.4 and 5.5,
// 7168 x 2048 6.0 and 5.9, x 4096 8.2 and 7.5, 28672 x 4096 17.6 and 15.1, 57344 x 8192
// 60.9 and 46.9, others 1.03 to 1.35). Two: always (6144 x 2048 6.8 and 5.9, 28672 x
// 4096 18.1 and 15.7, 57344 x 1024 18.9 and 13.2). From five on K up to 1024 only with
// few (22016 x 512 7.4 and 11.0, 22016 x 1024 1.04).
bool w4_tiles_pay(int64_t M, int64_t rows, int64_t K, bool glu) {
  if (glu) {
    if (M <= 2) return M == 2 || rows < 6144 || rows >= 7168;
    return M <= 4 || K > 1024 || rows <= 4096;
  }
  if (M == 1) return false;
  if (M == 2) return K > 2048 && rows * K >= 32 << 20;
  if (M <= 4) return K > 2048 || rows >= 4096;
  return K > 2048 || (K == 2048 && (M <= 8 || rows >= 6144));
}

template <bool GLU, bool NORM = false>
bool launch_w4_tiles(at::Tensor& out, const at::Tensor& x,
                     const at::Tensor& qweight, const at::Tensor& scales,
                     const at::Tensor& zeros, int64_t group,
                     const W4Norm& norm = {}) {
  const int M = x.size(0), K = x.size(1);
  const int N = qweight.size(0) / (GLU ? 2 : 1);
  const int depth = w4_tiles_depth(M, qweight.size(0), K, group);
  if (!depth || (uintptr_t)x.data_ptr() % 16 ||
      (uintptr_t)qweight.data_ptr() % 16)
    return false;
  const int ntiles = N / (GLU ? 8 : 16);
  // two workgroups of four waves per CU, where x fits twice
  const bool two = M <= 4 && ntiles >= 512 && w4_fits(4, 3, 4, M, K);
  // little of x, asked for behind the weights; few tiles: 3 rows, x ahead and behind,
  // 1024 x 3072 5.1 and 4.8, 4096 x 3584 5.84 and 5.72, but 4096 x 4096 5.9 and 6.1, 5 of
  // 1024 x 3584 5.2 and 5.5, 6 of 4608 x 3072 6.7 and 7.1
  const bool brief = K <= 2048
      ? M * K <= 16384 : ntiles <= 256 && M * K <= (K < 4096 ? 16384 : 8192);
#define W4T_LAUNCH(NW_, MR_, D_, ...)                                         \
  hipLaunchKernelGGL(                                                         \
      (w4a16_tiles_kernel<NW_, MR_, D_, GLU, NORM, ##__VA_ARGS__>),           \
      dim3(std::min(2048 / NW_, ntiles)), dim3(64 * NW_), 0,                  \
      at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),                 \
      (const short*)x.data_ptr(), (const uint32_t*)qweight.data_ptr(),        \
      scales.data_ptr<float>(), zeros.data_ptr<float>(), M, N, K, norm)
  if (two) {
    W4T_LAUNCH(4, 4, 3);
  } else if (M <= 4) {
    if (!NORM && brief) W4T_LAUNCH(8, 4, 3, 0);
    else if (depth == 3) W4T_LAUNCH(8, 4, 3);
    else W4T_LAUNCH(8, 4, 2);
  } else if constexpr (!NORM) {
    if (brief) W4T_LAUNCH(8, 16, 3, 0);
    else if (depth == 3) W4T_LAUNCH(8, 16, 3);
    else W4T_LAUNCH(8, 16, 2);
  }
#undef W4T_LAUNCH
  return true;
}

}  // namespace

// ---------------------------------------------------------------- dequant
// out[N, K] bf16 <- dequantized weights. Elementwise, one u32 pack per
// thread; writes are short8 (16B) so the store path is fully vectorized.
__global__ __launch_bounds__(256)
void w4a16_dequant_kernel(short* __restrict__ out,
                          const uint32_t* __restrict__ qw,
                          const float* __restrict__ scales,
                          const float* __restrict__ zeros,
                          int N, int K, int group) {
  const int kw = K >> 3;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)N * kw) return;
  const int n = idx / kw;
  const int w = idx % kw;
  const int k0 = w << 3;
  const int g = k0 / group;
  const int gstride = K / group;
  const float s = scales[(int64_t)n * gstride + g];
  const float z = zeros[(int64_t)n * gstride + g];
  const uint32_t q = qw[idx];
  short8_t o;
#pragma unroll
  for (int j = 0; j < 8; ++j)
    o[j] = f32_to_bf16(s * (float)((q >> (4 * j)) & 0xF) - z);
  *reinterpret_cast<short8_t*>(out + (int64_t)n * K + k0) = o;
}

// ------------------------------------------------------- fused MFMA GEMM
// Marlin-class mid/large-M path: C[M,N] = x[M,K]bf16 @ dequant(W)^T with
// the dequant INLINE in the K-loop — the 4-bit weights go HBM → register
// → (dequant) → swizzled LDS → MFMA, never touching a full-precision
// scratch buffer (the round-1 path dequantized the whole weight to
// global memory first: 5x the weight traffic, and it lost to bf16 at
// saturation — docs/ROADMAP.md #2).
//
// Structure: 2-barrier 64x64x64 tile, 4 waves as 2x2, MFMA 16x16x32
// (same skeleton as moe.hip). A staged with global_load_lds
// (pre-swizzled source); B: each thread loads u32 packed words (one
// word == one 16-B bf16 chunk after dequant), dequants with its group's
// (s, z), and ds_writes the chunk at the XOR-swizzled slot.
__global__ __launch_bounds__(256, 2)
void w4a16_gemm_kernel(short* __restrict__ out,          // [M, N] bf16
                       const short* __restrict__ x,      // [M, K] bf16
                       const uint32_t* __restrict__ qw,  // [N, K/8]
                       const float* __restrict__ scales, // [N, K/G]
                       const float* __restrict__ zeros,
                       int M, int N, int K, int group) {
  constexpr int BM = 64, BN = 64, BK = 64;
  const int m0 = blockIdx.x * BM;
  const int n0 = blockIdx.y * BN;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int lo = lane & 15, hi = lane >> 4;
  const int kw = K >> 3;
  const int gstride = K / group;

  __shared__ short lds_a[BM * BK];
  __shared__ short lds_b[BN * BK];

  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = 0; k0 < K; k0 += BK) {
    // ---- A tile via global_load_lds (rows clamped at the M tail) ----
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int seg = i * 4 + wave;
      const int idx = seg * 64 + lane;
      const int row = idx >> 3;
      const int c = (idx & 7) ^ (row & 7);
      const int srow = min(m0 + row, M - 1);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) unsigned int*)
              (x + (int64_t)srow * K + k0 + c * 8),
          (__attribute__((address_space(3))) unsigned int*)
              (lds_a + seg * 512),
          16, 0, 0);
    }
    // ---- B tile: packed u32 → inline dequant → swizzled ds_write ----
#pragma unroll
    for (int rep = 0; rep < 2; rep++) {
      const int id = rep * 256 + threadIdx.x;     // 512 words per tile
      const int row = id >> 3;                    // n row in tile
      const int wslot = id & 7;                   // 8 words (64 k) / row
      const int n = n0 + row;
      const uint32_t q = qw[(int64_t)n * kw + (k0 >> 3) + wslot];
      const int g = (k0 + wslot * 8) / group;
      const float s = scales[(int64_t)n * gstride + g];
      const float z = zeros[(int64_t)n * gstride + g];
      short8_t dq;
#pragma unroll
      for (int j = 0; j < 8; j++)
        dq[j] = f32_to_bf16(s * (float)((q >> (4 * j)) & 0xF) - z);
      const int c = wslot ^ (row & 7);
      *reinterpret_cast<short8_t*>(lds_b + row * BK + c * 8) = dq;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK / 32; kk++) {
      bf16x8 af[2], bf[2];
#pragma unroll
      for (int r = 0; r < 2; r++) {
        {
          const int row = wm * 32 + r * 16 + lo;
          const int c = (kk * 4 + hi) ^ (row & 7);
          af[r] = *reinterpret_cast<const bf16x8*>(lds_a + row * BK + c * 8);
        }
        {
          const int row = wn * 32 + r * 16 + lo;
          const int c = (kk * 4 + hi) ^ (row & 7);
          bf[r] = *reinterpret_cast<const bf16x8*>(lds_b + row * BK + c * 8);
        }
      }
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              af[a], bf[b], acc[a][b], 0, 0, 0);
    }
    __syncthreads();
  }

#pragma unroll
  for (int a = 0; a < 2; a++) {
    const int row_base = wm * 32 + a * 16 + hi * 4;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = m0 + row_base + r;
      if (row >= M) continue;
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int col = n0 + wn * 32 + b * 16 + lo;
        out[(int64_t)row * N + col] = f32_to_bf16(acc[a][b][r]);
      }
    }
  }
}

void w4a16_gemm(at::Tensor out, at::Tensor x, at::Tensor qweight,
                at::Tensor scales, at::Tensor zeros, int64_t group) {
  const int M = x.size(0), K = x.size(1), N = qweight.size(0);
  TORCH_CHECK(x.is_contiguous() && out.is_contiguous());
  TORCH_CHECK(K % 64 == 0 && N % 64 == 0 && group % 64 == 0 &&
              K % group == 0, "w4a16_gemm: 64|K, 64|N, 64|group required");
  dim3 grid((M + 63) / 64, N / 64), block(256);
  auto stream = at::hip::getCurrentHIPStream();
  w4a16_gemm_kernel<<<grid, block, 0, stream>>>(
      (short*)out.data_ptr(), (const short*)x.data_ptr(),
      (const uint32_t*)qweight.data_ptr(), scales.data_ptr<float>(),
      zeros.data_ptr<float>(), M, N, K, (int)group);
}

void w4a16_gemv(at::Tensor out, at::Tensor x, at::Tensor qweight,
                at::Tensor scales, at::Tensor zeros, int64_t group) {
  const int M = x.size(0), K = x.size(1), N = qweight.size(0);
  TORCH_CHECK(M <= 32, "w4a16_gemv: M must be <= 32 (use dequant+GEMM)");
  TORCH_CHECK(K % 64 == 0 && group % 64 == 0 && K % group == 0,
              "w4a16_gemv: 64|K and 64|group required");
  TORCH_CHECK(x.is_contiguous() && out.is_contiguous());
  if (M == 0 || N == 0) return;
  if (w4_tiles_pay(M, N, K, false) &&
      launch_w4_tiles<false>(out, x, qweight, scales, zeros, group))
    return;
  auto stream = at::hip::getCurrentHIPStream();
#define W4_ARGS                                                               \
  (short*)out.data_ptr(), (const short*)x.data_ptr(),                         \
      (const uint32_t*)qweight.data_ptr(), scales.data_ptr<float>(),          \
      zeros.data_ptr<float>()
#define W4_STREAM(M_, R_)                                                     \
  hipLaunchKernelGGL((w4a16_stream_kernel<M_, R_>),                           \
                     dim3((N + 4 * R_ - 1) / (4 * R_)), dim3(256), 0, stream, \
                     W4_ARGS, N, K, (int)group)
  // four rows per wave share what they do with x once there are waves to
  // spare (M = 4, N = 28672: 32.3 us against 36.4 with two; N = 6144: 13.0
  // against 10.3)
  const bool many = N >= 16384;
  switch (M) {
    case 1: W4_STREAM(1, 2); return;
    case 2: if (many) W4_STREAM(2, 4); else W4_STREAM(2, 2); return;
    case 3: if (many) W4_STREAM(3, 4); else W4_STREAM(3, 2); return;
    case 4: if (many) W4_STREAM(4, 4); else W4_STREAM(4, 2); return;
    default: break;
  }
#undef W4_STREAM
#define W4_MFMA(MT_, NT_, WORDS_)                                             \
  hipLaunchKernelGGL((w4a16_mfma_kernel<MT_, NT_, WORDS_>),                   \
                     dim3((N + 16 * NT_ - 1) / (16 * NT_)), dim3(256), 0,     \
                     stream, W4_ARGS, M, N, K, (int)group)
  // two tiles per workgroup halve the x reads; only where rows are many
  // enough to fill the chip all the same
  const bool wide = N >= 16 * 2 * 256;
  if (group % 128 == 0) {
    if (M <= 16) { if (wide) W4_MFMA(1, 2, 4); else W4_MFMA(1, 1, 4); }
    else { if (wide) W4_MFMA(2, 2, 4); else W4_MFMA(2, 1, 4); }
  } else {
    if (M <= 16) W4_MFMA(1, 1, 2); else W4_MFMA(2, 1, 2);
  }
#undef W4_MFMA
#undef W4_ARGS
}

// Whether M rows of x run in the tiles: alone or as a SwiGLU pair
bool w4a16_in_tiles(int64_t M, int64_t rows, int64_t K, int64_t group,
                    bool glu) {
  return w4_tiles_depth(M, rows, K, group) > 0 &&
         w4_tiles_pay(M, rows, K, glu);
}

// Whether the norm of up to two rows goes into their product in the tiles: but for
// one row of few whole streams and of some 350 tiles (us, norm and what else would
// follow it, and one launch: one row of 6144 x 4096 8.2 and 8.7, 5120 x 2048 5.7 and
// 6.3, 20480 x 2048 9.0 and 9.4, 28672 x 2048 1.06, 10240 x 4096 9.7 and 9.9, 12288 x
// 4096 1.10, 10240 x 8192 1.06; 6144 x 512 5.0 and 5.4, x 1024 5.2 and 5.6, 5120 x 5120
// 9.3 and 9.5, but 7168 x 5120 11.3 and 10.3, 4096 x 1024 1.06; 2048 x 1024 4.8 and 4.6,
// 28672 x 512 9.6 and 7.6; pairs 28672 x 4096 19.5 and 15.8, 57344 x 8192 48.0 and 44.6,
// 4096 x 512 6.3 and 4.6; two rows of 6144 x 4096 10.0 and 8.8, 10240 x 8192 18.0 and
// 15.5, 1536 x 512 5.3 and 4.6; pairs 28672 x 4096 18.1 and 16.0, 57344 x 1024 20.9 and
// 14.1).
bool w4a16_norm_in_tiles(int64_t M, int64_t rows, int64_t K, int64_t group,
                         bool glu) {
  const bool one = K % 2048 ? rows <= 4096 || rows >= 7168
                            : rows >= 10240 && rows * K >= 48 << 20;
  return M <= 2 && K <= 2048 * W4_NORM && (glu || M == 2 || one) &&
         w4_tiles_depth(M, rows, K, group) > 0;
}

// silu(x Wg^T) * (x Wu^T) of the stacked W = [Wg | Wu]

void w4a16_swiglu(at::Tensor out, at::Tensor x, at::Tensor qweight,
                  at::Tensor scales, at::Tensor zeros, int64_t group) {
  TORCH_CHECK(x.is_contiguous() && out.is_contiguous() &&
              x.dtype() == at::kBFloat16 && out.dtype() == at::kBFloat16 &&
              qweight.is_contiguous() && scales.is_contiguous() &&
              zeros.is_contiguous());
  TORCH_CHECK(qweight.size(0) % 2 == 0 && qweight.size(1) * 8 == x.size(1) &&
              out.size(0) == x.size(0) &&
              out.size(1) * 2 == qweight.size(0));
  TORCH_CHECK(launch_w4_tiles<true>(out, x, qweight, scales, zeros, group),
              "w4a16_swiglu: sizes of the tiles");
}

// x W^T of rms(x + residual) * g (glu: the same of the pair); sum: x + residual,
// not one of the others
void w4a16_norm_linear(at::Tensor out, at::Tensor sum, at::Tensor x,
                       at::Tensor residual, at::Tensor g, double eps,
                       at::Tensor qweight, at::Tensor scales, at::Tensor zeros,
                       int64_t group, bool glu) {
  const int64_t M = x.size(0), K = x.size(1), pair = glu ? 2 : 1;
  for (const auto& t : {x, residual, sum})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.sizes() == x.sizes() &&
                t.dtype() == at::kBFloat16 && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(g.is_cuda() && g.is_contiguous() && g.numel() == K &&
              g.dtype() == at::kBFloat16 && (uintptr_t)g.data_ptr() % 16 == 0);
  TORCH_CHECK(out.is_contiguous() && out.dtype() == at::kBFloat16 &&
              qweight.is_contiguous() && scales.is_contiguous() &&
              zeros.is_contiguous() && qweight.size(0) % pair == 0 &&
              qweight.size(1) * 8 == K && out.size(0) == M &&
              out.size(1) * pair == qweight.size(0));
  TORCH_CHECK(M >= 1 && M <= 2 && K <= 2048 * W4_NORM &&
              sum.data_ptr() != residual.data_ptr() &&
              sum.data_ptr() != x.data_ptr());
  const W4Norm norm = {(short*)sum.data_ptr(),
                       (const short*)residual.data_ptr(),
                       (const short*)g.data_ptr(), (float)eps};
  const bool fits = glu ? launch_w4_tiles<true, true>(out, x, qweight, scales,
                                                      zeros, group, norm)
                        : launch_w4_tiles<false, true>(out, x, qweight, scales,
                                                       zeros, group, norm);
  TORCH_CHECK(fits, "w4a16_norm_linear: sizes of the tiles");
}

void w4a16_dequant(at::Tensor out, at::Tensor qweight, at::Tensor scales,
                   at::Tensor zeros, int64_t group) {
  const int N = qweight.size(0), K = out.size(1);
  TORCH_CHECK(K % 8 == 0 && K % group == 0);
  const int64_t total = (int64_t)N * (K >> 3);
  dim3 grid((total + 255) / 256), block(256);
  auto stream = at::hip::getCurrentHIPStream();
  w4a16_dequant_kernel<<<grid, block, 0, stream>>>(
      (short*)out.data_ptr(), (const uint32_t*)qweight.data_ptr(),
      scales.data_ptr<float>(), zeros.data_ptr<float>(), N, K, (int)group);
}

}  // namespace kaito
