// Grouped GEMMs of prompt-sized MoE steps: rows sorted by expert, one launch
// per projection, tile bounds from the device's offsets (no host read).
//
//   moe_grouped_up    act[s] = act(x[tok_s] Wg[e]^T, x[tok_s] Wu[e]^T)
//   moe_grouped_down  y[s] = act[s] Wd[e]^T (+ bias), bf16 or f32
//   moe_combine       out[t] = sum over t's pairs of weight * y[row], f32
//                     sums in the order of the choice, plus identity and
//                     shared experts
//
// A workgroup of 8 waves (2 over rows x 4 over weight rows) computes BM rows
// x 256 weight rows (up: 128 gate rows beside their 128 up rows, 32 + 32 per
// wave, so a lane holds both of a pair) in K steps of 64 on
// v_mfma_f32_32x32x16_bf16, transposed (C^T = W X^T: a lane owns one token row
// and 4 neighbouring outputs at a time). Both operands arrive by 16-byte
// loads straight to LDS (16-byte chunk c of row r at c ^ (r & 7)); as buffer
// loads, behind which the compiler can count LDS reads (behind the global form
// it waits for all). At BM = 256 a step is 32 MFMA per wave, 2048 cycles of a
// SIMD's two waves, against 192 KB of LDS reads (1536 cycles) and 64 KB of
// staging per CU: all have to overlap, so fragments are read one step of 16 dims
// ahead and the loads go out a few at a time. The bound is the way from the
// caches to LDS: without the products the loads alone take nine tenths of the
// time, without the loads the rest takes four fifths. At 8 of 28672 x 4096 the matrix
// cores are busy 72 % of it and waves wait a quarter of theirs, for loads at the
// barrier; a library product of that width, 83 % busy, has the same hit rate in L2
// (79 %), bytes per operation and clock (1.57 GHz), but two thirds of the LDS reads
// per operation: 128 x 64 outputs per wave read 6 fragments for 8 products, 128 x
// 128 read 8 for 16. (K steps of 32 in four or five buffers, whose rows are half
// lines: a tenth slower; waves of a SIMD taking turns behind barriers, other starts
// in K per tile: no change.)
//
// Tiles are numbered expert by expert, in blocks of 4 column tiles x all row
// tiles, and every XCD takes one contiguous eighth of them: the 32 tiles in
// flight behind one L2 share rows and weights. A last round of up to 8 tiles for
// an XCD's 32 CUs is cut in quarters, 128 x 128, one per CU; so is a small step's
// only round of up to 16. Measured on one MI355X, 8 experts of 2048 x 2048, top
// 2, rows as drawn from 16 kinds of tokens, us, two buffers and whole tiles, now:
// 8192 tokens 317 and 278, with the epilogue of today 254 (1080 TFLOP/s), down 165
// and 139; 4096 174 and 149, 106 and 86; 2048 114 and 90; 1000 down 60 and 49. 8 of
// 4096 x 14336, 8192 tokens:
// 3419 and 3262 (1180 TFLOP/s), 1875 and 1676. 8-byte stores cost a tenth more. A
// library GEMM per expert with its gathers, casts and index_add took 958 us behind
// a host read at the first of these.
#include "flash_prefill.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <type_traits>

namespace kaito {

namespace {

using flash::f32x16;
using flash::hbf16x8;
using flash::mfma32;

constexpr int BK = 64;              // K step
constexpr int BN = 256;             // weight rows per tile
constexpr int NG = 4;               // column tiles that share row tiles
constexpr int XCD_CUS = 32;
// A quarter takes about two fifths of a tile's time, and the last round runs on
// caches of its own: 17 to 24 tiles in three rounds of quarters lost (2880 x 2880,
// 4096 tokens, down: 341 and 352 us), 9 to 16 in two broke even or lost 1 %, except
// where they are the whole step (58 and 50).
constexpr int QUARTER_REST = XCD_CUS / 4;

struct GemmArgs {
  short* out;                       // [TK, N]
  float* out32;                     // the same in f32 (DOWN), or nullptr
  const short* x;                   // up: [T, K]; down: [TK, K]
  const short* w;                   // [E, rows, K]
  const short* bias;                // [E, rows] or nullptr
  const int* rows;                  // x row of a sorted row; none: the same
  const int* offsets;               // [.., E + 1]
  int e_base, E, N, K;
  float limit;
};

enum Kind { UP_GATED, UP_CLAMPED, UP_PLAIN, DOWN };
constexpr bool is_gated(int kind) { return kind <= UP_CLAMPED; }

// 16 bytes per lane from r + lane offset + uniform offset to dst + 16 * lane
KAITO_DEV void buffer_copy16(__amdgpu_buffer_rsrc_t r, short* dst,
                             const uint32_t lane_off, const int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)dst, 16, lane_off, off, 0, 0);
}

// CLAMPED: min(g, limit) sigmoid(1.702 min(g, limit)) (clamp(u) + 1)
template <int KIND>
KAITO_DEV float gated(float g, float u, float limit) {
  if constexpr (KIND == UP_CLAMPED) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return (u + 1.f) * swish_f32(g, 1.702f);
  }
  return silu_f32(g) * u;
}

// elements of LDS: two and a half K steps of a whole tile, five of a quarter
constexpr int LDS = 5 * 256 * BK;

// BM rows x BW weight rows of one expert by 8 waves, WM of them over the rows;
// NST K steps in LDS, or 0: five slots of BM = BW rows. m0: first row, n0: first
// output.
template <int BM, int BW, int WM, int NST, int KIND>
KAITO_DEV void grouped_tile(const GemmArgs& a, short* lds, const int expert,
                            const int m0, const int row_end, const int n0) {
  constexpr int WN = 8 / WM, MT = BM / WM / 32;   // 32-row tiles of a wave
  constexpr int LX = BM * BK / 8 / 512, LW = BW * BK / 8 / 512;
  constexpr int STEP = (BM + BW) * BK;
  static_assert(WN * 64 == BW && NST * STEP <= LDS, "tile");
  const int lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;

  // ---- staging slots: slot s (16 bytes) is row s / 8, place s % 8; byte
  // offsets from the tile's first row (gathered rows: from x, which the caller
  // keeps below 4 GB)
  const int wrows = is_gated(KIND) ? 2 * a.N : a.N;
  const short* we = a.w + ((int64_t)expert * wrows + n0) * a.K;
  const short* xe = a.rows ? a.x : a.x + (int64_t)m0 * a.K;
  const auto xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<short*>(xe), 0, 0xffffffff, 0x27000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<short*>(we), 0, 0xffffffff, 0x27000);
  constexpr int CH = BK / 8;        // 16-byte chunks of a row
  auto place = [](const int row, const int c) { return c ^ (row >> 1 & 7); };
  uint32_t xs[LX], ws[LW];
  int src[LX];                      // one wait for all of them
#pragma unroll
  for (int j = 0; j < LX; j++)
    src[j] = min((int)(j * 512 + threadIdx.x) / CH, row_end - 1 - m0);
  if (a.rows) {
#pragma unroll
    for (int j = 0; j < LX; j++) src[j] = a.rows[m0 + src[j]];
  }
#pragma unroll
  for (int j = 0; j < LX; j++) {
    const int s = j * 512 + threadIdx.x;
    xs[j] = ((uint32_t)src[j] * a.K + place(s / CH, s % CH) * 8) * 2;
  }
#pragma unroll
  for (int j = 0; j < LW; j++) {
    const int s = j * 512 + threadIdx.x, row = s / CH;
    const int c = place(row, s % CH);
    // gated: every 64 tile rows are 32 gate rows, then their up rows
    const uint32_t n = is_gated(KIND)
        ? min((row / 64) * 32 + row % 32, a.N - 1 - n0) +
              (row % 64 >= 32 ? a.N : 0)
        : min(row, a.N - 1 - n0);
    ws[j] = (n * a.K + c * 8) * 2;
  }
  auto stage_x = [&](const int k, short* buf, const int j0, const int j1) {
#pragma unroll
    for (int j = 0; j < LX; j++)
      if (j >= j0 && j < j1)
        buffer_copy16(xr, buf + (j * 512 + wave * 64) * 8, xs[j], k * 2);
  };
  auto stage_w = [&](const int k, short* buf) {
#pragma unroll
    for (int j = 0; j < LW; j++)
      buffer_copy16(wr, buf + (j * 512 + wave * 64) * 8, ws[j], k * 2);
  };

  f32x16 acc[2][MT];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  // Fragments of 16 dims of K are read one step ahead of their products, the
  // first of the next tile beside the last products of this one: the barrier
  // that frees this tile stands between its last read and its last products.
  hbf16x8 wf[2][2], xf[2][MT];
  auto read = [&](const short* xbuf, const short* wbuf, const int kk) {
    const int c = place(lr, kk * 2 + h) * 8, f = kk & 1;
    const short* xb = xbuf + (wm * (BM / WM) + lr) * BK + c;
    const short* wb = wbuf + (wn * 64 + lr) * BK + c;
#pragma unroll
    for (int i = 0; i < 2; i++)
      wf[f][i] = *reinterpret_cast<const hbf16x8*>(wb + i * 32 * BK);
#pragma unroll
    for (int j = 0; j < MT; j++)
      xf[f][j] = *reinterpret_cast<const hbf16x8*>(xb + j * 32 * BK);
  };
  auto multiply = [&](const int kk) {
    const int f = kk & 1;
    __builtin_amdgcn_sched_barrier(0);      // the next reads are under way
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        acc[i][j] = mfma32(wf[f][i], xf[f][j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // own reads done and own loads landed but for the newest LATER: all's
  auto meet = [&](auto newest, const bool later) {
    constexpr int N = decltype(newest)::value;
    if (N > 0 && later)
      __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    else
      __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if constexpr (NST == 0) {
    // x and w by turns through five slots: x(s), w(s) and x(s + 1) are there
    // when step s begins, w(s + 1) and x(s + 2) are asked for in its course.
    // All of a step's loads at once, for the next but one, kept the caches busy
    // in bursts: 514 cycles from request to data where 360 are now.
    constexpr int SLOT = BM * BK;
    static_assert(BM == BW && 5 * SLOT <= LDS && BK == 64, "slots");
    constexpr std::integral_constant<int, LX> newest;
    stage_w(0, lds + SLOT);
    stage_x(0, lds, 0, LX);
    if (BK < a.K) stage_x(BK, lds + 2 * SLOT, 0, LX);
    meet(newest, BK < a.K);
    int slot = 0;                   // of x(s); w(s), x(s + 1) .. follow
    auto nth = [&](const int i) {
      return lds + (slot + i < 5 ? slot + i : slot + i - 5) * SLOT;
    };
    read(nth(0), nth(1), 0);
    for (int k = 0; k < a.K; k += BK) {
      const bool more = k + BK < a.K, more2 = k + 2 * BK < a.K;
      read(nth(0), nth(1), 1);
      if (more) stage_w(k + BK, nth(3));
      multiply(0);
      read(nth(0), nth(1), 2);
      if (more2) stage_x(k + 2 * BK, nth(4), 0, LX / 2);
      multiply(1);
      read(nth(0), nth(1), 3);
      if (more2) stage_x(k + 2 * BK, nth(4), LX / 2, LX);
      multiply(2);
      meet(newest, more2);
      slot = slot < 3 ? slot + 2 : slot - 3;
      if (more) read(nth(0), nth(1), 0);
      multiply(3);
    }
  } else {
    constexpr int STEPS = BK / 16;
    constexpr std::integral_constant<int, (NST - 2) * (LX + LW)> newest;
    auto stage = [&](const int k, const int at) {
      stage_x(k, lds + at * STEP, 0, LX);
      stage_w(k, lds + at * STEP + BM * BK);
    };
    auto next = [&](const int at, const int kk) {
      read(lds + at * STEP, lds + at * STEP + BM * BK, kk);
    };
    stage(0, 0);
#pragma unroll
    for (int i = 1; i < NST - 1; i++)
      if (i * BK < a.K) stage(i * BK, i);
    meet(newest, (NST - 2) * BK < a.K);
    if ((NST - 1) * BK < a.K) stage((NST - 1) * BK, NST - 1);
    next(0, 0);
    int cur = 0;
    for (int k = 0; k < a.K; k += BK) {
#pragma unroll
      for (int kk = 0; kk < STEPS - 1; kk++) {
        next(cur, kk + 1);
        multiply(kk);
      }
      meet(newest, k + (NST - 1) * BK < a.K);
      if (k + NST * BK < a.K) stage(k + NST * BK, cur);
      cur = cur == NST - 1 ? 0 : cur + 1;
      if (k + BK < a.K) next(cur, 0);
      multiply(STEPS - 1);
    }
  }

  // ---- outputs n = 8 b + 4 h + e of 32-row tile i, token row lr of tile j
  constexpr int NI = is_gated(KIND) ? 1 : 2;
  constexpr int WC = NI * 32;       // columns of a wave: all exist or none
  const int c0 = n0 + wn * WC;
  if (c0 >= a.N) return;            // N is a multiple of 64; no barrier below
  // added where a value leaves: ahead of that, over all of acc, it cost 132 bytes
  // of scratch per lane and 55 us of 312 (up, 8 experts of 2048 x 2048, 16384
  // pairs of uneven experts, weights out of the caches; with the activations'
  // divisions in half the instructions). Read once: for every 32 rows anew, a down
  // projection of 8192 tokens by 16 experts of 1024 x 512 took 51.9 us, now 47.9
  const short* be = a.bias + (int64_t)expert * wrows + c0 + 4 * h;
  short4_t bias[2][4] = {};
  if (a.bias) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int b = 0; b < 4; b++)
        bias[i][b] = *reinterpret_cast<const short4_t*>(
            be + (is_gated(KIND) ? i * a.N : i * 32) + 8 * b);
  }
  // bf16 rows pass through the wave's part of LDS (every wave is done with
  // its tiles) and leave as 16 bytes a lane
  constexpr int PITCH = WC + 8, LANES = WC / 8;
  short* slab = lds + wave * 32 * PITCH;
#pragma unroll
  for (int j = 0; j < MT; j++) {
    const int mj = m0 + wm * (BM / WM) + j * 32;
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int b = 0; b < 4; b++) {
        float4_t v, u;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          v[e] = acc[i][j][b * 4 + e];
          if constexpr (is_gated(KIND)) u[e] = acc[1][j][b * 4 + e];
        }
        if (a.bias) {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            v[e] += bf16_to_f32(bias[i][b][e]);
            if constexpr (is_gated(KIND)) u[e] += bf16_to_f32(bias[1][b][e]);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if constexpr (is_gated(KIND)) {
            v[e] = gated<KIND>(v[e], u[e], a.limit);
          } else if constexpr (KIND == UP_PLAIN) {
            v[e] = fmaxf(v[e], 0.f);
            v[e] *= v[e];
          }
        }
        const int n = i * 32 + 8 * b + 4 * h;
        if (KIND == DOWN && a.out32) {
          if (mj + lr < row_end)
            *reinterpret_cast<float4_t*>(
                a.out32 + (int64_t)(mj + lr) * a.N + c0 + n) = v;
        } else {
          *reinterpret_cast<short4_t*>(slab + lr * PITCH + n) =
              short4_t{f32_to_bf16(v[0]), f32_to_bf16(v[1]),
                       f32_to_bf16(v[2]), f32_to_bf16(v[3])};
        }
      }
    if (KIND == DOWN && a.out32) continue;
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < 32; r += 64 / LANES) {
      const int row = r + lane / LANES, n = lane % LANES * 8;
      const short8_t v =
          *reinterpret_cast<const short8_t*>(slab + row * PITCH + n);
      if (mj + row < row_end)
        *reinterpret_cast<short8_t*>(a.out + (int64_t)(mj + row) * a.N + c0 +
                                     n) = v;
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
  }
}

template <int BM, int KIND>
__global__ __launch_bounds__(512, 2) void moe_grouped_kernel(const GemmArgs a) {
  constexpr int COLS = is_gated(KIND) ? BN / 2 : BN;   // outputs per tile
  constexpr bool QUARTERS = BM == 256;
  __shared__ __attribute__((aligned(128)))
  short lds[BM == 256 ? LDS : 2 * (BM + BN) * BK];
  const int lane = threadIdx.x & 63;
  const int ntiles = (a.N + COLS - 1) / COLS;

  // ---- this workgroup's tile: every wave scans the experts, 64 at a time
  int total = 0;
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    const int e = a.e_base + e0 + lane;
    int n = e0 + lane < a.E
        ? (a.offsets[e + 1] - a.offsets[e] + BM - 1) / BM : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    total += n;
  }
  total = __builtin_amdgcn_readfirstlane(total) * ntiles;
  const int share = (total + 7) / 8, at = (blockIdx.x % 8) * share;
  const int here = min(share, total - at);  // tiles of this XCD
  int rest = here % XCD_CUS;        // of its last round
  if (!QUARTERS || rest > (here < XCD_CUS ? 2 : 1) * QUARTER_REST) rest = 0;
  int in_share = blockIdx.x / 8, quarter = -1;
  if (in_share >= here - rest) {
    const int p = in_share - (here - rest);
    if (p >= 4 * rest) return;
    in_share = here - rest + p / 4;
    quarter = p % 4;
  }
  int t = at + in_share;
  int expert = -1, mtiles = 0, row0 = 0, row_end = 0;
  for (int e0 = 0; e0 < a.E && expert < 0; e0 += 64) {
    const int e = a.e_base + e0 + lane;
    const int o0 = e0 + lane < a.E ? a.offsets[e] : 0;
    const int o1 = e0 + lane < a.E ? a.offsets[e + 1] : 0;
    const int n = (o1 - o0 + BM - 1) / BM;
    int scan = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int add = __shfl_up(scan, off, 64);
      if (lane >= off) scan += add;
    }
    const unsigned long long hit = __ballot(scan * ntiles > t);
    if (hit) {
      const int src = __builtin_ctzll(hit);
      expert = a.e_base + e0 + src;
      mtiles = __builtin_amdgcn_readlane(n, src);
      t -= (__builtin_amdgcn_readlane(scan, src) - mtiles) * ntiles;
      row0 = __builtin_amdgcn_readlane(o0, src);
      row_end = __builtin_amdgcn_readlane(o1, src);
    } else {
      t -= __builtin_amdgcn_readlane(scan, 63) * ntiles;
    }
  }
  // blocks of NG column tiles, column fastest
  const int blk = t / (NG * mtiles);
  const int wide = min(NG, ntiles - blk * NG);
  const int in_blk = t - blk * NG * mtiles;
  const int nt = blk * NG + in_blk % wide, mt0 = in_blk / wide;

  const int m0 = row0 + mt0 * BM, n0 = nt * COLS;
  if constexpr (QUARTERS) {
    if (quarter >= 0) {
      const int m = m0 + quarter / 2 * (BM / 2);
      const int n = n0 + quarter % 2 * (COLS / 2);
      if (m < row_end && n < a.N)
        grouped_tile<BM / 2, BN / 2, 4, 5, KIND>(a, lds, expert, m, row_end,
                                                 n);
      return;
    }
  }
  grouped_tile<BM, BN, 2, BM == 256 ? 0 : 2, KIND>(a, lds, expert, m0, row_end,
                                                   n0);
}

// ---- keys and values of latent rows ----------------------------------------
// [k | v][t] = c[t] [Wk | Wv^T]^T, tiles of 256 x 256 over both: the tiles of
// Wk's N1 rows first. Behind one another, as a library product and a batched one
// of Wv as it is stored, they took 32 + 42 us (8192 rows of 512, 16 heads of 128 +
// 128; 34 GFLOP, 80 MB), here 47 with the transposition: 8 K steps a tile, whose
// start and end take as long.
__global__ __launch_bounds__(512, 2) void latent_kv_kernel(GemmArgs a,
                                                               const short* w2,
                                                               const int N1,
                                                               const int T) {
  __shared__ __attribute__((aligned(128))) short lds[LDS];
  const int ntiles = (a.N + BN - 1) / BN, mtiles = (T + 255) / 256;
  const int total = ntiles * mtiles, share = (total + 7) / 8;
  const int t = blockIdx.x % 8 * share + blockIdx.x / 8;
  if ((int)blockIdx.x / 8 >= share || t >= total) return;
  const int blk = t / (NG * mtiles), in_blk = t - blk * NG * mtiles;
  const int wide = min(NG, ntiles - blk * NG);
  const int n0 = (blk * NG + in_blk % wide) * BN, m0 = in_blk / wide * 256;
  if (n0 >= N1) a.w = w2 - (int64_t)N1 * a.K;
  grouped_tile<256, BN, 2, 0, DOWN>(a, lds, 0, m0, T, n0);
}

// w [H, K, V] -> out [H, V, K], by squares of 64
__global__ __launch_bounds__(256) void transpose_heads_kernel(
    short* __restrict__ out, const short* __restrict__ w, const int K,
    const int V) {
  __shared__ short tile[64][72];
  const int k0 = blockIdx.x * 64, v0 = blockIdx.y * 64;
  const int64_t head = (int64_t)blockIdx.z * K * V;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int s = i * 256 + threadIdx.x, r = s / 8, c = s % 8 * 8;
    *reinterpret_cast<short8_t*>(&tile[r][c]) =
        *reinterpret_cast<const short8_t*>(w + head + (int64_t)(k0 + r) * V +
                                           v0 + c);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int s = i * 256 + threadIdx.x, r = s / 8, c = s % 8 * 8;
    short8_t o;
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = tile[c + j][r];
    *reinterpret_cast<short8_t*>(out + head + (int64_t)(v0 + r) * K + k0 + c) =
        o;
  }
}

struct CombineArgs {
  const void* y;
  const int *pos, *topi;            // pos: none where rows are the pairs
  const float* topw;
  const short* x;
  const float* w_id;
  const short* shared;
  int K, H, e_lo, e_hi;
};

// eight outputs of token t from c on
template <typename Y>
KAITO_DEV void combine8(const CombineArgs& a, const int64_t t, const int c,
                        float (&acc)[8]) {
  auto add = [&](const auto* p, const float w) {
    if constexpr (sizeof(*p) == 4) {
      const float4_t* v = reinterpret_cast<const float4_t*>(p + c);
      const float4_t lo = v[0], hi = v[1];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        acc[e] += w * lo[e];
        acc[e + 4] += w * hi[e];
      }
    } else {
      const short8_t v = *reinterpret_cast<const short8_t*>(p + c);
#pragma unroll
      for (int e = 0; e < 8; e++) acc[e] += w * bf16_to_f32(v[e]);
    }
  };
#pragma unroll
  for (int e = 0; e < 8; e++) acc[e] = 0.f;
  if (a.w_id) add(a.x + t * a.H, a.w_id[t]);
  for (int k = 0; k < a.K; k++) {
    const int64_t p = t * a.K + k;
    const int e = a.topi[p];
    if (e >= a.e_lo && e < a.e_hi)            // experts of this rank
      add((const Y*)a.y + (a.pos ? a.pos[p] : p) * a.H, a.topw[p]);
  }
  if (a.shared) add(a.shared + t * a.H, 1.0f);
}

// one workgroup per token, 8 outputs per thread and pass
template <typename O, typename Y>
__global__ __launch_bounds__(256) void moe_combine_kernel(O* __restrict__ out,
                                                          const CombineArgs a) {
  const int64_t t = blockIdx.x;
  for (int c = threadIdx.x * 8; c < a.H; c += 2048) {
    float acc[8];
    combine8<Y>(a, t, c, acc);
    if constexpr (sizeof(O) == 4) {
      float4_t* o = reinterpret_cast<float4_t*>(out + t * a.H + c);
      o[0] = float4_t{acc[0], acc[1], acc[2], acc[3]};
      o[1] = float4_t{acc[4], acc[5], acc[6], acc[7]};
    } else {
      short8_t o;
#pragma unroll
      for (int e = 0; e < 8; e++) o[e] = f32_to_bf16(acc[e]);
      *reinterpret_cast<short8_t*>(out + t * a.H + c) = o;
    }
  }
}

// The same with the residual norm behind it; rows stay in registers, up to 8 *
// ITER per thread. R bf16: residual += sum, out = rms(residual) * w; R f32:
// residual += rms(sum) * w, out = residual. The sum is rounded to bf16 first, as
// where it is stored. 32 rows of 2048: a launch less, 4.8 + 4.6 us -> 4.6; 8192:
// 19 + 24 -> 30.
template <typename R, typename Y, int ITER>
__global__ __launch_bounds__(256) void moe_combine_norm_kernel(
    short* __restrict__ out, R* __restrict__ residual,
    const R* __restrict__ w, const float eps, const CombineArgs a) {
  __shared__ float red[4];
  const int64_t t = blockIdx.x;
  float v[ITER][8], r[ITER][8], g[ITER][8];
  auto load8 = [](const R* p, float (&f)[8]) {
    if constexpr (sizeof(R) == 4) {
      const float4_t* q = reinterpret_cast<const float4_t*>(p);
#pragma unroll
      for (int e = 0; e < 8; e++) f[e] = q[e / 4][e % 4];
    } else {
      const short8_t q = *reinterpret_cast<const short8_t*>(p);
#pragma unroll
      for (int e = 0; e < 8; e++) f[e] = bf16_to_f32(q[e]);
    }
  };
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = i * 2048 + threadIdx.x * 8;
    if (c >= a.H) break;
    load8(residual + t * a.H + c, r[i]);
    load8(w + c, g[i]);
    combine8<Y>(a, t, c, v[i]);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] = bf16_to_f32(f32_to_bf16(v[i][e]));
      if constexpr (sizeof(R) == 2)
        v[i][e] = bf16_to_f32(f32_to_bf16(v[i][e] + r[i][e]));
      ss += v[i][e] * v[i][e];
    }
  }
  ss = wave_reduce_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = sizeof(R) == 2 ? rsqrtf(ss / (float)a.H + eps)
                                   : 1.0f / sqrtf(ss / (float)a.H + eps);
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int c = i * 2048 + threadIdx.x * 8;
    if (c >= a.H) break;
    short8_t o;
    if constexpr (sizeof(R) == 2) {
      short8_t s;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        s[e] = f32_to_bf16(v[i][e]);
        o[e] = f32_to_bf16(v[i][e] * inv * g[i][e]);
      }
      *reinterpret_cast<short8_t*>(residual + t * a.H + c) = s;
    } else {
      float4_t* q = reinterpret_cast<float4_t*>(residual + t * a.H + c);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        r[i][e] += v[i][e] * inv * g[i][e];
        o[e] = f32_to_bf16(r[i][e]);
      }
      q[0] = float4_t{r[i][0], r[i][1], r[i][2], r[i][3]};
      q[1] = float4_t{r[i][4], r[i][5], r[i][6], r[i][7]};
    }
    *reinterpret_cast<short8_t*>(out + t * a.H + c) = o;
  }
}

template <int KIND>
void launch_grouped(const GemmArgs& a, int64_t TK) {
  constexpr int COLS = is_gated(KIND) ? BN / 2 : BN;
  const int64_t ntiles = (a.N + COLS - 1) / COLS;
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto bm) {
    constexpr int BM = decltype(bm)::value;
    // most row tiles that TK rows in E groups can make
    const int64_t most = TK / BM + std::min<int64_t>(a.E, TK);
    // per XCD, a rest's quarters in place of its tiles
    const int64_t quarters = BM == 256 ? 3 * 2 * QUARTER_REST : 0;
    hipLaunchKernelGGL((moe_grouped_kernel<BM, KIND>),
        dim3(((most * ntiles + 7) / 8 + quarters) * 8), dim3(512), 0, stream,
        a);
  };
  // half tiles where an expert's rows would leave most of a whole one empty
  if (TK >= 192 * (int64_t)a.E) launch(std::integral_constant<int, 256>{});
  else launch(std::integral_constant<int, 128>{});
}

void check16(const at::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
              t.dtype() == at::kBFloat16 &&
              (uintptr_t)t.data_ptr() % 16 == 0);
}
void check_int(const at::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dtype() == at::kInt);
}

}  // namespace

void moe_grouped_up(at::Tensor act, at::Tensor x, at::Tensor w,
                    at::Tensor sorted_ids, at::Tensor offsets, at::Tensor bias,
                    int64_t act_mode, int64_t e_base, double act_limit) {
  check16(act); check16(x); check16(w);
  check_int(sorted_ids); check_int(offsets);
  const bool plain = act_mode == 2;
  TORCH_CHECK(act.dim() == 2 && x.dim() == 2 && w.dim() == 3);
  GemmArgs a{};
  a.E = (int)w.size(0); a.N = (int)act.size(1); a.K = (int)x.size(1);
  a.e_base = (int)e_base;
  TORCH_CHECK(w.size(1) == (plain ? 1 : 2) * (int64_t)a.N &&
              w.size(2) == a.K && a.K % BK == 0 && a.N % 64 == 0 && a.K > 0);
  TORCH_CHECK(e_base >= 0 && offsets.numel() > e_base + a.E &&
              sorted_ids.numel() == act.size(0));
  TORCH_CHECK(act_mode >= 0 && act_mode <= 2);
  if (bias.numel() > 0) {
    check16(bias);
    TORCH_CHECK(!plain && bias.numel() == (int64_t)a.E * 2 * a.N);
    a.bias = (const short*)bias.data_ptr();
  }
  a.out = (short*)act.data_ptr();
  a.x = (const short*)x.data_ptr();
  // expert indices count from e_base in the offsets, from 0 in the weights
  a.w = (const short*)w.data_ptr() - e_base * w.stride(0);
  if (a.bias) a.bias -= e_base * 2 * a.N;
  a.rows = sorted_ids.data_ptr<int>();
  at::Tensor gathered;
  if (x.numel() >= 1LL << 31) {     // beyond 32-bit byte offsets
    gathered = x.index_select(0, sorted_ids);
    a.x = (const short*)gathered.data_ptr();
    a.rows = nullptr;
  }
  a.offsets = offsets.data_ptr<int>();
  a.limit = (float)act_limit;
  if (act.size(0) == 0 || a.E == 0 || a.N == 0) return;
  if (plain) launch_grouped<UP_PLAIN>(a, act.size(0));
  else if (act_mode == 1) launch_grouped<UP_CLAMPED>(a, act.size(0));
  else launch_grouped<UP_GATED>(a, act.size(0));
}

void moe_grouped_down(at::Tensor y, at::Tensor act, at::Tensor w,
                      at::Tensor offsets, at::Tensor bias, int64_t e_base) {
  const bool wide = y.dtype() == at::kFloat;
  if (wide) {
    TORCH_CHECK(y.is_cuda() && y.is_contiguous() &&
                (uintptr_t)y.data_ptr() % 16 == 0);
  } else {
    check16(y);
  }
  check16(act); check16(w); check_int(offsets);
  TORCH_CHECK(y.dim() == 2 && act.dim() == 2 && w.dim() == 3 &&
              y.size(0) == act.size(0));
  GemmArgs a{};
  a.E = (int)w.size(0); a.N = (int)y.size(1); a.K = (int)act.size(1);
  a.e_base = (int)e_base;
  TORCH_CHECK(w.size(1) == a.N && w.size(2) == a.K && a.K % BK == 0 &&
              a.N % 64 == 0 && a.K > 0);
  TORCH_CHECK(e_base >= 0 && offsets.numel() > e_base + a.E);
  if (bias.numel() > 0) {
    check16(bias);
    TORCH_CHECK(bias.numel() == (int64_t)a.E * a.N);
    a.bias = (const short*)bias.data_ptr() - e_base * a.N;
  }
  if (wide) a.out32 = y.data_ptr<float>();
  else a.out = (short*)y.data_ptr();
  a.x = (const short*)act.data_ptr();
  a.w = (const short*)w.data_ptr() - e_base * w.stride(0);
  a.offsets = offsets.data_ptr<int>();
  if (y.size(0) == 0 || a.E == 0 || a.N == 0) return;
  launch_grouped<DOWN>(a, y.size(0));
}

// kv [T, H D + H V]: c [T, K] times wk [H, D, K] (rows K long) and wv [H, K, V]
void latent_kv(at::Tensor kv, at::Tensor c, at::Tensor wk, at::Tensor wv) {
  check16(kv); check16(c); check16(wk); check16(wv);
  TORCH_CHECK(c.dim() == 2 && kv.dim() == 2 && wk.dim() == 3 && wv.dim() == 3);
  const int64_t T = c.size(0), K = c.size(1), H = wk.size(0), V = wv.size(2);
  const int64_t N1 = H * wk.size(1);
  TORCH_CHECK(wk.size(2) == K && wv.size(0) == H && wv.size(1) == K &&
              kv.size(0) == T && kv.size(1) == N1 + H * V &&
              K % 64 == 0 && K > 0 && V % 64 == 0 && N1 % BN == 0 &&
              T < (1ll << 22) && kv.size(1) < (1ll << 22));
  if (T == 0 || H == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const at::Tensor wt = at::empty({H, V, K}, wv.options());
  hipLaunchKernelGGL(transpose_heads_kernel, dim3(K / 64, V / 64, H),
                     dim3(256), 0, stream, (short*)wt.data_ptr(),
                     (const short*)wv.data_ptr(), (int)K, (int)V);
  GemmArgs a{};
  a.out = (short*)kv.data_ptr();
  a.x = (const short*)c.data_ptr();
  a.w = (const short*)wk.data_ptr();
  a.E = 1;
  a.N = (int)kv.size(1);
  a.K = (int)K;
  const int64_t tiles = (T + 255) / 256 * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL(latent_kv_kernel, dim3((tiles + 7) / 8 * 8),
                     dim3(512), 0, stream, a, (const short*)wt.data_ptr(),
                     (int)N1, (int)T);
}

// checks shared by both sums
static CombineArgs combine_args(const at::Tensor& y, const at::Tensor& pos,
                                const at::Tensor& topi, const at::Tensor& topw,
                                const at::Tensor& x, const at::Tensor& w_id,
                                const at::Tensor& shared, int64_t T, int64_t H,
                                int64_t e_base, int64_t e_local) {
  if (y.dtype() == at::kFloat) {
    TORCH_CHECK(y.is_cuda() && y.is_contiguous() &&
                (uintptr_t)y.data_ptr() % 16 == 0);
  } else {
    check16(y);
  }
  const bool has_pos = pos.numel() > 0;
  check_int(topi);
  TORCH_CHECK(topw.is_cuda() && topw.is_contiguous() &&
              topw.dtype() == at::kFloat && topi.dim() == 2 &&
              topw.sizes() == topi.sizes());
  if (has_pos) {
    check_int(pos);
    TORCH_CHECK(pos.numel() == topi.numel());
  }
  const int64_t K = topi.size(1);
  TORCH_CHECK(H % 8 == 0 && topi.size(0) == T && y.size(0) == T * K &&
              y.size(1) == H);
  const bool ids = w_id.numel() > 0, sh = shared.numel() > 0;
  if (ids) {
    check16(x);
    TORCH_CHECK(x.size(0) == T && x.size(1) == H && w_id.numel() == T &&
                w_id.dtype() == at::kFloat && w_id.is_contiguous());
  }
  if (sh) {
    check16(shared);
    TORCH_CHECK(shared.dim() == 2 && shared.size(0) == T &&
                shared.size(1) == H);
  }
  CombineArgs a{};
  a.y = y.data_ptr();
  a.pos = has_pos ? pos.data_ptr<int>() : nullptr;
  a.topi = topi.data_ptr<int>();
  a.topw = topw.data_ptr<float>();
  a.x = ids ? (const short*)x.data_ptr() : nullptr;
  a.w_id = ids ? w_id.data_ptr<float>() : nullptr;
  a.shared = sh ? (const short*)shared.data_ptr() : nullptr;
  a.K = (int)K; a.H = (int)H;
  a.e_lo = (int)e_base; a.e_hi = (int)(e_base + e_local);
  return a;
}

void moe_combine(at::Tensor out, at::Tensor y, at::Tensor pos, at::Tensor topi,
                 at::Tensor topw, at::Tensor x, at::Tensor w_id,
                 at::Tensor shared, int64_t e_base, int64_t e_local) {
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() && out.dim() == 2 &&
              (out.dtype() == at::kFloat || out.dtype() == at::kBFloat16) &&
              (uintptr_t)out.data_ptr() % 16 == 0);
  const int64_t T = out.size(0), H = out.size(1);
  const CombineArgs a = combine_args(y, pos, topi, topw, x, w_id, shared, T, H,
                                     e_base, e_local);
  if (T == 0 || H == 0) return;
#define MC_LAUNCH(O_, Y_)                                                     \
  hipLaunchKernelGGL((moe_combine_kernel<O_, Y_>), dim3(T), dim3(256), 0,     \
      at::hip::getCurrentHIPStream(), (O_*)out.data_ptr(), a)
  const bool wide = y.dtype() == at::kFloat;
  if (out.dtype() == at::kFloat) {
    if (wide) MC_LAUNCH(float, float); else MC_LAUNCH(float, short);
  } else {
    if (wide) MC_LAUNCH(short, float); else MC_LAUNCH(short, short);
  }
#undef MC_LAUNCH
}

void moe_combine_norm(at::Tensor out, at::Tensor residual, at::Tensor y,
                      at::Tensor pos, at::Tensor topi, at::Tensor topw,
                      at::Tensor x, at::Tensor w_id, at::Tensor shared,
                      at::Tensor weight, double eps, int64_t e_base,
                      int64_t e_local) {
  check16(out);
  TORCH_CHECK(out.dim() == 2 && residual.sizes() == out.sizes() &&
              weight.numel() == out.size(1) &&
              weight.dtype() == residual.dtype());
  for (const auto& t : {residual, weight})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() &&
                (t.dtype() == at::kFloat || t.dtype() == at::kBFloat16) &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  const int64_t T = out.size(0), H = out.size(1);
  TORCH_CHECK(H <= 8192);
  const CombineArgs a = combine_args(y, pos, topi, topw, x, w_id, shared, T, H,
                                     e_base, e_local);
  if (T == 0 || H == 0) return;
#define MC_LAUNCH(R_, Y_, IT_)                                                \
  hipLaunchKernelGGL((moe_combine_norm_kernel<R_, Y_, IT_>), dim3(T),         \
      dim3(256), 0, at::hip::getCurrentHIPStream(), (short*)out.data_ptr(),   \
      (R_*)residual.data_ptr(), (const R_*)weight.data_ptr(), (float)eps, a)
#define MC_ITER(R_, Y_)                                                       \
  if (H <= 2048) MC_LAUNCH(R_, Y_, 1);                                        \
  else if (H <= 4096) MC_LAUNCH(R_, Y_, 2);                                   \
  else MC_LAUNCH(R_, Y_, 4)
  const bool wide = y.dtype() == at::kFloat;
  if (residual.dtype() == at::kFloat) {
    if (wide) { MC_ITER(float, float); } else { MC_ITER(float, short); }
  } else {
    if (wide) { MC_ITER(short, float); } else { MC_ITER(short, short); }
  }
#undef MC_ITER
#undef MC_LAUNCH
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("moe_grouped_up(Tensor(a!) act, Tensor x, Tensor w, Tensor sorted_ids, Tensor offsets, Tensor bias, int act_mode, int e_base, float act_limit) -> ()");
  m.def("moe_grouped_down(Tensor(a!) y, Tensor act, Tensor w, Tensor offsets, Tensor bias, int e_base) -> ()");
  m.def("latent_kv(Tensor(a!) kv, Tensor c, Tensor wk, Tensor wv) -> ()");
  m.def("moe_combine(Tensor(a!) out, Tensor y, Tensor pos, Tensor topi, Tensor topw, Tensor x, Tensor w_id, Tensor shared, int e_base, int e_local) -> ()");
  m.def("moe_combine_norm(Tensor(a!) out, Tensor(b!) residual, Tensor y, Tensor pos, Tensor topi, Tensor topw, Tensor x, Tensor w_id, Tensor shared, Tensor weight, float eps, int e_base, int e_local) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("moe_combine_norm", &kaito::moe_combine_norm);
  m.impl("moe_grouped_up", &kaito::moe_grouped_up);
  m.impl("moe_grouped_down", &kaito::moe_grouped_down);
  m.impl("latent_kv", &kaito::latent_kv);
  m.impl("moe_combine", &kaito::moe_combine);
}
