// Products of few rows with a large weight matrix, out[M, N] = x[M, K] W^T:
// the linear layers of a decode step. They stream W once, so the designs are
// about bytes in flight and the order of addresses; arithmetic is small.
//
// M <= 4: a wave streams whole rows, 1 KB of one row per load (full lines, in
// address order, marked non-temporal), and multiplies on the vector unit
// (dot2, f32 sums). On one MI355X, N = 28672, K = 4096, M = 1: 33.6 us, 7.0
// TB/s; the same rows read as MFMA operands (64 B of 16 rows per load) 45.7
// us, hipBLASLt's tuned choice 57.5 us.
//
// Up to 32 rows of x, and experts with a few rows each: the same streams
// through LDS into v_mfma_f32_16x16x32_bf16 (stream_tile). A workgroup owns
// 16 rows of W; its waves take every fourth slice of K and meet in LDS, in
// f32. 28672 x 4096: 44.4 us at M = 8 (library 56.8), 50.9 at 16 (57.4), 72.8 at
// 32 (48.6): x comes through the caches once per workgroup, so the gain ends
// where its rows cost what those of W do. Where x fits the registers,
// workgroups stay for many tiles (stream_tiles): 40.1 at 8, 41.8 at 16. K in
// stages of 64, 2880 x 2880: 6.5 at 8 (16.3), 6.8 at 16 (16.4).
//
// 4-bit weights run as integers. Read as fp8 (e4m3, subnormals and the first
// binade), a byte of 0 to 15 is exactly q / 512: two masks and four packed
// conversions turn a word's nibbles into bf16 (x is permuted to match), and
// per group of K, in f32,
//     y += 512 s (sum (q / 512) x) - z sum x
#pragma once
#include "common.h"

namespace kaito {
namespace skinny {

typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 hbf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

KAITO_DEV f32x4 mfma16(hbf16x8 a, hbf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// streamed once: leave the caches to x
template <typename V>
KAITO_DEV V load_stream(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const V*>(p));
}

KAITO_DEV hbf16x8 load_x(const short* p) {
  return *reinterpret_cast<const hbf16x8*>(p);
}

// ---- up to 32 rows of x: 16 rows of W per workgroup through LDS -------------
// A stage is 16 rows x KS k, copied by 16-byte direct loads in pieces of KS *
// 2 contiguous bytes (whole lines), 16-byte chunk c of row r at c ^ (r & 7).
// Two stages per wave: the next one, and the x operands beside it, are under
// way while the present one is multiplied. Nothing is shared between waves, so
// the waits are counts of this wave's own loads and there are no barriers.
constexpr int TILE_NW = 4;          // waves per workgroup, over K

// direct loads per lane and stage of 16 rows x KS k
template <int KS>
constexpr int tile_loads() { return 16 * KS / 512; }

// row of the 16 that load j of this lane copies, and the element offset of
// its piece inside the row's stage
template <int KS>
KAITO_DEV int tile_row(const int j, const int lane) {
  return j * (512 / KS) + lane / (KS / 8);
}
template <int KS>
KAITO_DEV int tile_col(const int j, const int lane) {
  return ((lane % (KS / 8)) ^ (tile_row<KS>(j, lane) & 7)) * 8;
}

template <int N>
KAITO_DEV void wait_loads() {       // until N of this wave's loads are left
  __builtin_amdgcn_sched_barrier(0);        // every one of them is issued
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

// acc[mt] += x rows 16 mt.. times the 16 rows of W. src[j]: source of load j
// (tile_row, tile_col); xp[mt]: the lane's x row (lane & 15) at 8 (lane >> 4);
// ring: [2][16 * KS] of this wave. K is a multiple of KS.
template <int MT, int KS>
KAITO_DEV void stream_tile(f32x4 (&acc)[MT],
                           const short* const (&src)[tile_loads<KS>()],
                           const short* const (&xp)[MT], short* ring,
                           const int K, const int wave, const int lane) {
  constexpr int NI = tile_loads<KS>(), STEPS = KS / 32;
  const int n = K / KS, lo = lane & 15, hi = lane >> 4;
  hbf16x8 xf[2][MT][STEPS];
  auto fetch = [&](const int s, const int b) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int i = 0; i < STEPS; i++)
        xf[b][mt][i] = load_x(xp[mt] + s * KS + i * 32);
#pragma unroll
    for (int j = 0; j < NI; j++)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) unsigned int*)(src[j] +
                                                                  s * KS),
          (__attribute__((address_space(3))) unsigned int*)(
              ring + b * 16 * KS + j * 512),
          16, 0, 2 /* non-temporal */);
  };
  auto multiply = [&](const int b) {
    const short* w = ring + b * 16 * KS + lo * KS;
#pragma unroll
    for (int i = 0; i < STEPS; i++) {
      const hbf16x8 wf =
          load_x(w + (((i * 4 + hi) ^ (lo & 7)) * 8));
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
        acc[mt] = mfma16(xf[b][mt][i], wf, acc[mt]);
    }
  };
  // Every step fetches or none does: where the two met in one product, the
  // compiler could no longer count the loads and waited for all of them.
  auto step = [&](const int s, const int b) {
    // the other stage's reads are done before it is overwritten
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
    fetch(s + TILE_NW, b ^ 1);
    wait_loads<MT * STEPS + NI>();
    multiply(b);
  };
  auto last = [&](const int b) {
    wait_loads<0>();
    multiply(b);
  };
  if (wave >= n) return;
  fetch(wave, 0);
  int s = wave;
  for (; s + 2 * TILE_NW < n; s += 2 * TILE_NW) {
    step(s, 0);
    step(s + TILE_NW, 1);
  }
  if (s + TILE_NW < n) {
    step(s, 0);
    last(1);
  } else {
    last(0);
  }
}

// ---- the same over many tiles ----------------------------------------------
// Where K is 4 S stages of 256, a wave's slices of x fit its registers: they
// are read once, and the workgroup goes from tile to tile with the next stage
// always under way, also across the sum over its waves. Tiles of their own
// workgroups (stream_tile) spend as long on offsets, x and the sum as on 64 KB
// of weights, and no more than two of them fit a CU.
constexpr int TILES_KS = 256;

// Sums of the 16 rows of W of tiles first, first + step .. < n. rows(j): byte
// offset of load j's piece from the start of tile 0, which lies at w, and with TWO
// so from tile n1, which lies at w2; tile: bytes from a tile to the next; xp: as
// for stream_tile, asked for once the first weights are under way. ring: [2][16 * 256] of this wave, red:
// [2][4][MT * 64] of the workgroup. out(tile, sums): on every thread, the sums
// of the waves for fold().
template <int MT, int S, bool TWO, typename Rows, typename X, typename Out>
KAITO_DEV void stream_tiles(const void* w, const void* w2, const int n1,
                            const Rows& rows, const uint32_t tile,
                            const int first, const int step, const int n,
                            const X& x, short* ring, f32x4* red,
                            const int wave, const int lane, const Out& out) {
  constexpr int KS = TILES_KS, NI = tile_loads<KS>(), STEPS = KS / 32;
  static_assert(S % 2 == 0, "a tile starts in ring 0");
  if (first >= n) return;           // uniform
  uint32_t off[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) off[j] = rows(j);
  const auto wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(w), 0, 0xffffffff, 0x27000);
  // past the last tile: loads of nothing, so that the waits stay counts
  const auto none = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(w), 0, 0, 0x27000);
  auto fetch = [&](const int t, const int s) {
    auto r = t < n ? wb : none;
    bool second = false;
    if constexpr (TWO) {
      // a descriptor that is scalar for sure: one of two chosen by the tile was
      // looked for lane by lane, which doubled the time
      second = t >= n1;
      const uint64_t from = reinterpret_cast<uint64_t>(second ? w2 : w);
      r = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<void*>(
              (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)from) |
              (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(
                  (int)(from >> 32)) << 32),
          0, __builtin_amdgcn_readfirstlane(t < n ? -1 : 0), 0x27000);
    }
    const uint32_t at = __builtin_amdgcn_readfirstlane(
        (second ? t - n1 : t) * tile + (wave + s * TILE_NW) * KS * 2);
#pragma unroll
    for (int j = 0; j < NI; j++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r,
          (__attribute__((address_space(3))) void*)(ring + (s & 1) * 16 * KS +
                                                    j * 512),
          16, off[j], at, 0, 2 /* non-temporal */);
  };
  fetch(first, 0);
  fetch(first, 1);
  hbf16x8 xf[S][MT][STEPS];
  {
    const short* xp[MT];
    x(xp);
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < STEPS; i++)
          xf[s][mt][i] =
              load_x(xp[mt] + (wave + s * TILE_NW) * KS + i * 32);
  }
  wait_loads<0>();                  // none of x is left for the loop's counts
  const int lo = lane & 15, hi = lane >> 4;
  int par = 0;
  for (int t = first; t < n; t += step) {
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; s++) {
      wait_loads<NI>();             // this stage's; the next is under way
      const short* p = ring + (s & 1) * 16 * KS + lo * KS;
#pragma unroll
      for (int i = 0; i < STEPS; i++) {
        const hbf16x8 wf = load_x(p + (((i * 4 + hi) ^ (lo & 7)) * 8));
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          acc[mt] = mfma16(xf[s][mt][i], wf, acc[mt]);
      }
      // its reads are done before it is overwritten
      __builtin_amdgcn_s_waitcnt(0xc07f);
      asm volatile("" ::: "memory");
      if (s + 2 < S) fetch(t, s + 2);
      else fetch(t + step, s + 2 - S);
    }
    f32x4* sums = red + par * TILE_NW * MT * 64;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
      sums[(wave * MT + mt) * 64 + lane] = acc[mt];
    // own sums written, the next weights still under way; the other half of
    // red is free once all are here
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    out(t, sums);
    par ^= 1;
  }
  wait_loads<0>();                  // no copy to LDS outlives the workgroup's
}

// the eight nibbles of a word as bf16 q / 512, in the order 0 2 4 6 1 3 5 7
KAITO_DEV hbf16x8 nibbles(const unsigned int w) {
  const unsigned int even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
  const hbf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 1.f, false);
  const hbf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 1.f, true);
  const hbf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 1.f, false);
  const hbf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 1.f, true);
  return hbf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
constexpr float NIBBLE = 512.f;     // q over its bf16 form

// x in that order
KAITO_DEV hbf16x8 nibble_order(const hbf16x8 x) {
  return __builtin_shufflevector(x, x, 0, 2, 4, 6, 1, 3, 5, 7);
}

// 4-bit weights [N, K / 8]; WORDS words per lane and slice: a slice is
// WORDS * 32 k and lies in one group (WORDS 4: groups of 128 n, 2: of 64 n).
// A lane's k are 8 WORDS (l >> 4) onward; sc/ze: the lane's rows.
template <int MT, int NT, int WORDS>
KAITO_DEV void accumulate_w4(f32x4 (&acc)[MT][NT],
                             const unsigned int* const (&wp)[NT],
                             const float* const (&sc)[NT],
                             const float* const (&ze)[NT],
                             const short* const (&xp)[MT], const int K,
                             const int group, const int wave, const int nw) {
  constexpr int KC = WORDS * 32;
  constexpr int U = MT * NT <= 2 ? 2 : 1;       // slices under way
  typedef unsigned int wordv __attribute__((ext_vector_type(WORDS)));
  const hbf16x8 ones = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
  for (int k0 = wave * U * KC; k0 < K; k0 += nw * U * KC) {
    wordv w[U][NT];
    float s[U][NT], z[U][NT];
    hbf16x8 xf[U][MT][WORDS];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = min(k0 + u * KC, K - KC);   // past the end: weighed zero
      const float live = k0 + u * KC < K ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < NT; j++) {
        w[u][j] = load_stream<wordv>(wp[j] + k / 8);
        s[u][j] = sc[j][k / group] * (live * NIBBLE);
        z[u][j] = ze[j][k / group] * live;
      }
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < WORDS; i++)
          xf[u][mt][i] = load_x(xp[mt] + k + i * 8);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      f32x4 xs[MT], dot[MT][NT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        xs[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NT; j++) dot[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int i = 0; i < WORDS; i++) {
        hbf16x8 q[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) q[j] = nibbles(w[u][j][i]);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          const hbf16x8 xv = nibble_order(xf[u][mt][i]);
          xs[mt] = mfma16(xv, ones, xs[mt]);
#pragma unroll
          for (int j = 0; j < NT; j++)
            dot[mt][j] = mfma16(xv, q[j], dot[mt][j]);
        }
      }
#pragma unroll
      for (int j = 0; j < NT; j++) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[mt][j][r] += s[u][j] * dot[mt][j][r] - z[u][j] * xs[mt][r];
      }
    }
  }
}

// Sums of the waves' tiles: thread (slot = tile * 64 + lane) gets its f32x4.
// red: [NW][TILES * 64]
template <int TILES, int NW>
KAITO_DEV f32x4 fold(const f32x4* red, const int slot) {
  f32x4 v = red[slot];
#pragma unroll
  for (int w = 1; w < NW; w++) v += red[w * TILES * 64 + slot];
  return v;
}

// ---- M <= 4: rows streamed by a wave ---------------------------------------

KAITO_DEV float dot8(const hbf16x8 a, const hbf16x8 b, float c) {
  const hbf16x2* p = reinterpret_cast<const hbf16x2*>(&a);
  const hbf16x2* q = reinterpret_cast<const hbf16x2*>(&b);
#pragma unroll
  for (int i = 0; i < 4; i++)
    c = __builtin_amdgcn_fdot2_f32_bf16(p[i], q[i], c, false);
  return c;
}

// acc[m][r] += x row m . W row r, this lane's k only. wp: row starts.
template <int M, int R>
KAITO_DEV void stream_rows(float (&acc)[M][R], const short* const (&wp)[R],
                           const short* x, const int64_t x_stride,
                           const int K, const int lane) {
  constexpr int U = M * R <= 4 ? 4 : 2;
  int k0 = 0;
  for (; k0 + 512 * U <= K; k0 += 512 * U) {
    hbf16x8 w[U][R], v[U][M];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int r = 0; r < R; r++)
        w[u][r] = load_stream<hbf16x8>(wp[r] + k0 + u * 512 + lane * 8);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int m = 0; m < M; m++)
        v[u][m] = load_x(x + m * x_stride + k0 + u * 512 + lane * 8);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[m][r] = dot8(w[u][r], v[u][m], acc[m][r]);
  }
  for (int k = k0 + lane * 8; k < K; k += 512) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const hbf16x8 w = load_stream<hbf16x8>(wp[r] + k);
#pragma unroll
      for (int m = 0; m < M; m++)
        acc[m][r] = dot8(w, load_x(x + m * x_stride + k), acc[m][r]);
    }
  }
}

// the same for 4-bit rows: a lane's 16 bytes are 32 k of one group
template <int M, int R>
KAITO_DEV void stream_rows_w4(float (&acc)[M][R],
                              const unsigned int* const (&wp)[R],
                              const float* const (&sc)[R],
                              const float* const (&ze)[R], const short* x,
                              const int64_t x_stride, const int K,
                              const int group, const int lane) {
  const hbf16x8 ones = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
  for (int k0 = lane * 32; k0 - lane * 32 < K; k0 += 2048) {
    const int k = min(k0, K - 32);
    const float live = k0 < K ? 1.f : 0.f;      // past the end: weighed zero
    u32x4 w[R];
    float s[R], z[R];
    hbf16x8 xv[M][4];
#pragma unroll
    for (int r = 0; r < R; r++) {
      w[r] = load_stream<u32x4>(wp[r] + k / 8);
      s[r] = sc[r][k / group] * (live * NIBBLE);
      z[r] = ze[r][k / group] * live;
    }
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        xv[m][i] = load_x(x + m * x_stride + k + i * 8);
    float dot[M][R], xs[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
      xs[m] = 0.f;
#pragma unroll
      for (int r = 0; r < R; r++) dot[m][r] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      hbf16x8 q[R];
#pragma unroll
      for (int r = 0; r < R; r++) q[r] = nibbles(w[r][i]);
#pragma unroll
      for (int m = 0; m < M; m++) {
        const hbf16x8 v = nibble_order(xv[m][i]);
        xs[m] = dot8(v, ones, xs[m]);
#pragma unroll
        for (int r = 0; r < R; r++) dot[m][r] = dot8(v, q[r], dot[m][r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int m = 0; m < M; m++)
        acc[m][r] += s[r] * dot[m][r] - z[r] * xs[m];
    }
  }
}

KAITO_DEV float silu(float v) { return silu_f32(v); }

}  // namespace skinny
}  // namespace kaito
