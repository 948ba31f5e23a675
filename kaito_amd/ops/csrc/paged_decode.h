// Paged-attention DECODE kernel for gfx950: one query row per sequence, the
// heads of a kv group in one pass over its K and V pages.
//
// A wave walks a contiguous span of keys, 32 at a time, with the products on
// v_mfma_f32_16x16x32_bf16, transposed as in flash_prefill.h (the group's
// heads are the 16 columns, unused ones ride along):
//   - S^T = K Q^T reads K straight from the pages into operand registers (a
//     16-byte load per lane is 8 dims of one key);
//   - the scores of one head sit in one column: maximum and rescale factor
//     are per-lane scalars after two exchanges;
//   - O^T += V^T P^T takes P from the score registers; V goes to wave-private
//     LDS by 16-byte direct loads and comes back by transposing reads.
// P enters as the sum of three bf16 terms, which hold every bit of the f32
// weight (two of them 16 of its 24). fp8 (e4m3) pages are widened to bf16,
// exactly, on the way: by pairs straight to bf16, 16 bytes a load (dims of K permuted
// to match, with q's), V through registers a tile ahead. By way of f32, 8 bytes a
// load and V asked for at the head of its own tile: 250 rows of 200 to 400 keys 48.9
// us, now 42.9; 64 of 700 to 1400 34.9, 31.7; 16 of 2050 to 4100 30.8, 28.2. bf16
// pages are bound by memory (57 us alone for the first, 66 here): the table and K
// ahead of q's rotation and the row's own key from registers changed nothing there,
// and cost 0.7 us of 8 where the code is fetched anew for every launch. The waves of a workgroup, and with SPLIT the
// workgroups of a (sequence, kv head), hold partial (max, sum, O) that are
// folded at the end.
//
// What bounds it: bytes in flight. K and V of a tile (16 KB per wave at
// D = 128) are all under way at once, while the arithmetic of a tile is
// about 500 cycles (2 x 16 scores and weights on the vector unit took
// 3000). Small steps are bound by the chain lengths -> table -> K -> V -> fold:
// hence 8 waves per workgroup, so that each walks few tiles, and workgroups per
// pair while those do not fill the chip; fewer waves where there are pairs
// enough (launch_paged_decode). Measured on one MI355X against a kernel with 4
// waves per pair, 16-byte K and V streams in two phases and dot products by dot2 +
// DPP sums (before -> now; 8 kv heads of 128, groups of 4):
//   1 row, 217 keys: 11.0 -> 6.4 us (8.0 where the table is wide enough for
//   splits);  16 rows of 4000: 194 -> 43, of 4000 fp8 keys 180 -> 28;  64 rows
//   of 800: 47 -> 34;  250 of 300: 68 -> 55;  2048 of 220: 429 -> 335 us.
// Two terms of P would take 0.1 to 5 % off.
//
// BIASED is the form of the hybrid stacks' windowed layers
// (window_attention.hip): scores with a tanh cap and a distance penalty, the
// mask on keys and not on values. The penalty is a log1pf, whose argument may be
// far below 1 (ln(1 + 1e-6) by logf is off by a twentieth); on every lane, unused
// columns too, it took 4 us of 23 (32 rows of a 1024-key window, 4 heads per kv
// head), shared out over the lanes and read back from LDS none, with 8 heads 2 of
// 16.
//
// ROPE takes q without its rotation and the row's own key and value beside the
// pages: a launch of 4.5 us less before it. The wave of the last keys stores them
// and then reads its pages as ever. The same bits as rope.hip and this kernel
// behind it; 1 row of 217 keys 9.3 -> 7.6 us, 32 of a 1024-key window 23.1 -> 19.7.
//
// Cache layout: [num_blocks, KV_HEADS, BLOCK_SIZE, HEAD_DIM] bf16 | e4m3.
#pragma once
#include "flash_prefill.h"
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

namespace {

using flash::hbf16x8;
using flash::LOG2E;
typedef uint8_t u8x16_t __attribute__((ext_vector_type(16)));

constexpr int BS = 16;              // tokens per page
constexpr int KT = 32;              // keys per wave step: two pages
constexpr int WIDE = 8;             // waves per workgroup while pairs are few
constexpr int64_t SPLIT_FILL = 256;  // workgroups that splits aim at
constexpr int SPLIT_MIN = 2;        // tiles per wave that a split keeps

struct DecodeArgs {
  short* out;                       // [T, QH, D]
  const short* q;
  const void *k, *v;                // [NB, KH, BS, D] bf16 | e4m3
  const int* block_tables;          // [T, max_blocks]
  const int* seq_lens;              // [T]
  float scale;
  int KH, G, max_blocks;
  int64_t q_stride;
  int window;                       // 0 = all keys
  const float* sinks;               // [QH] or nullptr
  float* part;                      // SPLIT: [splits, T, QH, D + 2]
  // BIASED: rows of any sequence, at positions of their own, scores in natural
  // units cap * tanh(scale q.k / cap) - r1 ln(1 + r2 distance)
  const int* token_seq;             // [T]: row of block_tables, < 0: none
  const int64_t* positions;         // [T], in place of seq_lens - 1
  float cap;                        // 0 = none
  const float *r1, *r2;             // [QH] or nullptr
  const short* gate;                // [T, ..]: sigmoid of it times the output
  int64_t gate_stride;
  // ROPE: q comes without its rotation, the row's own key and value outside the
  // pages; both go to their slot (< 0: none) first. positions as above
  const short *k_row, *v_row;       // [T, KH * D]
  int64_t k_stride, v_stride;
  const float* cos_sin;             // [positions, D]
  const int64_t* slots;             // [T]

  template <bool BIASED> KAITO_DEV int len(const int64_t row) const {
    return BIASED ? (int)positions[row] + 1 : seq_lens[row];
  }
};

// chunk of a V row -> its place: 8 rows x 16 columns, which half a wave's
// transposing read takes at once, lie in different eighths of 256 bytes
template <int D>
KAITO_DEV int place_v(const int row, const int c) {
  if constexpr (D == 64) return c ^ ((row >> 1 & 3) << 1);
  else return c ^ ((row & 7) << 1);
}

// eight of 16 e4m3 as bf16, exactly: half 0 the first, 1 the last
KAITO_DEV hbf16x8 widen8(const u8x16_t raw, const int half) {
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
  typedef __bf16 hbf16x2 __attribute__((ext_vector_type(2)));
  const u32x4 u = __builtin_bit_cast(u32x4, raw);
  hbf16x8 w;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const unsigned x = u[2 * half + i];
    const hbf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.f, false);
    const hbf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, 1.f, true);
    w[4 * i] = a[0];
    w[4 * i + 1] = a[1];
    w[4 * i + 2] = b[0];
    w[4 * i + 3] = b[1];
  }
  return w;
}

// weights of the partial results of one head: exponent of each maximum
// against the largest, summed with the sink's into the denominator. Natural units
// take expf: exp2 of the rounded product is off by up to 1e-6 of a weight of
// e^-20, expf by 8e-8 (32 rows of a 1024-key window: 19.8 and 20.9 us).
template <bool BIASED>
KAITO_DEV float fold_weight(float m, float gm) {
  return BIASED ? expf(m - gm) : __builtin_amdgcn_exp2f(m - gm);
}

template <bool BIASED>
KAITO_DEV void store_head(const DecodeArgs& a, const int64_t row, const int QH,
                          const int head, const int D, const int d,
                          const float num, const float den) {
  float v;
  if constexpr (BIASED) {
    v = num / den;
    if (a.gate)
      v /= 1.f + expf(-bf16_to_f32(a.gate[row * a.gate_stride + head]));
  } else {
    v = num / fmaxf(den, 1e-20f);
  }
  a.out[(row * QH + head) * D + d] = f32_to_bf16(v);
}

// The rotation of 8 dims x at d and their partners y at d + D / 2 of a head.
// Products and rounding as the compiler forms them in rope.hip: the same bits.
template <typename V>
KAITO_DEV void rotate8(V& x, V& y, const float* cs, const int half) {
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float c = cs[j], s = cs[half + j];
    const float a = (float)x[j], b = (float)y[j];
    x[j] = (__bf16)__builtin_fmaf(a, c, -(b * s));
    y[j] = (__bf16)__builtin_fmaf(b, c, a * s);
  }
}

// One wave: the row's key, rotated, and its value go to their slot of the pages
// and can be read from there by this wave.
template <int D, bool FP8>
KAITO_DEV void append_row(const DecodeArgs& a, const int64_t row, const int kvh,
                          const float* cs, const int lane) {
  const int64_t slot = a.slots[row];
  if (slot < 0) return;             // uniform
  const int64_t at = ((slot / BS * a.KH + kvh) * BS + slot % BS) * D;
  auto put = [&](const void* cache, const int d, const hbf16x8 x) {
    if constexpr (FP8) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; j++)
        w[j] = f32x2_to_fp8x2((float)x[2 * j], (float)x[2 * j + 1]) & 0xffff;
      const uint2 o = {w[0] | w[1] << 16, w[2] | w[3] << 16};
      *reinterpret_cast<uint2*>((uint8_t*)const_cast<void*>(cache) + at + d) = o;
    } else {
      *reinterpret_cast<hbf16x8*>((short*)const_cast<void*>(cache) + at + d) = x;
    }
  };
  const short* v = a.v_row + row * a.v_stride + kvh * D;
  const short* k = a.k_row + row * a.k_stride + kvh * D;
  if (lane < D / 8)
    put(a.v, lane * 8, *reinterpret_cast<const hbf16x8*>(v + lane * 8));
  if (lane < D / 16) {
    hbf16x8 x = *reinterpret_cast<const hbf16x8*>(k + lane * 8);
    hbf16x8 y = *reinterpret_cast<const hbf16x8*>(k + D / 2 + lane * 8);
    rotate8(x, y, cs + lane * 8, D / 2);
    put(a.k, lane * 8, x);
    put(a.k, D / 2 + lane * 8, y);
  }
  __threadfence_block();            // ahead of this wave's loads of the page
}

// how a sequence's keys are shared out: 32-key tiles from the page that
// holds the window's first key on, a contiguous run of `per` for every wave.
// A split is the share of a workgroup's waves, so that with `used` == 1 the
// first one has every key and writes the result itself.
struct Spans {
  int start, base, tiles, per, used;
};
KAITO_DEV Spans spans_of(const int seq_len, const int window, const int nsplit,
                         const int nw) {
  Spans p;
  p.start = window > 0 && seq_len > window ? seq_len - window : 0;
  p.base = p.start / BS * BS;
  p.tiles = (seq_len - p.base + KT - 1) / KT;
  p.per = (p.tiles + nsplit * nw - 1) / (nsplit * nw);
  p.used = p.per > 0 ? (p.tiles + p.per * nw - 1) / (p.per * nw) : 1;
  return p;
}

template <int D, bool FP8, int NW, bool SPLIT, bool BIASED, bool ROPE>
__global__ __launch_bounds__(NW * 64, NW <= 4 && D <= 128 ? 3 : 2)
void paged_decode_kernel(const DecodeArgs a) {
  constexpr int KK = D / 32;        // 16x16x32 steps over the dims
  constexpr int DT = D / 16;        // 16-row tiles of O^T
  constexpr int CV = D / 8;         // 16-byte chunks of a V row
  constexpr int LV = KT * CV / 64;  // V chunks per lane and tile
  // Dims of a lane in product step kk: 8 from d0 + step_dim(kk) on. fp8 rows of 128
  // dims and more: those of two steps are one load of 16 bytes
  constexpr bool QUADS = FP8 && D >= 128;
  auto step_dim = [](const int kk) {
    return QUADS ? kk / 2 * 64 + kk % 2 * 8 : kk * 32;
  };
  __shared__ __attribute__((aligned(128))) short lds_v[NW][KT * D];
  __shared__ float s_m[NW][16], s_l[NW][16];
  // BIASED: penalties of a wave's tile, heads by keys
  constexpr int PH = BIASED ? D <= 128 ? 8 : 4 : 1;
  __shared__ __attribute__((aligned(16))) float s_pen[BIASED ? NW : 1][PH * KT];

  const int seq = blockIdx.x / a.KH, kvh = blockIdx.x % a.KH;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int QH = a.KH * a.G;
  const int table = BIASED ? a.token_seq[seq] : seq;
  if (BIASED && table < 0) {        // a padding row
    if (!SPLIT || blockIdx.y == 0)
      for (int i = threadIdx.x; i < a.G * D; i += NW * 64)
        a.out[((int64_t)seq * QH + kvh * a.G) * D + i] = 0;
    return;
  }
  const int seq_len = a.len<BIASED>(seq);
  const int* bt = a.block_tables + (int64_t)table * a.max_blocks;

  const int nsplit = SPLIT ? gridDim.y : 1, split = SPLIT ? blockIdx.y : 0;
  const Spans sp = spans_of(seq_len, a.window, nsplit, NW);
  if (split >= sp.used) return;     // no keys: the fold does not look here
  const bool partial = SPLIT && sp.used > 1;
  const int start = sp.start, base = sp.base;
  const int t0 = min(sp.tiles, (split * NW + wave) * sp.per);
  const int t1 = min(sp.tiles, t0 + sp.per);
  const int last_page = (seq_len - 1) / BS;

  const int d0 = hi * (QUADS ? 16 : 8);
  hbf16x8 qf[KK];
  {
    const short* qp = a.q + (int64_t)seq * a.q_stride +
        (int64_t)(kvh * a.G) * D;
#pragma unroll
    for (int kk = 0; kk < KK; kk++)
      qf[kk] = *reinterpret_cast<const hbf16x8*>(
          qp + min(lo, a.G - 1) * D + d0 + step_dim(kk));
  }
  if constexpr (ROPE) {
    const float* cs = a.cos_sin + a.positions[seq] * D;
    // the wave of the last key, which is the row's own
    if (sp.tiles ? t0 < t1 && t1 == sp.tiles : wave == 0)
      append_row<D, FP8>(a, seq, kvh, cs, lane);
#pragma unroll
    for (int kk = 0; kk < KK / 2; kk++)
      rotate8(qf[kk], qf[kk + KK / 2], cs + d0 + step_dim(kk), D / 2);
  }
  constexpr float NONE = BIASED ? -INFINITY : -1e30f;
  float m = NONE, l = 0.f;
  // Penalties are evaluated once for each head and key, and not by the lanes of
  // unused columns too: lane % 32 is the key, its heads are lane / 32 + 2 j.
  float r1[PH / 2 + 1], r2[PH / 2 + 1];
  if (BIASED && a.r1) {
#pragma unroll
    for (int j = 0; j < PH / 2; j++) {
      const int head = kvh * a.G + min((lane >> 5) + 2 * j, a.G - 1);
      r1[j] = a.r1[head];
      r2[j] = a.r2[head];
    }
  }
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  short* vl = lds_v[wave];
  const int vrow = 4 * hi + (lo >> 2), vc = (lo & 3) >> 1, ve = (lo & 1) * 4;
  const float c = a.scale * LOG2E;

  int pages = 0, pages_at = -64;    // lane i: page pages_at + i of the table
  auto page_row = [&](const int p) {        // first cache row of page p
    const int pc = min(p, last_page);
    if (pc >= pages_at + 64) {              // uniform; spans move forward
      pages_at = pc;
      pages = bt[min(pc + lane, last_page)];
    }
    const int page = __builtin_amdgcn_readlane(pages, pc - pages_at);
    return ((int64_t)page * a.KH + kvh) * BS;
  };
  hbf16x8 kf[2][KK];
  u8x16_t k8[FP8 ? 2 : 1][FP8 ? KK / 2 : 1];
  auto load_k = [&](const int64_t r0, const int64_t r1) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // uniform page address, 32-bit lane offset
      const int64_t at = (i ? r1 : r0) * D;
      const uint32_t off = lo * D + d0;
      if constexpr (FP8) {
#pragma unroll
        for (int kk = 0; kk < KK; kk += 2) {
          const uint8_t* k = (const uint8_t*)a.k + at + (off + step_dim(kk));
          if constexpr (QUADS) {
            k8[i][kk / 2] = *reinterpret_cast<const u8x16_t*>(k);
          } else {
            const u8x8_t x = *reinterpret_cast<const u8x8_t*>(k);
            const u8x8_t y = *reinterpret_cast<const u8x8_t*>(k + step_dim(1));
            k8[i][kk / 2] = __builtin_shufflevector(
                x, y, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
          }
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < KK; kk++)
          kf[i][kk] = *reinterpret_cast<const hbf16x8*>(
              (const short*)a.k + at + (off + step_dim(kk)));
      }
    }
  };
  // fp8: V of the tile at r0 and r1, a tile ahead; 16 bytes are two chunks of a row
  u8x16_t v8[FP8 ? LV / 2 : 1];
  auto load_v8 = [&](const int64_t r0, const int64_t r1) {
#pragma unroll
    for (int j = 0; j < LV / 2; j++) {
      const int s = (j * 64 + lane) * 2;
      const int64_t at = (j * 128 / CV < BS ? r0 : r1) * D;
      v8[j] = *reinterpret_cast<const u8x16_t*>(
          (const uint8_t*)a.v + at + (uint32_t)(s / CV % BS * D + s % CV * 8));
    }
  };

  // `wild`: an infinity among the values is multiplied by the leading term of its
  // weight alone; with a remainder of the other sign, or of 0, it would be NaN.
  auto walk = [&](const bool wild) {
    int64_t row0 = 0, row1 = 0;
    if (t0 < t1) {
      row0 = page_row(base / BS + t0 * 2);
      row1 = page_row(base / BS + t0 * 2 + 1);
      load_k(row0, row1);
      if constexpr (FP8) load_v8(row0, row1);
    }
    for (int t = t0; t < t1; t++) {
      // ---- V of this tile: slot j * 64 + lane is row s / CV, place s % CV
      if constexpr (!FP8) {
#pragma unroll
        for (int j = 0; j < LV; j++) {
          const int row = j * (64 / CV) + lane / CV;
          const int64_t at = (j * (64 / CV) < BS ? row0 : row1) * D;
          const uint32_t off =
              row % BS * D + place_v<D>(row, lane % CV) * 8;
          flash::lds_copy16((const short*)a.v + at + off, vl + j * 512);
        }
      }
      // ---- S^T: keys 16 i + 4 hi + r of head lo
      f32x4 s[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < KK; kk++) {
          if constexpr (FP8) kf[i][kk] = widen8(k8[i][kk / 2], kk & 1);
          s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i][kk], qf[kk],
                                                         s[i], 0, 0, 0);
        }
      }
      if (t + 1 < t1) {               // K of the next tile, under way with V
        row0 = page_row(base / BS + t * 2 + 2);
        row1 = page_row(base / BS + t * 2 + 3);
        load_k(row0, row1);
      }
      // ---- softmax
      const int key0 = base + t * KT;
      const bool whole = key0 >= start && key0 + KT <= seq_len;
      float mx = NONE;
      if constexpr (BIASED) {
#pragma unroll
        for (int i = 0; i < 2; i++) s[i] *= a.scale;
        if (a.cap > 0.f)
#pragma unroll
          for (int i = 0; i < 8; i++)
            s[i / 4][i % 4] = a.cap * tanhf(s[i / 4][i % 4] / a.cap);
        if (a.r1) {
          float* pen = s_pen[wave];
          const float dist = (float)(seq_len - 1 - key0 - (lane & 31));
#pragma unroll
          for (int j = 0; j < PH / 2; j++)
            if (2 * j < a.G) pen[lane + 64 * j] = r1[j] * log1pf(r2[j] * dist);
          __builtin_amdgcn_wave_barrier();
          const float* mine = pen + min(lo, a.G - 1) * KT + 4 * hi;
#pragma unroll
          for (int i = 0; i < 2; i++)
            s[i] -= *reinterpret_cast<const f32x4*>(mine + 16 * i);
          __builtin_amdgcn_wave_barrier();
        }
      }
      auto seen = [&](const int i, const int r) {
        const int key = key0 + 16 * i + 4 * hi + r;
        return whole || (key >= start && key < seq_len);
      };
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          if (!BIASED) s[i][r] *= c;
          if (!seen(i, r)) s[i][r] = NONE;
          mx = fmaxf(mx, s[i][r]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      if (__any(mx > m)) {
        const float mn = fmaxf(m, mx);
        const float corr = BIASED && m == mn ? 1.f : fold_weight<BIASED>(m, mn);
        m = mn;
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] *= corr;
      }
      hbf16x8 p[3];                   // the weight's leading bits, the rest
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          // a masked key weighs nothing even where a lane saw no other yet; so
          // does one whose score is -infinity
          const bool live = BIASED ? s[i][r] != NONE : s[i][r] > -1e29f;
          float w = live ? fold_weight<BIASED>(s[i][r], m) : 0.f;
          l += w;
#pragma unroll
          for (int n = 0; n < 3; n++) {
            p[n][i * 4 + r] = (__bf16)w;
            w -= (float)p[n][i * 4 + r];
          }
        }
      if constexpr (FP8) {
#pragma unroll
        for (int j = 0; j < LV / 2; j++) {
          const int s0 = (j * 64 + lane) * 2, row = s0 / CV;
#pragma unroll
          for (int h = 0; h < 2; h++)
            *reinterpret_cast<hbf16x8*>(
                vl + row * D + place_v<D>(row, s0 % CV + h) * 8) =
                widen8(v8[j], h);
        }
        if (t + 1 < t1) load_v8(row0, row1);
      } else {
        // the direct loads' data: this wave's own, so no barrier
        __builtin_amdgcn_s_waitcnt(0x0f70);     // vmcnt(0)
      }
      if (!whole) {
        // slots outside the sequence hold what their last user left, and a
        // weight of zero does not silence an infinity
#pragma unroll
        for (int j = 0; j < LV; j++) {
          const int key = key0 + j * (64 / CV) + lane / CV;
          if (key < start || key >= seq_len)
            *reinterpret_cast<short8_t*>(vl + (j * 64 + lane) * 8) =
                short8_t{0, 0, 0, 0, 0, 0, 0, 0};
        }
      }
      __builtin_amdgcn_wave_barrier();
      // ---- O^T: dims 16 dt + 4 hi + r of head lo
#pragma unroll
      for (int dt = 0; dt < DT; dt += 2) {    // in pairs: neither waits for itself
        hbf16x8 vf[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const short* at = vl + vrow * D +
              place_v<D>(vrow, (dt + u) * 2 + vc) * 8 + ve;
          const short4_t a4 = flash::read_tr(at);
          const short4_t b4 = flash::read_tr(at + 16 * D);
          vf[u] = __builtin_bit_cast(
              hbf16x8, __builtin_shufflevector(a4, b4, 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int n = 2; n >= 0; n--)
#pragma unroll
          for (int u = 0; u < 2; u++) {
            hbf16x8 v = vf[u];
            if (BIASED && wild && n > 0) {
#pragma unroll
              for (int e = 0; e < 8; e++)
                if (!(fabsf((float)v[e]) < INFINITY)) v[e] = (__bf16)0.f;
            }
            o[dt + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                v, p[n], o[dt + u], 0, 0, 0);
          }
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  walk(false);
  if constexpr (BIASED) {
    bool nan = false;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 4; r++) nan |= o[dt][r] != o[dt][r];
    if (__any(nan)) {
      m = NONE;
      l = 0.f;
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
      pages_at = -64;
      walk(true);
    }
  }

  // ---- fold the waves: O of the used heads through LDS (the V stage)
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float* acc = reinterpret_cast<float*>(&lds_v[0][0]) + wave * a.G * D;
  __syncthreads();
  if (lo < a.G) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
      *reinterpret_cast<f32x4*>(acc + lo * D + dt * 16 + hi * 4) = o[dt];
    if (hi == 0) { s_m[wave][lo] = m; s_l[wave][lo] = l; }
  }
  __syncthreads();
  acc = reinterpret_cast<float*>(&lds_v[0][0]);
  for (int idx = threadIdx.x; idx < a.G * D; idx += NW * 64) {
    const int g = idx / D, d = idx % D, head = kvh * a.G + g;
    float gm = NONE;
#pragma unroll
    for (int w = 0; w < NW; w++) gm = fmaxf(gm, s_m[w][g]);
    const float sink = a.sinks && !partial
        ? a.sinks[head] * (BIASED ? 1.f : LOG2E) : NONE;
    gm = fmaxf(gm, sink);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float e = fold_weight<BIASED>(s_m[w][g], gm);
      num += e * acc[(w * a.G + g) * D + d];
      den += e * s_l[w][g];
    }
    if (partial) {
      const int64_t T = gridDim.x / a.KH;
      float* row = a.part + ((split * T + seq) * QH + head) * (D + 2);
      row[d] = num;
      if (d == 0) { row[D] = gm; row[D + 1] = den; }
    } else {
      if (a.sinks) den += fold_weight<BIASED>(sink, gm);
      store_head<BIASED>(a, seq, QH, head, D, d, num, den);
    }
  }
}

// One workgroup per (sequence, head) folds the splits that had keys, unless
// the first had them all. A chain of loads, so a short one: lane s of every
// wave has split s's weight.
template <int D, bool BIASED>
__global__ __launch_bounds__(D)
void paged_fold_kernel(const DecodeArgs a, const int QH, const int splits) {
  const int64_t row = blockIdx.x, rows = gridDim.x;
  if (BIASED && a.token_seq[row / QH] < 0) return;
  const int used =
      spans_of(a.len<BIASED>(row / QH), a.window, splits, WIDE).used;
  if (used == 1) return;
  constexpr float NONE = BIASED ? -INFINITY : -1e30f;
  const int d = threadIdx.x, lane = d & 63;
  const float sink =
      a.sinks ? a.sinks[row % QH] * (BIASED ? 1.f : LOG2E) : NONE;
  float m = NONE, l = 0.f;
  if (lane < used) {
    const float* p = a.part + (lane * rows + row) * (D + 2) + D;
    m = p[0];
    l = p[1];
  }
  const float gm = fmaxf(wave_reduce_max(m), sink);
  const float e = lane < used ? fold_weight<BIASED>(m, gm) : 0.f;
  float den = wave_reduce_sum(e * l);
  if (a.sinks) den += fold_weight<BIASED>(sink, gm);
  float num = 0.f;
#pragma unroll 4
  for (int s = 0; s < used; s++)
    num += __builtin_bit_cast(float, __builtin_amdgcn_readlane(
               __builtin_bit_cast(int, e), s)) *
        a.part[(s * rows + row) * (D + 2) + d];
  store_head<BIASED>(a, row / QH, QH, (int)(row % QH), D, d, num, den);
}

template <int D, bool FP8, bool BIASED, bool ROPE = false>
void launch_paged_decode(DecodeArgs a, const at::Tensor& out, int T) {
  auto stream = at::hip::getCurrentHIPStream();
  const int64_t pairs = (int64_t)T * a.KH;
  // Waves per workgroup and workgroups per pair, by the number of pairs and the
  // longest context that the table can hold (the lengths are on the device).
  // Times in us, bf16 / fp8 pages, 4 heads per pair of 128 unless stated.
  //   Splits up to 128 pairs, two or more workgroups each until 256, as long as
  // every wave keeps two tiles: 1 row of 16000 keys 24.5 / 21.8, 142 / 140 in one
  // workgroup per pair, 16 of 4000 43.6 / 28.3 and 44.3 / 40.7; 24 rows, which
  // would get one and a third, 84 / 49 and 69 / 41. 16 waves in each: 4 of 4000
  // 20.5 / 21.9, with 8 18.2 / 15.5. Short contexts under a wide table pay
  // for the fold's launch: 1 row of 40 keys 6.6, 5.0 under a table of 64 (6.0 in
  // one workgroup of 4 waves before; with one head per pair 6.1, 4.6 and 4.0).
  //   8 waves while a workgroup has a CU to itself: 32 of 1000 23 / 16, with 16
  // 24 / 19. Then 4: 64 of 200 12 / 9, with 8 15 / 13; heads of 64 are small
  // enough for two of 8 (48 of 4000: 71 / 38, with 4 83 / 45).
  //   2 waves where one round of the chip then takes the pairs that would need
  // two rounds of 4 (ROUND2 workgroups fit: 128 of 64 keys 7.6 / 7.2, with 4 9.8
  // / 8.6; of 2000 176 / 94, 186 / 108), and from 4096 pairs on, whose many rounds
  // cost by the wave (1024 of 64 keys 44 / 31, with 4 55 / 47; heads of 256 44 / 33,
  // 51 / 45, with 8 twice that), except bf16 pages of grouped heads, where the
  // contexts to be expected there want 4 (1024 of 300 keys 232 / 130, 223 / 143;
  // 2048 of 400 594 / 318, 573 / 344) unless windows keep them to a few tiles (2048
  // of 220 in a window of 128, heads of 64: 124, 141).
  int64_t longest = (int64_t)a.max_blocks * BS;
  if (a.window > 0) longest = std::min<int64_t>(longest, a.window + BS);
#define PA_LAUNCH(NW_, SPLIT_, GRID_)                                         \
  hipLaunchKernelGGL((paged_decode_kernel<D, FP8, NW_, SPLIT_, BIASED, ROPE>), GRID_, \
                     dim3(NW_ * 64), 0, stream, a)
  const int64_t splits = std::min<int64_t>(
      {SPLIT_FILL / pairs, longest / (WIDE * KT * SPLIT_MIN), 64});
  constexpr int64_t ROUND2 = D <= 64 ? 2048 : D <= 128 ? 1536 : 1024;
  if (splits > 1) {
    at::Tensor part = at::empty({splits, T, a.KH * a.G, D + 2},
                                out.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
    PA_LAUNCH(WIDE, true, dim3(pairs, splits));
    hipLaunchKernelGGL((paged_fold_kernel<D, BIASED>), dim3(T * a.KH * a.G),
                       dim3(D), 0, stream, a, a.KH * a.G, (int)splits);
  } else if (pairs <= (D <= 64 ? 512 : 256)) {
    PA_LAUNCH(WIDE, false, dim3(pairs));
  } else if ((pairs > ROUND2 / 2 && pairs <= ROUND2) ||
             (pairs >= 4096 &&
              (FP8 || D > 128 || a.G == 1 || longest <= 5 * KT))) {
    PA_LAUNCH(2, false, dim3(pairs));
  } else {
    PA_LAUNCH(4, false, dim3(pairs));
  }
#undef PA_LAUNCH
}

}  // namespace

}  // namespace kaito
