// Causal attention of prompt rows for gfx950 (bf16, f32 softmax): the one
// MFMA kernel behind prefill_attention (K/V rows of the step's own tokens),
// context_attention and window_attention_tiles (paged cache).
//
// A workgroup is 4 waves x 32 query rows of one key/value head. The rows of
// the heads that share it are flattened (row = position << gs | head), so
// that a group of 4 heads takes 32 positions per workgroup: every K/V tile
// is staged once for the whole group and little of the causal diagonal is
// computed for nothing. Groups that are no power of two run head by head.
// Prompts of up to 32 rows take one wave per head and half as many keys.
//
// Products are transposed, S^T = K Q^T and O^T = V^T P^T on
// v_mfma_f32_32x32x16_bf16:
//   - a lane holds ONE query row (column lane & 31) and half its keys, so
//     the row maximum is in-lane work and one exchange with lane ^ 32, and
//     the running maximum, sum and rescale factor are plain per-lane
//     scalars;
//   - the accumulator layout of S^T is, per 16 keys, the operand layout
//     that P^T needs once the contraction's keys are numbered accordingly
//     (slot j of half h <-> key 16 s + 4 h + (j < 4 ? j : j + 4)): P goes
//     from registers to the second product with no trip through LDS;
//   - V^T fragments in that numbering are pairs of ds_read_b64_tr_b16 on
//     the untransposed V tile.
// K and V tiles go to LDS by 16-byte global_load_lds, one tile ahead of the
// one in use (two buffers, one barrier per tile). The swizzles are applied
// to the global side of the copy: 16-byte chunk c of K row r sits at
// c ^ (r & 15) (D = 128), so that the sixteen rows of a quarter of a ds_read_b128
// touch all banks; V rows move by 64 bytes for the transposing reads.
//
// What bounds it: per 64 keys a wave runs 32 MFMA (1024 cycles at D = 128)
// beside about 900 cycles of softmax VALU work and a 32 KB LDS read, so two
// waves per SIMD that are out of step are the aim; register and LDS budgets
// (KVT) are set for that. Measured on one MI355X against the 16x16x32 kernels
// with V transposed by 2-byte LDS writes and P through LDS (before -> now):
//   whole prompts 4 x 2048, 16/4 heads of 128, window 1024: 447 -> 89 us;
//   one prompt of 8192, 32/8 heads of 128: 140 -> 762 TFLOP/s;
//   latent prompts 4 x 2048, 16 heads: 2307 us (padded to 256) -> 113 us;
//   8192 suffix rows over 20000 paged keys: 140 -> 825 TFLOP/s (997 over 16384
//   with the pages' addresses as scalars);
//   paged window 1024 with cap and penalty, 4 x 2048, 16/4 heads: 583 -> 176
//   (with the bare hardware reciprocal in cap and sigmoid 161).
#pragma once
#include "common.h"
#include <type_traits>

namespace kaito {
namespace flash {

typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 hbf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int TILE = 64;            // granularity of the caller's tile list
constexpr float LOG2E = 1.4426950408889634f;

enum Src { ROWS_BF16, PAGED_BF16, PAGED_FP8 };

// what a launch needs; the fields behind `window` serve the EXT variants
struct Args {
  short* out;                       // [T, QH, DV]
  const short* q;                   // row stride q_ts, head stride q_hs
  const short* q2;                  // dims behind D1 (split heads)
  const void* k;
  const short* k2;                  // dims behind D1, shared by the heads
  const void* v;
  int64_t q_ts, q_hs, q2_ts, q2_hs, k_ts, k_hs, k2_ts, v_ts, v_hs;
  const int* tile_seq;              // 64-row tiles of the step's chunks
  const int* tile_qbase;
  const int* cu;                    // [B + 1] chunk row offsets
  const int* kv_lens;               // [B] keys after the step, or nullptr
  const int* starts;                // [B] position of a chunk's first row
  const int* block_tables;
  int max_blocks, BS, KH, QH;
  int gs;                           // log2 of the heads flattened together
  float scale;
  int window;                       // 0 = all earlier keys
  const float* sinks;               // [QH] or nullptr
  int keep_first, chunk;
  float softcap;
  const float *r1, *r2;             // distance penalty per head
  const float* pb;                  // sigmoid weights: bias per head
  const short* gate;
  int64_t gate_s0;
  const float* db;                  // distance bias table [QH, db_n]
  int db_n;
  float temp_coef;
  int temp_every;
};

// LDS serves 256 bytes per cycle, 16 lanes of a 16-byte read, 32 of an 8-byte
// one: as many rows have to lie in different sixteenths (eighths) of 256 bytes.
// Places that do so for 8 rows only take twice as long (1 KB reads by four waves
// at once: 32 and 16 cycles each, 512 transposed bytes 16 and 10.5). One prompt of
// 8192, 32/8 heads of 128: 593 -> 584 us; 4 x 2048, 16/4 heads, window 1024: 91 ->
// 87; with pages 1157 -> 1139 (3627 rows over 20011 keys).
// chunk of a K row -> its place
template <int D>
KAITO_DEV int swz_k(int row, int c) {
  if constexpr (D == 96) return c ^ ((row >> 2) & 3);
  else if constexpr (D % 128 == 0) return c ^ (row & 15);
  else return c ^ ((row >> 1) & 7);
}

// chunk of a V row -> its place; pairs of chunks (16 columns) stay together, and
// four where a row is 256 bytes or more: 4 rows of them are read at once
template <int DV>
KAITO_DEV int swz_v(int row, int c) {
  if constexpr (DV == 32 || DV == 96) return c ^ (((row >> 1) & 1) << 1);
  else if constexpr (DV == 64) return c ^ ((row & 3) << 1);
  else return c ^ ((row & 3) << 2);
}

KAITO_DEV void lds_copy16(const short* src, short* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) unsigned int*)src,
      (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 0);
}

KAITO_DEV f32x16 mfma32(hbf16x8 a, hbf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 1 / d for d >= 1, to a division's precision: one Newton step on the
// hardware's reciprocal, which gives 0 by itself where the step would not end
KAITO_DEV float recip(const float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return d > 0x1p125f ? r : fmaf(fmaf(-d, r, 1.0f), r, r);
}

// 4 rows x 16 columns per 16 lanes -> lane i: column i of the 4 rows
KAITO_DEV short4_t read_tr(const short* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4_t*)p);
}

// keys per tile: two buffers of K and V of two workgroups fit the 160 KB
template <int D, int DV>
constexpr int kvt() { return D + DV <= 320 ? 64 : 32; }

// D1: dims of q and k that come from q/k; the others come from q2/k2. KVT: keys
// per tile; NW: waves of 32 rows.
// EXT: capping, penalty, kept first keys, chunked mask, head gate, and
// softmax weights that enter P.V as a bf16 value + remainder pair.
template <int D, int DV, int SRC, bool EXT, bool SIG = false, bool DB = false,
          int D1 = D, int KVT = kvt<D, DV>(), int NW = 4>
__global__ __launch_bounds__(NW * 64, (D + DV > 384 ? 1 : 2))
void flash_prefill_kernel(const Args a) {
  constexpr int NK = KVT / 32, KK = D / 16, NS = KVT / 16, DT = DV / 32;
  constexpr int CK = D / 8, CV = DV / 8;          // 16-byte chunks of a row
  constexpr int NT = NW * 64, ROWS = NW * 32;     // threads, query rows
  constexpr int LK = KVT * CK / NT, LV = KVT * CV / NT;
  // with nothing but a positive factor between product and exponent, it
  // rides in the exponent's multiply-add
  const bool fold = !EXT && !SIG && !DB && a.scale > 0.f;
  static_assert(KVT * CK % NT == 0 && KVT * CV % NT == 0 && DV % 32 == 0);
  static_assert(SRC != PAGED_FP8 || !EXT);

  const int HG = a.QH >> a.gs;                    // head groups
  const int hg = blockIdx.x % HG;
  const int rest = blockIdx.x / HG;
  const int QP = ROWS >> a.gs;                    // positions per workgroup
  const int sub = QP < TILE ? TILE / QP : 1;
  const int tile = rest / sub;
  const int seq = a.tile_seq[tile];
  const int q0 = a.tile_qbase[tile] + (rest % sub) * QP;
  const int tok0 = a.cu[seq];
  const int q_len = a.cu[seq + 1] - tok0;
  // 128-position workgroups serve two tiles: the even one stands for both
  if ((QP > TILE && (q0 & (QP - 1))) || q0 >= q_len) return;
  const int h0 = hg << a.gs;
  const int kvh = h0 / (a.QH / a.KH);
  const int q_abs0 = a.starts ? a.starts[seq]
      : (a.kv_lens ? a.kv_lens[seq] - q_len : 0);
  const int kv_len = q_abs0 + q_len;
  const int* bt = SRC == ROWS_BF16 ? nullptr
      : a.block_tables + (int64_t)seq * a.max_blocks;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, h = lane >> 5;

  __shared__ __attribute__((aligned(128))) short lds[2][KVT * (D + DV)];
  __shared__ float lds_db[2][DB ? ROWS + KVT : 1];

  // ---- this lane's query row
  const int R = wave * 32 + lr;
  const int qrow = q0 + (R >> a.gs);
  const int head = h0 + (R & ((1 << a.gs) - 1));
  const int q_abs = q_abs0 + qrow;
  const int64_t qtok = tok0 + min(qrow, q_len - 1);
  hbf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) {
    const int d = kk * 16 + h * 8;
    const short* p = d < D1 ? a.q + qtok * a.q_ts + head * a.q_hs + d
                            : a.q2 + qtok * a.q2_ts + head * a.q2_hs + d - D1;
    qf[kk] = *reinterpret_cast<const hbf16x8*>(p);
  }
  // positions of the wave's first and last row
  const int w_first = q_abs0 + q0 + ((wave * 32) >> a.gs);
  const int w_last = q_abs0 + q0 + ((wave * 32 + 31) >> a.gs);

  float qs = a.scale;                 // score = product * qs (* log2 e)
  if constexpr (DB)
    if (a.temp_coef != 0.f)
      qs *= 1.0f + a.temp_coef * logf((float)((q_abs + 1) / a.temp_every + 1));
  const float hr1 = EXT && a.r1 ? a.r1[head] : 0.f;
  const float hr2 = EXT && a.r1 ? a.r2[head] : 0.f;
  const float hpb = SIG ? a.pb[head] : 0.f;

  // running maximum (log2 domain) and this lane's share of the sum. It is
  // finite from the start (a sink may be -inf) and masked scores are -inf, at
  // any scale: a tile in which a row sees nothing neither moves the maximum
  // nor weighs anything.
  float m = a.sinks ? fmaxf(a.sinks[head] * LOG2E, -1e30f) : -1e30f;
  float l = (a.sinks || SIG) && h == 0 ? 1.0f : 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[dt][i] = 0.f;

  // ---- key tiles: those with kept first keys, then the visible range
  const int kv_end = min(kv_len, q_abs0 + q0 + QP);
  const int vis0 = EXT && a.chunk > 0 ? ((q_abs0 + q0) / a.chunk) * a.chunk
      : (a.window > 0 ? q_abs0 + q0 - a.window + 1 : 0);
  const int kv_begin = vis0 > 0 ? vis0 / KVT * KVT : 0;
  const int first_end =
      EXT ? min((a.keep_first + KVT - 1) / KVT * KVT, kv_begin) : 0;
  const int kv_first = first_end > 0 ? 0 : kv_begin;
  auto next_tile = [&](const int kv0) {
    return EXT && kv0 + KVT == first_end ? kv_begin : kv0 + KVT;
  };

  // ---- staging. Slot s of a tile (16 bytes of LDS) is row s / C, place
  // s % C; thread tid fills slots j * NT + tid.
  // Pages of 16 keys: a wave's instruction reads rows of one page, so that page
  // numbers and addresses are scalars and a lane's offset does not change. With a
  // page, a quotient and a 64-bit address per lane and copy, the vector unit
  // had more to do than the matrix cores (before -> now): 8192 suffix rows over
  // 8192 keys, 32/8 heads of 128, 883 -> 999 TFLOP/s; 3627 over 16384 810 ->
  // 932; fp8 cache, 4096 over 4096, 757 -> 893; heads of 64 and 256, 2048 over
  // 2048, 78 -> 65 and 297 -> 244 us; window 1024 with key size 128, value
  // size 256, 118 -> 107 us. The same for rows of the step gave 3 % at 8192 and
  // took 2 % at 4 x 2048.
  static_assert(SRC == ROWS_BF16 || (64 % CK == 0 && 64 % CV == 0));
  constexpr bool PAGED = SRC != ROWS_BF16;
  // The distance bias at 128 x 128 has no registers left for it: 13 spilled, 4 x
  // 2048, 16/4 heads, window 1024: 128.7 -> 139.8 us.
  constexpr bool SCALAR_PAGES = PAGED && !(DB && D == 128 && DV == 128);
  const bool by16 = SCALAR_PAGES && (!EXT || a.BS == 16);
  int pages_k = 0, pages_v = 0;     // lane j: page of this wave's j-th copy
  int pk[PAGED && EXT ? LK : 1], pv[PAGED && EXT ? LV : 1];
  auto fetch_pages = [&](const int kv0) {       // pages of the tile at kv0
    if constexpr (PAGED) {
      if (by16) {
        auto number = [&](const int chunks, const int copies) {
          const int key = kv0 + min(lane, copies - 1) * (NT / chunks) +
              wave * (64 / chunks);
          return bt[min(key, kv_len - 1) >> 4];
        };
        pages_k = number(CK, LK);
        if constexpr (CV != CK) pages_v = number(CV, LV);
      } else if constexpr (EXT) {
#pragma unroll
        for (int j = 0; j < LK; j++)
          pk[j] = bt[min(kv0 + (j * NT + tid) / CK, kv_len - 1) / a.BS];
        if constexpr (CV != CK) {
#pragma unroll
          for (int j = 0; j < LV; j++)
            pv[j] = bt[min(kv0 + (j * NT + tid) / CV, kv_len - 1) / a.BS];
        }
      }
    }
  };
  u8x8_t rk[SRC == PAGED_FP8 ? LK : 1], rv[SRC == PAGED_FP8 ? LV : 1];
  auto stage_pages = [&](const int kv0, short* buf, auto whole) {
    auto at = [&](const int pages, const int j, const int chunks) {
      const int64_t page = __builtin_amdgcn_readlane(pages, j);
      return (page * a.KH + kvh) * 16 * (chunks * 8);
    };
    // row of its page; behind the last key that one again
    auto place = [&](const int j, const int chunks) {
      const int row = tid / chunks, step = j * (NT / chunks);
      if (decltype(whole)::value) return (row & 15) + (step & 15);
      return min(kv0 + step + row, kv_len - 1) & 15;
    };
#pragma unroll
    for (int j = 0; j < LK; j++) {
      const int s = j * NT + tid;
      const int off = place(j, CK) * D + swz_k<D>(s / CK, s % CK) * 8;
      if constexpr (SRC == PAGED_FP8)
        rk[j] = *reinterpret_cast<const u8x8_t*>(
            (const uint8_t*)a.k + at(pages_k, j, CK) + (uint32_t)off);
      else
        lds_copy16((const short*)a.k + at(pages_k, j, CK) + (uint32_t)off,
                   buf + (j * NT + wave * 64) * 8);
    }
#pragma unroll
    for (int j = 0; j < LV; j++) {
      const int s = j * NT + tid;
      const int off = place(j, CV) * DV + swz_v<DV>(s / CV, s % CV) * 8;
      const int64_t page = at(CV == CK ? pages_k : pages_v, j, CV);
      if constexpr (SRC == PAGED_FP8)
        rv[j] = *reinterpret_cast<const u8x8_t*>((const uint8_t*)a.v + page +
                                                 (uint32_t)off);
      else
        lds_copy16((const short*)a.v + page + (uint32_t)off,
                   buf + KVT * D + (j * NT + wave * 64) * 8);
    }
  };
  // Split keys: a lane's copies of a tile come from either part, those PERIOD
  // apart from the same dims; their places move on by one tile at a time. One
  // prompt of 8192, 16 heads, 601 -> 562 us; 4 x 2048 132 -> 125; 128 heads, 16 x
  // 128, 79 -> 73 to 78.
  constexpr bool SPLIT_K = !PAGED && D1 < D;
  constexpr int PERIOD = SPLIT_K ? 3 : 1, AHEAD = PERIOD * NT / CK;
  static_assert(!SPLIT_K || (LK % PERIOD == 0 && PERIOD * NT % CK == 0 &&
                             AHEAD % 16 == 0 && KVT == LK / PERIOD * AHEAD));
  const short* k_lane[PERIOD];
  const short* v_lane = nullptr;
  if constexpr (SPLIT_K) {
    const int64_t tok = tok0 + kv_first;
#pragma unroll
    for (int j = 0; j < PERIOD; j++) {
      const int s = j * NT + tid, row = s / CK;
      const int col = swz_k<D>(row, s % CK) * 8;
      k_lane[j] = col < D1
          ? (const short*)a.k + (tok + row) * a.k_ts + kvh * a.k_hs + col
          : a.k2 + (tok + row) * a.k2_ts + col - D1;
    }
    v_lane = (const short*)a.v + (tok + tid / CV) * a.v_ts + kvh * a.v_hs +
        swz_v<DV>(tid / CV, tid % CV) * 8;
    static_assert(NT / CV % 4 == 0);
  }
  auto stage = [&](const int kv0, short* buf) {
    if constexpr (PAGED) {
      if (by16) {
        if (kv0 + KVT <= kv_len) stage_pages(kv0, buf, std::true_type{});
        else stage_pages(kv0, buf, std::false_type{});
        return;
      }
      if constexpr (!EXT) return;
    }
    if constexpr (SPLIT_K) {
      if (kv0 + KVT <= kv_len) {    // no row to stand for another
#pragma unroll
        for (int j = 0; j < LK; j++) {
          const short*& p = k_lane[j % PERIOD];
          lds_copy16(p, buf + (j * NT + wave * 64) * 8);
          const int s = j % PERIOD * NT + tid;
          const bool first = swz_k<D>(s / CK, s % CK) * 8 < D1;
          p += AHEAD * (first ? a.k_ts : a.k2_ts);
        }
#pragma unroll
        for (int j = 0; j < LV; j++)
          lds_copy16(v_lane + j * (NT / CV) * a.v_ts,
                     buf + KVT * D + (j * NT + wave * 64) * 8);
        v_lane += KVT * a.v_ts;
        return;
      }
    }
#pragma unroll
    for (int j = 0; j < LK; j++) {
      const int s = j * NT + tid, row = s / CK;
      const int col = swz_k<D>(row, s % CK) * 8;
      const int key = min(kv0 + row, kv_len - 1);
      if constexpr (SRC == ROWS_BF16) {
        const int64_t tok = tok0 + key;
        const short* p = col < D1
            ? (const short*)a.k + tok * a.k_ts + kvh * a.k_hs + col
            : a.k2 + tok * a.k2_ts + col - D1;
        lds_copy16(p, buf + (j * NT + wave * 64) * 8);
      } else if constexpr (EXT) {
        lds_copy16((const short*)a.k +
                       (((int64_t)pk[j] * a.KH + kvh) * a.BS + key % a.BS) * D +
                       col,
                   buf + (j * NT + wave * 64) * 8);
      }
    }
    short* vbuf = buf + KVT * D;
#pragma unroll
    for (int j = 0; j < LV; j++) {
      const int s = j * NT + tid, row = s / CV;
      const int col = swz_v<DV>(row, s % CV) * 8;
      const int key = min(kv0 + row, kv_len - 1);
      if constexpr (SRC == ROWS_BF16) {
        lds_copy16((const short*)a.v + (int64_t)(tok0 + key) * a.v_ts +
                       kvh * a.v_hs + col,
                   vbuf + (j * NT + wave * 64) * 8);
      } else if constexpr (EXT) {
        const int64_t page = CV == CK ? pk[j] : pv[j];
        lds_copy16((const short*)a.v +
                       ((page * a.KH + kvh) * a.BS + key % a.BS) * DV + col,
                   vbuf + (j * NT + wave * 64) * 8);
      }
    }
  };
  // fp8 caches are widened on the way: registers -> LDS behind the compute
  auto widen = [&](short* buf) {
    if constexpr (SRC == PAGED_FP8) {
      auto put = [&](const u8x8_t raw, short* dst) {
        float f[8];
        fp8x8_to_f32(raw, f);
        hbf16x8 w;
#pragma unroll
        for (int e = 0; e < 8; e++) w[e] = (__bf16)f[e];
        *reinterpret_cast<hbf16x8*>(dst) = w;
      };
#pragma unroll
      for (int j = 0; j < LK; j++) put(rk[j], buf + (j * NT + tid) * 8);
#pragma unroll
      for (int j = 0; j < LV; j++)
        put(rv[j], buf + KVT * D + (j * NT + tid) * 8);
    }
  };
  // the tile's bias by (position of the row) - key + KVT - 1
  auto stage_bias = [&](const int kv0, float* dst) {
    if constexpr (DB) {
      if (tid < ROWS + KVT - 1) {
        const int dist = q_abs0 + q0 - kv0 + tid - (KVT - 1);
        dst[tid] = a.db[(int64_t)h0 * a.db_n + min(max(dist, 0), a.db_n - 1)];
      }
    }
  };

  fetch_pages(kv_first);
  stage(kv_first, lds[0]);
  stage_bias(kv_first, lds_db[0]);
  fetch_pages(next_tile(kv_first));
  widen(lds[0]);
  __syncthreads();

  // lane-constant parts of the V^T fragment addresses
  const int li = lane & 15;
  const int vrow = 4 * h + (li >> 2);
  const int vc = ((lane >> 4) & 1) * 2 + ((li & 3) >> 1);
  const int ve = (li & 1) * 4;

  int cur = 0;
  for (int kv0 = kv_first; kv0 < kv_end;) {
    const int kvn = next_tile(kv0);
    if (kvn < kv_end) {
      stage(kvn, lds[cur ^ 1]);
      stage_bias(kvn, lds_db[cur ^ 1]);
      fetch_pages(next_tile(kvn));
    }
    const short* kb = lds[cur];
    const short* vb = kb + KVT * D;

    // ---- S^T: key 32 kt + 8 (i / 4) + 4 h + i % 4 of this lane's row
    f32x16 s[NK];
#pragma unroll
    for (int kt = 0; kt < NK; kt++) {
#pragma unroll
      for (int i = 0; i < 16; i++) s[kt][i] = 0.f;
      const int row = kt * 32 + lr;
#pragma unroll
      for (int kk = 0; kk < KK; kk++)
        s[kt] = mfma32(*reinterpret_cast<const hbf16x8*>(
                           kb + row * D + swz_k<D>(row, kk * 2 + h) * 8),
                       qf[kk], s[kt]);
    }

    // ---- scores in the log2 domain (SIG: weights)
    const int dist0 = q_abs - kv0 - 4 * h;      // distance to key i = 0
    auto key_off = [](const int kt, const int i) {
      return kt * 32 + 8 * (i / 4) + i % 4;
    };
    if (EXT && a.softcap > 0.f) {
      const float c2 = a.softcap * LOG2E, g2 = qs * 2.0f * LOG2E / a.softcap;
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++)          // cap * tanh(s / cap), via exp
          s[kt][i] = c2 - 2.0f * c2 * recip(
              __builtin_amdgcn_exp2f(s[kt][i] * g2) + 1.0f);
    } else if (!fold) {
      const float c = qs * LOG2E;
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) s[kt][i] *= c;
    }
    if (EXT && a.r1) {
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          s[kt][i] -= hr1 * __builtin_amdgcn_logf(
              1.0f + hr2 * (float)max(dist0 - key_off(kt, i), 0));
    }
    if constexpr (DB) {
      const float* b = lds_db[cur] + R - 4 * h + KVT - 1;
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++)
          s[kt][i] += b[-key_off(kt, i)] * LOG2E;
    }
    // tiles that every row of the wave sees whole need no mask
    const bool whole = kv0 + KVT - 1 <= w_first &&
        (a.window <= 0 || w_last - kv0 < a.window) &&
        (!EXT || a.chunk <= 0 || kv0 >= (w_last / a.chunk) * a.chunk);
    if (!whole) {
      const int low = EXT && a.chunk > 0 ? (q_abs / a.chunk) * a.chunk : 0;
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int dist = dist0 - key_off(kt, i);
          const int key = q_abs - dist;
          bool dead = dist < 0 || (a.window > 0 && dist >= a.window &&
                                   !(EXT && key < a.keep_first));
          if (EXT) dead = dead || key < low;
          if (dead) s[kt][i] = -INFINITY;
        }
    }
    if constexpr (SIG) {
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++)          // a masked score weighs zero
          s[kt][i] = recip(
              1.0f + __builtin_amdgcn_exp2f(-s[kt][i] - hpb * LOG2E));
    } else {
      float mx = s[0][0];
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[kt][i]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float c = fold ? a.scale * LOG2E : 1.0f;
      mx *= c;
      // most tiles move no row's maximum: the accumulators stay as they are
      if (__any(mx > m)) {
        const float mn = fmaxf(m, mx);
        const float corr = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
          for (int i = 0; i < 16; i++) o[dt][i] *= corr;
      }
#pragma unroll
      for (int kt = 0; kt < NK; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          s[kt][i] = __builtin_amdgcn_exp2f(fmaf(s[kt][i], c, -m));
          l += s[kt][i];
        }
    }

    // ---- O^T += V^T P^T, 16 keys at a time
#pragma unroll
    for (int st = 0; st < NS; st++) {
      hbf16x8 p, pl;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float f = s[st / 2][8 * (st & 1) + j];
        p[j] = (__bf16)f;
        if constexpr (EXT) pl[j] = (__bf16)(f - (float)p[j]);
      }
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const int row = st * 16 + vrow;
        const short* at = vb + row * DV + swz_v<DV>(row, dt * 4 + vc) * 8 + ve;
        const short4_t lo4 = read_tr(at), hi4 = read_tr(at + 8 * DV);
        const short8_t v8 = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4,
                                                    5, 6, 7);
        const hbf16x8 vf = __builtin_bit_cast(hbf16x8, v8);
        o[dt] = mfma32(vf, p, o[dt]);
        if constexpr (EXT) o[dt] = mfma32(vf, pl, o[dt]);
      }
    }
    if (kvn < kv_end) widen(lds[cur ^ 1]);
    __syncthreads();
    kv0 = kvn;
    cur ^= 1;
  }

  // ---- epilogue
  l = SIG ? 1.0f : l + __shfl_xor(l, 32, 64);
  if (qrow >= q_len) return;
  float inv = 1.0f / fmaxf(l, 1e-30f);
  if (EXT && a.gate) {
    const float g =
        bf16_to_f32(a.gate[(int64_t)(tok0 + qrow) * a.gate_s0 + head]);
    inv *= 1.0f / (1.0f + __expf(-g));
  }
  short* orow = a.out + ((int64_t)(tok0 + qrow) * a.QH + head) * DV + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int b = 0; b < 4; b++) {
      short4_t w;
#pragma unroll
      for (int e = 0; e < 4; e++)
        w[e] = f32_to_bf16(o[dt][b * 4 + e] * inv);
      *reinterpret_cast<short4_t*>(orow + dt * 32 + 8 * b) = w;
    }
}

// heads flattened into a workgroup's rows: a power-of-two group whole
inline int group_shift(int QH, int KH) {
  const int G = QH / KH;
  for (int s = 0; s <= 4; s++)
    if ((1 << s) == G) return s;
  return 0;
}

// workgroups of `waves` waves over `tiles` 64-row tiles
inline int64_t grid_size(const Args& a, int64_t tiles, int waves = 4) {
  const int QP = waves * 32 >> a.gs;
  return tiles * (QP < TILE ? TILE / QP : 1) * (a.QH >> a.gs);
}

}  // namespace flash
}  // namespace kaito
