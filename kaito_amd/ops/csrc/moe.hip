// MoE feed-forward of decode-sized steps for gfx950: few rows per expert, so
// both products stream the weights once (skinny.h stream_tile) and are bound
// by that. Everything is device-side and static-shaped, so that MoE decode
// steps capture into hipGraphs:
//
//   * tokens are sorted by expert on the GPU (moe_route.hip) and the kernels
//     get `sorted_ids` (token per sorted row) and `offsets` ([E+1] exclusive
//     prefix sums, by global expert); in small steps of few experts
//     (ops.moe_pairs_pay) a workgroup finds its expert's rows among the pairs
//     (moe_up_pairs, moe_down_pairs);
//   * moe_gate_silu: act[s] = silu(x[tok] Wg^T) * (x[tok] Wu^T), the rows
//     gathered through sorted_ids (ungated experts, act_mode 2: relu(.)^2). A
//     workgroup's 16 weight rows are 8 gate rows and their 8 up rows;
//   * moe_down_rows: y[s] = act[s] Wd^T in f32, summed per token by
//     moe_combine.
//
// One workgroup per (16 weight rows, expert), or with K = 2048 about one per CU
// that goes from tile to tile; an expert with more rows than 16 MT is walked in
// passes, whose weights come back from the caches. Measured on one MI355X (32
// tokens, 8 experts of 2048 x 2048, top 2) against 64 x 128 tiles with both
// operands staged behind barriers, on 128 workgroups: 89 us for both products, 47
// in tiles of their own, now 38.5 (201 MB of weights: 5.2 TB/s, launches
// included). 32 experts of 2880 x 2880 (K in stages of 64), top 4, whole layer: 8
// tokens 491 -> 178, 64 tokens 440 -> 297.
//
// Expert parallelism: callers pass `e_base` and the LOCAL weights; TP shards
// the expert intermediate dim. Both use these kernels unchanged.
#include "skinny.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <algorithm>
#include <cmath>

namespace kaito {

namespace {

struct StreamArgs {
  const short* x;                   // up: [T, K]; down: [TK, K]
  const short* w;                   // [E local, rows, K]
  const short* bias;                // [E local, rows] or nullptr
  const int* rows;                  // token of a sorted row
  const int* offsets;               // [global E + 1]
  // or, in place of both, rows in the order of the pairs themselves:
  const int* topi;                  // [pairs] expert of a pair
  int pairs, top;                   // top pairs per token
  int e_base, N, K;
  int act_mode;
  float limit;
  short* act;                       // up: [TK, N]
  float* y;                         // down: [TK, N]
  // an expert of every token behind the local ones, of the same sizes, or none
  // (PAIRS, without biases): its weights; up: act [T, N]; down: act [T, K], y in
  // bf16 [T, N]
  const short* all_w;
  short* all_act;
  short* all_y;
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

// The rows begin .. end - 1 of an expert: sorted ones, or the pairs that chose it,
// found by every wave for itself, 64 at a time, and listed in LDS. The sort's
// launch is 4.3 us of a decode step's layer; the scan takes the place of the
// loads of offsets and rows, one after the other. A kernel of its own: with both
// in one, sorted rows of 256 experts took 37.4 us a layer in place of 33.1 (one
// token, 2048 x 512, top 8).
constexpr int PAIRS_MAX = 256;

template <int PAIRS>
struct Rows {
  int begin, end;
  const unsigned short* list;       // of PAIRS

  // row of act and y
  KAITO_DEV int at(const int m) const { return PAIRS ? list[m] : m; }
};

// PAIRS: rows by sorted pairs (0), by the pairs themselves (1), so and with an
// expert of every token (2), which would cost the others 0.7 us of a launch.
// The arguments as local expert le sees them: the one of all lies behind the rest.
template <int KIND, int PAIRS>
KAITO_DEV StreamArgs as_expert(const StreamArgs& a, const int le) {
  StreamArgs b = a;
  const int64_t wrows = KIND == UP_GATED ? 2 * a.N : a.N;
  const bool all = PAIRS == 2 && le == (int)gridDim.y - 1;
  b.w = all ? a.all_w : a.w + le * wrows * a.K;
  if (b.bias) b.bias += le * wrows;
  if constexpr (PAIRS == 2) {
    if (KIND == DOWN) {
      b.x = all ? a.all_act : a.x;
      b.all_y = all ? a.all_y : nullptr;
    } else {
      b.act = all ? a.all_act : a.act;
    }
    b.pairs = all ? a.pairs / a.top : a.pairs;
    b.top = all ? 1 : a.top;
    b.topi = all ? nullptr : a.topi;
  }
  return b;
}

template <int PAIRS>
KAITO_DEV Rows<PAIRS> rows_of(const StreamArgs& a, const int expert,
                              unsigned short* list, const int lane) {
  if constexpr (!PAIRS)
    return {a.offsets[expert], a.offsets[expert + 1], nullptr};
  if (PAIRS == 2 && !a.topi) {      // every token
#pragma unroll
    for (int i = 0; i < PAIRS_MAX; i += 64) list[i + lane] = i + lane;
    __builtin_amdgcn_wave_barrier();
    return {0, a.pairs, list};
  }
  int n = 0, e[PAIRS_MAX / 64];
#pragma unroll
  for (int i = 0; i < PAIRS_MAX / 64; i++) {
    const int p = i * 64 + lane;
    e[i] = p < a.pairs ? a.topi[p] : -1;
  }
#pragma unroll
  for (int i = 0; i < PAIRS_MAX / 64; i++) {
    if (i * 64 >= a.pairs) break;
    const unsigned long long hit = __ballot(e[i] == expert);
    if (e[i] == expert)
      list[n + __builtin_popcountll(hit & ((1ull << lane) - 1))] =
          i * 64 + lane;
    n += __builtin_popcountll(hit);
  }
  __builtin_amdgcn_wave_barrier();
  return {0, n, list};
}

// column n of rows m .. m + 3 below the end: v, or gate v and up u
template <int KIND, int PAIRS>
KAITO_DEV void store_rows(const StreamArgs& a, const f32x4 v, const f32x4 u,
                          const int m0, const Rows<PAIRS>& rows,
                          const int n) {
#pragma unroll
  for (int r = 0; r < 4; r++) {
    if (m0 + r >= rows.end) break;
    const int m = rows.at(m0 + r);
    if constexpr (KIND == UP_GATED) {
      a.act[(int64_t)m * a.N + n] =
          f32_to_bf16(moe_act_f(a.act_mode, v[r], u[r], a.limit));
    } else if constexpr (KIND == UP_PLAIN) {
      const float p = fmaxf(v[r], 0.f);
      a.act[(int64_t)m * a.N + n] = f32_to_bf16(p * p);
    } else if (PAIRS == 2 && a.all_y) {
      a.all_y[(int64_t)m * a.N + n] = f32_to_bf16(v[r]);
    } else {
      a.y[(int64_t)m * a.N + n] = v[r];
    }
  }
}

// x of row m, the last one's past the end
template <int KIND, int PAIRS>
KAITO_DEV const short* x_row(const StreamArgs& a, const Rows<PAIRS>& rows,
                             const int m) {
  const int r = rows.at(min(m, rows.end - 1));
  const int64_t row = KIND == DOWN ? r : PAIRS ? r / a.top : a.rows[r];
  return a.x + row * a.K;
}

template <int MT, int KS, int KIND, int PAIRS>
__global__ __launch_bounds__(256, 2) void moe_stream_kernel(
    const StreamArgs args) {
  constexpr int NI = skinny::tile_loads<KS>();
  constexpr bool GATED = KIND == UP_GATED;
  __shared__ __attribute__((aligned(128))) short ring[4][2][16 * KS];
  static_assert(sizeof(ring) >= 4 * MT * 64 * sizeof(f32x4), "fold");
  __shared__ unsigned short list[PAIRS ? 4 : 1][PAIRS ? PAIRS_MAX : 1];
  const int le = blockIdx.y;
  const StreamArgs a = as_expert<KIND, PAIRS>(args, le);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const auto rows =
      rows_of<PAIRS>(a, a.e_base + le, list[PAIRS ? wave : 0], lane);
  const int begin = rows.begin, end = rows.end;
  if (begin >= end) return;
  const int n0 = blockIdx.x * (GATED ? 8 : 16);
  const short* src[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int r = skinny::tile_row<KS>(j, lane);
    const int64_t n = GATED ? n0 + r % 8 + (r >= 8 ? a.N : 0) : n0 + r;
    src[j] = a.w + n * a.K + skinny::tile_col<KS>(j, lane);
  }
  f32x4* red = reinterpret_cast<f32x4*>(&ring[0][0][0]);
  const int slot = threadIdx.x, l = slot & 63, c = l & 15;
  const bool mine = slot < MT * 64 && !(GATED && c >= 8);
  const short* be = a.bias ? a.bias + n0 + c : nullptr;
  for (int m0 = begin; m0 < end; m0 += 16 * MT) {
    const short* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      xp[mt] = x_row<KIND>(a, rows, m0 + mt * 16 + (lane & 15)) +
          (lane >> 4) * 8;
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
      store_rows<KIND>(a, v, u, m0 + (slot >> 6) * 16 + (l >> 4) * 4, rows,
                       n0 + c);
    }
    __syncthreads();                // sums read before the next pass's stages
  }
}

// K = 1024 S: see skinny::stream_tiles. gridDim.x workgroups share an expert's
// ntiles tiles; MT row tiles of 16 in a pass.
template <int MT, int S, int KIND, int PAIRS>
KAITO_DEV void stream_pass(const StreamArgs& a, const int ntiles,
                           const int m0, const Rows<PAIRS>& rows, short* ring,
                           f32x4* red, const int wave, const int lane) {
  constexpr int KS = skinny::TILES_KS, NW = skinny::TILE_NW;
  constexpr bool GATED = KIND == UP_GATED;
  constexpr int COLS = GATED ? 8 : 16;
  const int slot = threadIdx.x, l = slot & 63, c = l & 15;
  const bool mine = slot < MT * 64 && !(GATED && c >= 8);
  skinny::stream_tiles<MT, S, false>(
      a.w, nullptr, 0,
      [&](const int j) {
        const int r = skinny::tile_row<KS>(j, lane);
        const uint32_t n = GATED ? r % 8 + (r >= 8 ? a.N : 0) : r;
        return (n * a.K + skinny::tile_col<KS>(j, lane)) * 2;
      },
      COLS * a.K * 2, blockIdx.x, gridDim.x, ntiles,
      [&](const short* (&xp)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          xp[mt] = x_row<KIND>(a, rows, m0 + mt * 16 + (lane & 15)) +
              (lane >> 4) * 8;
      },
      ring, red, wave, lane,
      [&](const int t, const f32x4* sums) {
        if (!mine) return;
        const int n = t * COLS + c;
        f32x4 v = skinny::fold<MT, NW>(sums, slot), u{0.f, 0.f, 0.f, 0.f};
        if constexpr (GATED) u = skinny::fold<MT, NW>(sums, slot + 8);
        if (a.bias) {
          const short* be = a.bias + n;
          v += bf16_to_f32(be[0]);
          if constexpr (GATED) u += bf16_to_f32(be[a.N]);
        }
        store_rows<KIND>(a, v, u, m0 + (slot >> 6) * 16 + (l >> 4) * 4, rows,
                         n);
      });
  __syncthreads();                  // sums read before the next pass's
}

template <int S, int KIND, int PAIRS>
__global__ __launch_bounds__(256, 2) void moe_tiles_kernel(
    const StreamArgs args, const int ntiles) {
  constexpr int KS = skinny::TILES_KS, NW = skinny::TILE_NW;
  __shared__ __attribute__((aligned(128))) short ring[NW][2][16 * KS];
  __shared__ f32x4 red[2][NW][2 * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ unsigned short list[PAIRS ? NW : 1][PAIRS ? PAIRS_MAX : 1];
  const int le = blockIdx.y;
  const StreamArgs a = as_expert<KIND, PAIRS>(args, le);
  const auto rows =
      rows_of<PAIRS>(a, a.e_base + le, list[PAIRS ? wave : 0], lane);
  // An expert that many tokens share would hold up its workgroups for a second
  // pass: as many row tiles as it has.
  for (int m0 = rows.begin; m0 < rows.end; m0 += 32) {
    if (rows.end - m0 > 16)
      stream_pass<2, S, KIND>(a, ntiles, m0, rows, ring[wave][0],
                              &red[0][0][0], wave, lane);
    else
      stream_pass<1, S, KIND>(a, ntiles, m0, rows, ring[wave][0],
                              &red[0][0][0], wave, lane);
  }
}

// pairs: (token, expert) pairs of the step, over all E experts
template <int KIND, int PAIRS>
void launch_rows(const StreamArgs& a, int64_t E_local, int64_t pairs,
                 int64_t E) {
  const int64_t E_chosen = E_local;
  E_local += PAIRS == 2;
  const dim3 grid(a.N / (KIND == UP_GATED ? 8 : 16), E_local), block(256);
  auto stream = at::hip::getCurrentHIPStream();
  // two row tiles once most experts have more than one
  const bool two = pairs > 12 * E;
  // With K = 2048 and up to 32 experts, workgroups that stay
  // (skinny::stream_tiles), from three tiles per CU on of the experts that are
  // likely hit, where equal shares of them come out even. us, per tile and
  // staying. By pairs, 8 experts of 2048 x 2048, top 2, up 15.0 and 12.7, 20.0 and
  // 18.8, 28.5 and 24.3, 30.1 and 24.4, 40.3 and 25.7 at 2, 4, 16, 32 and 64
  // tokens; down 14.2 and 12.6, 17.0 and 13.9, 21.5 and 15.3 at 6, 32 and 64; 16
  // experts up 23.3 and 18.7 at 4, 49.8 and 41.9 at 32, but 21.8 and 24.6 at 3: 6
  // pairs, 42 workgroups each for 256 tiles. Sorted, 32 of 2048 x 768, top 8, up
  // 39.5 and 33.7 at 32 tokens (all hit), 31.3 and 30.2 at 8 (0.87 of them), 25.2
  // and 25.3 at 4 (0.64), 18.3 and 21.4 at 2 (0.4); 8 of 2048 x 8192 78.2 and 80.6
  // at 8 (0.88), 93.2 and 88.1 at 24: equal shares leave CUs idle when experts are
  // not hit, and equal runs over those that are cost more to find than they give
  // (26.0 and 15.5 for the 32 tokens). 64 of 2048 x 1408, top 6, 39.5 and 53.8 at
  // 4, 99 and 105 at 16. Wider K streams as fast in tiles of their own: 8 of 28672 x
  // 4096, 16 tokens, 275 and 282.
  const double hit =
      E_chosen * (1.0 - std::pow(1.0 - 1.0 / E, (double)pairs)) +
      (E_local - E_chosen);
  // never more than the CUs: a CU with two of them ends late (264
  // workgroups for the 32 tokens: 31.2 and 18.4)
  const int most = (int)(std::min<int64_t>(E_chosen, pairs) + E_local - E_chosen);
  const int per = std::max(1, std::min<int>(grid.x, 256 / most));
  const int rounds = (grid.x + per - 1) / per;
  if (a.K == 2048 && E_local <= 32 && hit * grid.x >= 768 &&
      rounds * per * 8 <= (int)grid.x * 9 &&
      (PAIRS || hit >= 0.9 * E_local)) {
    hipLaunchKernelGGL((moe_tiles_kernel<2, KIND, PAIRS>), dim3(per, E_local),
                       block, 0, stream, a, (int)grid.x);
    return;
  }
#define MS_LAUNCH(MT_, KS_)                                                   \
  hipLaunchKernelGGL((moe_stream_kernel<MT_, KS_, KIND, PAIRS>), grid, block, \
                     0, stream, a)
  if (a.K % 256 == 0) {
    if (two) MS_LAUNCH(2, 256); else MS_LAUNCH(1, 256);
  } else {
    if (two) MS_LAUNCH(2, 64); else MS_LAUNCH(1, 64);
  }
#undef MS_LAUNCH
}

template <int KIND>
void launch_stream(const StreamArgs& a, int64_t E_local, int64_t pairs,
                   int64_t E) {
  if (a.all_w) {
    if constexpr (KIND != UP_PLAIN) launch_rows<KIND, 2>(a, E_local, pairs, E);
  } else if (a.topi) {
    launch_rows<KIND, 1>(a, E_local, pairs, E);
  } else {
    launch_rows<KIND, 0>(a, E_local, pairs, E);
  }
}

void check16(const at::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 &&
              t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0);
}

}  // namespace

namespace {

// rows of `act`/`y` by sorted rows (offsets, ids) or by pairs (topi [T, top])
struct RowArgs {
  at::Tensor offsets, ids, topi;
  int64_t pairs, E;                 // of all experts
};

void set_rows(StreamArgs& a, const RowArgs& r, int64_t e_base, int64_t n_local,
              const at::Tensor& w) {
  TORCH_CHECK(e_base >= 0 && n_local >= 0 && w.size(0) >= n_local);
  a.e_base = (int)e_base;
  if (r.topi.defined()) {
    TORCH_CHECK(r.topi.is_cuda() && r.topi.is_contiguous() &&
                r.topi.dim() == 2 && r.topi.dtype() == at::kInt &&
                r.pairs <= PAIRS_MAX);
    a.topi = r.topi.data_ptr<int>();
    a.pairs = (int)r.pairs;
    a.top = (int)r.topi.size(1);
  } else {
    TORCH_CHECK(r.offsets.dtype() == at::kInt &&
                r.offsets.numel() > e_base + n_local);
    a.offsets = r.offsets.data_ptr<int>();
    if (r.ids.defined()) {
      TORCH_CHECK(r.ids.dtype() == at::kInt);
      a.rows = r.ids.data_ptr<int>();
    }
  }
}

void up_rows(at::Tensor& act, const at::Tensor& x, const at::Tensor& w_gate_up,
             const RowArgs& rows, const at::Tensor& bias, int64_t act_mode,
             int64_t e_base, int64_t n_local, double act_limit,
             const at::Tensor& all_w, const at::Tensor& all_act) {
  check16(act); check16(x); check16(w_gate_up);
  const bool gated = act_mode != 2;
  StreamArgs a{};
  a.N = act.size(1); a.K = x.size(1);
  TORCH_CHECK(a.K % 64 == 0 && a.N % 64 == 0,
              "H/IE must be multiples of 64 for the fused MoE path");
  TORCH_CHECK(w_gate_up.size(1) == (gated ? 2 : 1) * (int64_t)a.N &&
              w_gate_up.size(2) == a.K && act.size(0) >= rows.pairs);
  if (bias.numel() > 0) {
    TORCH_CHECK(bias.dtype() == at::kBFloat16 && bias.is_contiguous() &&
                bias.numel() == w_gate_up.size(0) * 2 * a.N);
    a.bias = (const short*)bias.data_ptr();
  }
  TORCH_CHECK(gated || a.bias == nullptr, "ungated experts take no bias");
  set_rows(a, rows, e_base, n_local, w_gate_up);
  if (rows.pairs == 0 || n_local == 0 || a.N == 0) return;
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w_gate_up.data_ptr();
  a.act_mode = (int)act_mode;
  a.limit = (float)act_limit;
  a.act = (short*)act.data_ptr();
  if (all_w.defined() && all_w.numel() > 0) {
    check16(all_w); check16(all_act);
    const int64_t T = x.size(0);
    TORCH_CHECK(rows.topi.defined() && gated && act_mode == 0 && !a.bias &&
                all_w.numel() == 2 * (int64_t)a.N * a.K &&
                all_act.numel() == T * a.N && T * a.top == rows.pairs);
    a.all_w = (const short*)all_w.data_ptr();
    a.all_act = (short*)all_act.data_ptr();
  }
  if (gated) launch_stream<UP_GATED>(a, n_local, rows.pairs, rows.E);
  else launch_stream<UP_PLAIN>(a, n_local, rows.pairs, rows.E);
}

void down_rows(at::Tensor& y, const at::Tensor& act, const at::Tensor& w_down,
               const RowArgs& rows, const at::Tensor& bias, int64_t e_base,
               int64_t n_local, const at::Tensor& all_w,
               const at::Tensor& all_act, const at::Tensor& all_y) {
  TORCH_CHECK(y.is_cuda() && y.dtype() == at::kFloat && y.is_contiguous());
  check16(act); check16(w_down);
  StreamArgs a{};
  a.N = y.size(1); a.K = act.size(1);
  TORCH_CHECK(a.N % 64 == 0 && a.K % 64 == 0);
  TORCH_CHECK(w_down.size(1) == a.N && w_down.size(2) == a.K &&
              act.size(0) >= y.size(0));
  if (bias.numel() > 0) {
    TORCH_CHECK(bias.dtype() == at::kBFloat16 && bias.is_contiguous() &&
                bias.numel() == w_down.size(0) * a.N);
    a.bias = (const short*)bias.data_ptr();
  }
  set_rows(a, rows, e_base, n_local, w_down);
  if (y.size(0) == 0 || n_local == 0 || a.N == 0) return;
  a.x = (const short*)act.data_ptr();
  a.w = (const short*)w_down.data_ptr();
  a.y = y.data_ptr<float>();
  if (all_w.defined() && all_w.numel() > 0) {
    check16(all_w); check16(all_act); check16(all_y);
    const int64_t T = rows.topi.defined() ? rows.topi.size(0) : -1;
    TORCH_CHECK(!a.bias && all_w.numel() == (int64_t)a.N * a.K &&
                all_act.numel() == T * a.K && all_y.numel() == T * a.N);
    a.all_w = (const short*)all_w.data_ptr();
    a.all_act = (short*)all_act.data_ptr();
    a.all_y = (short*)all_y.data_ptr();
  }
  launch_stream<DOWN>(a, n_local, rows.pairs, rows.E);
}

}  // namespace

void moe_gate_silu(at::Tensor act, at::Tensor x, at::Tensor w_gate_up,
                   at::Tensor sorted_ids, at::Tensor offsets,
                   at::Tensor bias, int64_t act_mode,
                   int64_t e_base, int64_t n_local_experts,
                   double act_limit) {
  up_rows(act, x, w_gate_up,
          {offsets, sorted_ids, {}, sorted_ids.numel(), offsets.numel() - 1},
          bias, act_mode, e_base, n_local_experts, act_limit,
          at::Tensor(), at::Tensor());
}

void moe_down_rows(at::Tensor y, at::Tensor act, at::Tensor w_down,
                   at::Tensor offsets, at::Tensor bias, int64_t e_base,
                   int64_t n_local_experts) {
  down_rows(y, act, w_down,
            {offsets, {}, {}, y.size(0), offsets.numel() - 1}, bias, e_base,
            n_local_experts, at::Tensor(), at::Tensor(), at::Tensor());
}

void moe_up_pairs(at::Tensor act, at::Tensor x, at::Tensor w_gate_up,
                  at::Tensor topi, at::Tensor bias, int64_t act_mode,
                  int64_t n_experts, int64_t e_base, int64_t n_local_experts,
                  double act_limit, at::Tensor all_w, at::Tensor all_act) {
  TORCH_CHECK(x.size(0) == topi.size(0));
  up_rows(act, x, w_gate_up, {{}, {}, topi, topi.numel(), n_experts}, bias,
          act_mode, e_base, n_local_experts, act_limit, all_w, all_act);
}

void moe_down_pairs(at::Tensor y, at::Tensor act, at::Tensor w_down,
                    at::Tensor topi, at::Tensor bias, int64_t n_experts,
                    int64_t e_base, int64_t n_local_experts, at::Tensor all_w,
                    at::Tensor all_act, at::Tensor all_y) {
  TORCH_CHECK(y.size(0) == topi.numel());
  down_rows(y, act, w_down, {{}, {}, topi, topi.numel(), n_experts}, bias,
            e_base, n_local_experts, all_w, all_act, all_y);
}

}  // namespace kaito
