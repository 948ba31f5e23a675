// Expert choice for routed feed-forwards, in two launches.
//
//   moe_route: one wave per token, from f32 logits; moe_gate_route: one
//     workgroup per token (of long steps per 16 tokens), which also forms the
//     logits x W^T. Modes:
//     SOFTMAX: s = softmax(logits), choice = s + correction (none given: s);
//       a group of `groups` equal groups of neighbours scores its largest
//       choice;
//     SIGMOID: s = sigmoid(logits), choice alike; a group scores the sum of
//       its two largest choices;
//     LOGITS: the choice is the logit itself, the weights are a softmax over
//       the taken logits.
//     Only the `keep` best groups stay eligible; the `top` largest eligible
//     choices are taken (ties: lower index; a NaN counts as larger than every
//     number, and where fewer than `top` are above -inf the lowest indices
//     among the others fill up). Weights are the taken s
//     (without the correction), divided by their sum + 1e-20 when `renorm`,
//     times `scale`. Outputs with index >= n_real are identity experts: their
//     weights are also summed per token.
//   moe_sort: stable counting sort of the (token, expert) pairs by expert:
//     token and weight of every sorted row, exclusive offsets, row of every
//     pair. Ranks among 64 pairs come from a ballot per bit of the expert's
//     number, so the order does not depend on timing and the time not on how
//     many experts there are. One workgroup up to 2048 pairs; beyond, one per
//     1024 pairs behind a counting launch (16384 pairs took 46 us in one
//     workgroup).
//
// A decode step's choice is launches and latency, not work: as torch ops
// (product, cast, top-k, softmax, sort, gathers, scatter, scan) it was about
// 25 launches, 130 us of a layer's 240 at 32 tokens and 8 experts. Now it is
// 4.4 us for logits and choice (rows of 2048, one launch behind another; 9.5
// where the row before has to arrive from its norm) and 4.8 for the sort.
//
// An output's place in the row lives in lane e % 64, register e / 64.
#include "mix_common.h"
#include "skinny.h"
#include <type_traits>

namespace kaito {

namespace {

constexpr int ROUTE_MAX = 1024;      // router outputs

// largest value over `width` neighbouring lanes (a power of two), ties to the lower
// index. A choice is a chain of these: within 16 lanes the neighbours' values come
// by DPP and not through LDS, and few outputs need few steps (32 rows of 8 outputs
// in 4 groups, of which 2 stay, top 2: 9.3 us with 6 steps of two LDS exchanges each,
// one group after the other, now 5.4; 600 rows of 16 14.1 and 9.8; without groups 5.0
// and 4.4).
template <int CTRL>
KAITO_DEV int dpp(const int x) {
  return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false);
}
KAITO_DEV void lanes_argmax(float& v, int& i, const int width) {
  auto take = [&](const float ov, const int oi) {
    if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
  };
  // behind a step all lanes of its width agree, so that a mirror is as good as an
  // exchange
#define ROUTE_STEP(W_, CTRL_)                                                 \
  if (width > W_)                                                             \
    take(__int_as_float(dpp<CTRL_>(__float_as_int(v))), dpp<CTRL_>(i))
  ROUTE_STEP(1, 0xB1);              // quad_perm 1 0 3 2
  ROUTE_STEP(2, 0x4E);              // quad_perm 2 3 0 1
  ROUTE_STEP(4, 0x141);             // row_half_mirror
  ROUTE_STEP(8, 0x128);             // row_ror 8
#undef ROUTE_STEP
  if (width > 16) take(__shfl_xor(v, 16, 64), __shfl_xor(i, 16, 64));
  if (width > 32) take(__shfl_xor(v, 32, 64), __shfl_xor(i, 32, 64));
}
KAITO_DEV float lanes_max(float v, const int width) {
#define ROUTE_STEP(W_, CTRL_)                                                 \
  if (width > W_) v = fmaxf(v, __int_as_float(dpp<CTRL_>(__float_as_int(v))))
  ROUTE_STEP(1, 0xB1);
  ROUTE_STEP(2, 0x4E);
  ROUTE_STEP(4, 0x141);
  ROUTE_STEP(8, 0x128);
#undef ROUTE_STEP
  if (width > 16) v = fmaxf(v, __shfl_xor(v, 16, 64));
  if (width > 32) v = fmaxf(v, __shfl_xor(v, 32, 64));
  return v;
}
KAITO_DEV int lanes_for(const int n) {      // the width that holds n lanes
  return n <= 1 ? 1 : n > 32 ? 64 : 1 << (32 - __builtin_clz(n - 1));
}

constexpr int NONE = 1 << 30;        // a lane without a candidate

enum Mode { SOFTMAX = 0, SIGMOID = 1, LOGITS = 2 };

struct RouteArgs {
  int* topi;                        // [T, top]
  float* topw;                      // [T, top]
  float* w_id;                      // [T]
  const float* correction;          // [N] or nullptr
  int T, N, n_real, top, groups, keep;
  bool renorm;
  float scale;
};

// one wave: the choice of token t from its logits (row: N floats)
template <int NPL, int MODE>
KAITO_DEV void route_row(const RouteArgs& a, const float* row, const int64_t t,
                         const int lane) {
  const int N = a.N;
  float s[NPL], ch[NPL];
  float mx = -INFINITY;
#pragma unroll
  for (int r = 0; r < NPL; r++) {
    const int e = r * 64 + lane;
    s[r] = e < N ? row[e] : -INFINITY;
    mx = fmaxf(mx, s[r]);
  }
  if constexpr (MODE == SIGMOID) {
#pragma unroll
    for (int r = 0; r < NPL; r++) {
      const int e = r * 64 + lane;
      s[r] = sigmoid_f(s[r]);
      ch[r] = e < N ? s[r] + (a.correction ? a.correction[e] : 0.f)
                    : -INFINITY;
    }
  } else {
    mx = lanes_max(mx, NPL == 1 ? lanes_for(N) : 64);
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < NPL; r++) {
      if constexpr (MODE == LOGITS) ch[r] = s[r];
      s[r] = r * 64 + lane < N ? expf(s[r] - mx) : 0.f;
      sum += s[r];
    }
    if constexpr (MODE == SOFTMAX) {
      sum = wave_reduce_sum(sum);
#pragma unroll
      for (int r = 0; r < NPL; r++) {
        const int e = r * 64 + lane;
        s[r] = s[r] / sum;
        ch[r] = e < N ? s[r] + (a.correction ? a.correction[e] : 0.f)
                      : -INFINITY;
      }
    }
  }
  // as in a sort, a NaN is larger than every number
  auto rank = [](const float v) { return v == v ? v : INFINITY; };
#pragma unroll
  for (int r = 0; r < NPL; r++) ch[r] = rank(ch[r]);
  if (a.groups > 1) {
    const int n = N / a.groups;
    float mine = -INFINITY;                 // lane g: group g's score
    if (NPL == 1 && (n & (n - 1)) == 0) {   // all at once
      float score = ch[0];
      int mi = lane;
      lanes_argmax(score, mi, n);
      if (MODE == SIGMOID && n > 1) {
        float m2 = lane == mi ? -INFINITY : ch[0];      // the second largest
        int at = lane;
        lanes_argmax(m2, at, n);
        score += m2;
      }
      score = rank(__shfl(score, lane * n & 63, 64));
      if (lane < a.groups) mine = score;
    } else {
      for (int g = 0; g < a.groups; g++) {
        float m = -INFINITY;
        int mi = N;
#pragma unroll
        for (int r = 0; r < NPL; r++) {
          const int e = r * 64 + lane;
          if (e >= g * n && e < (g + 1) * n && (ch[r] > m || mi == N)) {
            m = ch[r];
            mi = e;
          }
        }
        float score;
        if constexpr (MODE == SIGMOID) {
          lanes_argmax(m, mi, 64);
          score = m;
          float m2 = -INFINITY;               // the second largest
#pragma unroll
          for (int r = 0; r < NPL; r++) {
            const int e = r * 64 + lane;
            if (e >= g * n && e < (g + 1) * n && e != mi) m2 = fmaxf(m2, ch[r]);
          }
          if (n > 1) score += wave_reduce_max(m2);
        } else {
          score = wave_reduce_max(m);
        }
        if (lane == g) mine = rank(score);
      }
    }
    unsigned long long kept = 0;
    for (int k = 0; k < a.keep; k++) {
      const bool open = lane < a.groups && !((kept >> lane) & 1);
      float v = open ? mine : -INFINITY;
      int i = open ? lane : NONE;
      lanes_argmax(v, i, lanes_for(a.groups));
      kept |= 1ull << __builtin_amdgcn_readfirstlane(i);
    }
#pragma unroll
    for (int r = 0; r < NPL; r++) {
      const int e = r * 64 + lane;
      if (e < N && !((kept >> (e / n)) & 1)) ch[r] = -INFINITY;
    }
  }
  float wsum = 0.f, mine = 0.f;             // lane k: k-th taken weight
  int mine_i = 0;
  unsigned open = 0;                        // outputs of this lane not taken
#pragma unroll
  for (int r = 0; r < NPL; r++)
    if (r * 64 + lane < N) open |= 1u << r;
  for (int k = 0; k < a.top; k++) {         // top <= N: one is always open
    float v = -INFINITY;
    int i = NONE;
#pragma unroll
    for (int r = 0; r < NPL; r++)
      if ((open >> r & 1) && (ch[r] > v || i == NONE)) {
        v = ch[r];
        i = r * 64 + lane;
      }
    lanes_argmax(v, i, NPL == 1 ? lanes_for(N) : 64);
    i = __builtin_amdgcn_readfirstlane(i);
    float sv = 0.f;
#pragma unroll
    for (int r = 0; r < NPL; r++) {
      const float b = __int_as_float(
          __builtin_amdgcn_readlane(__float_as_int(s[r]), i & 63));
      if (r == (i >> 6)) sv = b;
      if (r * 64 + lane == i) open &= ~(1u << r);
    }
    wsum += sv;
    if (lane == k) { mine = sv; mine_i = i; }
  }
  if constexpr (MODE == LOGITS)
    mine = mine / wsum * a.scale;
  else
    mine *= a.renorm ? a.scale / (wsum + 1e-20f) : a.scale;
  if (lane < a.top) {
    a.topi[t * a.top + lane] = mine_i;
    a.topw[t * a.top + lane] = mine;
  }
  const float idw = wave_reduce_sum(lane < a.top && mine_i >= a.n_real ? mine
                                                                       : 0.f);
  if (lane == 0) a.w_id[t] = idw;
}

template <int NPL, int MODE>
__global__ __launch_bounds__(256) void moe_route_kernel(
    const RouteArgs a, const float* __restrict__ logits) {
  const int64_t t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.T) return;                     // whole waves; no barriers below
  route_row<NPL, MODE>(a, logits + t * a.N, t, threadIdx.x & 63);
}

constexpr int GATE_MAX = 32;         // outputs whose logits a workgroup forms

KAITO_DEV float dot_gate(const skinny::hbf16x8 x, const short* w, float c) {
  return skinny::dot8(x, skinny::load_x(w), c);
}
KAITO_DEV float dot_gate(const skinny::hbf16x8 x, const float* w, float c) {
  const float4_t a = *reinterpret_cast<const float4_t*>(w);
  const float4_t b = *reinterpret_cast<const float4_t*>(w + 4);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c = fmaf((float)x[i], a[i], c);
    c = fmaf((float)x[i + 4], b[i], c);
  }
  return c;
}

// W: the router's element (bf16 or f32); H is a multiple of 8
template <int MODE, typename W>
__global__ __launch_bounds__(256) void moe_gate_route_kernel(
    const RouteArgs a, const short* __restrict__ x, const int64_t x_stride,
    const W* __restrict__ w, const int H) {
  __shared__ float part[4][GATE_MAX];
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const short* xr = x + t * x_stride;
  for (int e0 = 0; e0 < a.N; e0 += 8) {
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = 0.f;
    for (int k = threadIdx.x * 8; k < H; k += 2048) {
      const skinny::hbf16x8 xv = skinny::load_x(xr + k);
#pragma unroll
      for (int i = 0; i < 8; i++)
        acc[i] = dot_gate(xv, w + (int64_t)min(e0 + i, a.N - 1) * H + k,
                          acc[i]);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc[i] = wave_reduce_sum(acc[i]);
      if (lane == 0 && e0 + i < a.N) part[wave][e0 + i] = acc[i];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  if (lane < a.N)
    part[0][lane] += part[1][lane] + part[2][lane] + part[3][lane];
  __builtin_amdgcn_wave_barrier();
  route_row<1, MODE>(a, part[0], t, lane);
}

// Prompts: 16 rows per workgroup, products on v_mfma_f32_16x16x32_bf16. A wave
// takes the dims 128 w .. of every 2048 and, once the 16 partial sums are added,
// the choice of one row: logits never leave the workgroup. An f32 router is three
// bf16 terms to the last bit, so three products have the exact terms of an f32 one
// and rows need no cast. Bound by latency up to 2048 rows, behind them by reading
// rows and router through L2; a workgroup per row reads the router 16 times as
// often (us, product by the library and choice -> here, rows of 2048, 8 outputs:
// bf16 router 9.1 -> 7.0 at 600 rows, 14.7 -> 10.8 at 8192 (row by row 20.4); f32
// 15.7 -> 8.4 and 38.0 -> 14.4 (27.2)). Loads of a round's router ahead of its
// products cost f32 routers half their waves: a fifth more. Error of the weights
// against f64 logits at 8192 rows: 1.8e-7, of the library's 3.0e-7 and 6.6e-7.
constexpr int GATE_ROWS = 16, GATE_STEPS = 4;

// the terms of 8 elements of the router, largest first
KAITO_DEV void gate_terms(const short* w, skinny::hbf16x8 (&b)[1]) {
  b[0] = skinny::load_x(w);
}
KAITO_DEV void gate_terms(const float* w, skinny::hbf16x8 (&b)[3]) {
  const float4_t lo = *reinterpret_cast<const float4_t*>(w);
  const float4_t hi = *reinterpret_cast<const float4_t*>(w + 4);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    __bf16 t[3];
    bf16_terms(i < 4 ? lo[i & 3] : hi[i & 3], t);
#pragma unroll
    for (int n = 0; n < 3; n++) b[n][i] = t[n];
  }
}

// NT: 16 outputs each; H is a multiple of 32
template <int MODE, typename W, int NT>
__global__ __launch_bounds__(1024) void moe_gate_route_tiles_kernel(
    const RouteArgs a, const short* __restrict__ x, const int64_t x_stride,
    const W* __restrict__ w, const int H) {
  constexpr int TERMS = sizeof(W) == 4 ? 3 : 1, COLS = NT * 16 + 1;
  __shared__ float part[16][GATE_ROWS][COLS], logit[GATE_ROWS][COLS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, q = lane >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * GATE_ROWS;
  const short* xr = x + min(t0 + c, (int64_t)a.T - 1) * x_stride + q * 8;
  float4_t acc[NT][TERMS > 1 ? 2 : 1];      // the largest terms, the rest
#pragma unroll
  for (int n = 0; n < NT; n++)
    for (auto& v : acc[n]) v = float4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = wave * 32 * GATE_STEPS; k0 < H; k0 += 512 * GATE_STEPS) {
    skinny::hbf16x8 xv[GATE_STEPS];
#pragma unroll
    for (int i = 0; i < GATE_STEPS; i++)
      xv[i] = skinny::load_x(xr + min(k0 + 32 * i, H - 32));
#pragma unroll
    for (int i = 0; i < GATE_STEPS; i++) {
      const int k = k0 + 32 * i;
      if (k >= H) break;
      bool wild = false;                    // an infinity or a NaN in x
      if constexpr (TERMS > 1) {
#pragma unroll
        for (int e = 0; e < 8; e++)
          wild |= !(fabsf((float)xv[i][e]) < INFINITY);
        wild = __any(wild);
      }
#pragma unroll
      for (int n = 0; n < NT; n++) {
        skinny::hbf16x8 b[TERMS];
        gate_terms(w + (int64_t)min(n * 16 + c, a.N - 1) * H + k + q * 8, b);
        acc[n][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[i], b[0],
                                                            acc[n][0], 0, 0, 0);
        if constexpr (TERMS > 1) {
          // an infinity is multiplied once: its product with a smaller term
          // could have the other sign, or be 0 times it
          auto xs = xv[i];
          if (wild) {
#pragma unroll
            for (int e = 0; e < 8; e++)
              if (!(fabsf((float)xs[e]) < INFINITY)) xs[e] = (__bf16)0.f;
          }
#pragma unroll
          for (int j = TERMS - 1; j > 0; j--)
            acc[n][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xs, b[j], acc[n][1], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float v = acc[n][0][r];
      if constexpr (TERMS > 1) v += acc[n][1][r];
      part[wave][q * 4 + r][n * 16 + c] = v;
    }
  __syncthreads();
  // wave r: row r. Lane: output lane % 16 (% 32), and a share of the sums
  constexpr int SHARE = 64 / (NT * 16), EACH = 16 / SHARE;
  const int col = lane % (NT * 16), first = lane / (NT * 16) * EACH;
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < EACH; i++) sum += part[first + i][wave][col];
#pragma unroll
  for (int off = NT * 16; off < 64; off <<= 1) sum += __shfl_xor(sum, off, 64);
  if (lane < NT * 16) logit[wave][lane] = sum;
  __builtin_amdgcn_wave_barrier();
  if (t0 + wave < a.T) route_row<1, MODE>(a, logit[wave], t0 + wave, lane);
}

// The residual norm ahead of the router in the same launch: residual += x, xn =
// rms(residual) * w, logits of xn as rounded to bf16. A thread keeps its 8 * ITER
// elements. 32 rows of 2048 with 8 outputs: 4.6 + 5.3 us -> 5.7.
template <int MODE, typename W, int ITER>
__global__ __launch_bounds__(256) void moe_norm_gate_route_kernel(
    const RouteArgs a, short* __restrict__ xn, short* __restrict__ residual,
    const short* __restrict__ x, const short* __restrict__ nw,
    const float eps, const W* __restrict__ w, const int H) {
  __shared__ float part[4][GATE_MAX], red[4];
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  short8_t v[ITER], g[ITER];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int k = i * 2048 + threadIdx.x * 8;
    if (k >= H) break;
    const short8_t xv = *reinterpret_cast<const short8_t*>(x + t * H + k);
    const short8_t rv =
        *reinterpret_cast<const short8_t*>(residual + t * H + k);
    g[i] = *reinterpret_cast<const short8_t*>(nw + k);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] = f32_to_bf16(bf16_to_f32(xv[e]) + bf16_to_f32(rv[e]));
      const float f = bf16_to_f32(v[i][e]);
      ss += f * f;
    }
    *reinterpret_cast<short8_t*>(residual + t * H + k) = v[i];
  }
  ss = wave_reduce_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  const float inv = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < ITER; i++) {
    const int k = i * 2048 + threadIdx.x * 8;
    if (k >= H) break;
#pragma unroll
    for (int e = 0; e < 8; e++)
      v[i][e] = f32_to_bf16(bf16_to_f32(v[i][e]) * inv * bf16_to_f32(g[i][e]));
    *reinterpret_cast<short8_t*>(xn + t * H + k) = v[i];
  }
  for (int e0 = 0; e0 < a.N; e0 += 8) {
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = 0.f;
#pragma unroll
    for (int j = 0; j < ITER; j++) {
      const int k = j * 2048 + threadIdx.x * 8;
      if (k >= H) break;
      const auto xv = __builtin_bit_cast(skinny::hbf16x8, v[j]);
#pragma unroll
      for (int i = 0; i < 8; i++)
        acc[i] = dot_gate(xv, w + (int64_t)min(e0 + i, a.N - 1) * H + k,
                          acc[i]);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc[i] = wave_reduce_sum(acc[i]);
      if (lane == 0 && e0 + i < a.N) part[wave][e0 + i] = acc[i];
    }
  }
  __syncthreads();
  if (wave != 0) return;
  if (lane < a.N)
    part[0][lane] += part[1][lane] + part[2][lane] + part[3][lane];
  __builtin_amdgcn_wave_barrier();
  route_row<1, MODE>(a, part[0], t, lane);
}

// lanes of the wave with this lane's expert e (< 2^bits; any lane with -1 is
// in no group): a ballot per bit, however many experts there are
KAITO_DEV unsigned long long same_expert(const int e, const int bits) {
  unsigned long long m = __ballot(e >= 0);
  for (int b = 0; b < bits; b++) {
    const bool one = (e >> b) & 1;
    const unsigned long long ones = __ballot(one);
    m &= one ? ones : ~ones;
  }
  return m;
}

constexpr int SORT_BLOCK = 1024;     // pairs of a workgroup when several sort

// hist[b][e]: pairs of expert e in block b
__global__ __launch_bounds__(1024) void moe_count_kernel(
    int* __restrict__ hist, const int* __restrict__ topi, const int TK,
    const int N) {
  extern __shared__ int cnt[];              // [N]
  const int tid = threadIdx.x;
  for (int i = tid; i < N; i += SORT_BLOCK) cnt[i] = 0;
  __syncthreads();
  const int i = blockIdx.x * SORT_BLOCK + tid;
  if (i < TK) atomicAdd(&cnt[topi[i]], 1);
  __syncthreads();
  for (int e = tid; e < N; e += SORT_BLOCK)
    hist[(int64_t)blockIdx.x * N + e] = cnt[e];
}

// Pairs are cut into one contiguous run per wave. cnt[w][e]: first the pairs
// of expert e in wave w's run, then the next row of such a pair; row w = waves
// is the experts' starts. hist: counts of SORT_BLOCK pairs each, or nullptr
// for one workgroup
__global__ __launch_bounds__(1024) void moe_sort_kernel(
    int* __restrict__ sorted_tok, float* __restrict__ gates,
    int* __restrict__ offsets, int* __restrict__ pos,
    const int* __restrict__ topi, const float* __restrict__ topw,
    const int* __restrict__ hist, const int TK, const int top, const int N,
    const int bits) {
  extern __shared__ int cnt[];              // [waves + 1][N]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nw = blockDim.x >> 6;
  const int begin = hist ? blockIdx.x * SORT_BLOCK : 0;
  const int end = hist ? min(TK, begin + SORT_BLOCK) : TK;
  const int per = (end - begin + nw * 64 - 1) / (nw * 64) * 64;
  const int first = min(end, begin + wave * per), last = min(end, first + per);
  int* mine = cnt + wave * N;
  int* start = cnt + nw * N;
  for (int i = tid; i < nw * N; i += blockDim.x) cnt[i] = 0;
  __syncthreads();
  for (int i = first + lane; i < last; i += 64) atomicAdd(&mine[topi[i]], 1);
  __syncthreads();
  // a thread per expert: its pairs, and those before each wave's in this block
  for (int e = tid; e < N; e += blockDim.x) {
    int here = 0, before = 0, all = 0;
    if (hist)
      for (unsigned b = 0; b < gridDim.x; b++) {
        const int n = hist[(int64_t)b * N + e];
        if (b < blockIdx.x) before += n;
        all += n;
      }
    for (int w = 0; w < nw; w++) {
      const int c = cnt[w * N + e];
      cnt[w * N + e] = before + here;
      here += c;
    }
    start[e] = hist ? all : here;
  }
  __syncthreads();
  if (wave == 0) {                          // exclusive scan over the experts
    int base = 0;
    for (int e0 = 0; e0 < N; e0 += 64) {
      const int e = e0 + lane, n = e < N ? start[e] : 0;
      int scan = n;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int add = __shfl_up(scan, off, 64);
        if (lane >= off) scan += add;
      }
      if (e < N) {
        start[e] = base + scan - n;
        if (blockIdx.x == 0) offsets[e] = base + scan - n;
      }
      base += __shfl(scan, 63, 64);
    }
    if (blockIdx.x == 0 && lane == 0) offsets[N] = TK;
  }
  __syncthreads();
  for (int i0 = first; i0 < last; i0 += 64) {
    const int i = i0 + lane;
    const int e = i < last ? topi[i] : -1;
    const unsigned long long same = same_expert(e, bits);
    const int rank = __builtin_popcountll(same & ((1ull << lane) - 1));
    if (e >= 0) {
      const int at = start[e] + mine[e] + rank;
      sorted_tok[at] = i / top;
      gates[at] = topw[i];
      pos[i] = at;
    }
    __builtin_amdgcn_wave_barrier();        // all have read mine
    if (e >= 0 && rank == 0) mine[e] += __builtin_popcountll(same);
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace

// checks shared by both entries
static RouteArgs route_args(const at::Tensor& topi, const at::Tensor& topw,
                            const at::Tensor& w_id,
                            const at::Tensor& correction, int64_t T, int64_t N,
                            int64_t n_real, int64_t groups, int64_t keep,
                            bool renorm, double scale, int64_t mode) {
  const bool corr = correction.numel() > 0;
  if (corr) KAITO_CHECK_F32(correction);
  KAITO_CHECK_I32(topi); KAITO_CHECK_F32(topw); KAITO_CHECK_F32(w_id);
  TORCH_CHECK(topi.dim() == 2);
  const int64_t top = topi.size(1);
  TORCH_CHECK(topi.size(0) == T && topw.sizes() == topi.sizes() &&
              w_id.numel() == T && (!corr || correction.numel() == N));
  TORCH_CHECK(N >= 1 && N <= ROUTE_MAX && top >= 1 && top <= 64 && top <= N);
  TORCH_CHECK(groups >= 1 && groups <= 64 && N % groups == 0 && keep >= 1 &&
              keep <= groups);
  TORCH_CHECK(mode >= 0 && mode <= 2 && !(mode == LOGITS && corr));
  RouteArgs a{};
  a.topi = topi.data_ptr<int>();
  a.topw = topw.data_ptr<float>();
  a.w_id = w_id.data_ptr<float>();
  a.correction = corr ? correction.data_ptr<float>() : nullptr;
  a.T = (int)T; a.N = (int)N; a.n_real = (int)n_real; a.top = (int)top;
  a.groups = (int)groups; a.keep = (int)keep;
  a.renorm = renorm; a.scale = (float)scale;
  return a;
}

template <typename F>
static void with_mode(int64_t mode, const F& f) {
  if (mode == SOFTMAX) f(std::integral_constant<int, SOFTMAX>{});
  else if (mode == SIGMOID) f(std::integral_constant<int, SIGMOID>{});
  else f(std::integral_constant<int, LOGITS>{});
}

void moe_route(at::Tensor topi, at::Tensor topw, at::Tensor w_id,
               at::Tensor logits, at::Tensor correction, int64_t n_real,
               int64_t groups, int64_t keep, bool renorm, double scale,
               int64_t mode) {
  KAITO_CHECK_F32(logits);
  TORCH_CHECK(logits.dim() == 2);
  const int T = logits.size(0), N = logits.size(1);
  const RouteArgs a = route_args(topi, topw, w_id, correction, T, N, n_real,
                                 groups, keep, renorm, scale, mode);
  if (T == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  with_mode(mode, [&](auto md) {
    auto launch = [&](auto npl) {
      hipLaunchKernelGGL(
          (moe_route_kernel<decltype(npl)::value, decltype(md)::value>),
          dim3((T + 3) / 4), dim3(256), 0, stream, a,
          logits.data_ptr<float>());
    };
    if (N <= 64) launch(std::integral_constant<int, 1>{});
    else if (N <= 128) launch(std::integral_constant<int, 2>{});
    else if (N <= 256) launch(std::integral_constant<int, 4>{});
    else launch(std::integral_constant<int, 16>{});
  });
}

void moe_gate_route(at::Tensor topi, at::Tensor topw, at::Tensor w_id,
                    at::Tensor x, at::Tensor gate, at::Tensor correction,
                    int64_t n_real, int64_t groups, int64_t keep, bool renorm,
                    double scale, int64_t mode) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == at::kBFloat16 && x.dim() == 2 &&
              x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
              (uintptr_t)x.data_ptr() % 16 == 0);
  TORCH_CHECK(gate.is_cuda() && gate.dim() == 2 && gate.is_contiguous() &&
              gate.size(1) == x.size(1) && x.size(1) % 8 == 0 &&
              (uintptr_t)gate.data_ptr() % 16 == 0);
  const int T = x.size(0), N = gate.size(0), H = x.size(1);
  TORCH_CHECK(N <= GATE_MAX);
  const RouteArgs a = route_args(topi, topw, w_id, correction, T, N, n_real,
                                 groups, keep, renorm, scale, mode);
  if (T == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const bool f32 = gate.dtype() == at::kFloat;
  TORCH_CHECK(f32 || gate.dtype() == at::kBFloat16);
  // short steps go row by row: 512 rows of 2048, 8 outputs, 6.5 us and 7.6
  if (H % 32 == 0 && (T > 512 || (int64_t)T * N > 8192)) {
    const int blocks = (T + GATE_ROWS - 1) / GATE_ROWS;
    with_mode(mode, [&](auto md) {
      auto launch = [&](auto nt, auto wt) {
        using W = decltype(wt);
        hipLaunchKernelGGL(
            (moe_gate_route_tiles_kernel<decltype(md)::value, W,
                                         decltype(nt)::value>),
            dim3(blocks), dim3(1024), 0, stream, a, (const short*)x.data_ptr(),
            x.stride(0), (const W*)gate.data_ptr(), H);
      };
      auto sized = [&](auto wt) {
        if (N <= 16) launch(std::integral_constant<int, 1>{}, wt);
        else launch(std::integral_constant<int, 2>{}, wt);
      };
      if (f32) sized(0.f); else sized((short)0);
    });
    return;
  }
  with_mode(mode, [&](auto md) {
    if (f32) {
      hipLaunchKernelGGL((moe_gate_route_kernel<decltype(md)::value, float>),
          dim3(T), dim3(256), 0, stream, a, (const short*)x.data_ptr(),
          x.stride(0), gate.data_ptr<float>(), H);
    } else {
      hipLaunchKernelGGL((moe_gate_route_kernel<decltype(md)::value, short>),
          dim3(T), dim3(256), 0, stream, a, (const short*)x.data_ptr(),
          x.stride(0), (const short*)gate.data_ptr(), H);
    }
  });
}

void moe_norm_gate_route(at::Tensor topi, at::Tensor topw, at::Tensor w_id,
                         at::Tensor xn, at::Tensor residual, at::Tensor x,
                         at::Tensor norm_w, double eps, at::Tensor gate,
                         at::Tensor correction, int64_t n_real, int64_t groups,
                         int64_t keep, bool renorm, double scale,
                         int64_t mode) {
  for (const auto& t : {xn, residual, x, norm_w})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 &&
                t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(x.dim() == 2 && xn.sizes() == x.sizes() &&
              residual.sizes() == x.sizes() && norm_w.numel() == x.size(1));
  TORCH_CHECK(gate.is_cuda() && gate.dim() == 2 && gate.is_contiguous() &&
              gate.size(1) == x.size(1) && x.size(1) % 8 == 0 &&
              (uintptr_t)gate.data_ptr() % 16 == 0);
  const int T = x.size(0), N = gate.size(0), H = x.size(1);
  TORCH_CHECK(N <= GATE_MAX && H <= 8192);
  const RouteArgs a = route_args(topi, topw, w_id, correction, T, N, n_real,
                                 groups, keep, renorm, scale, mode);
  if (T == 0) return;
  const bool f32 = gate.dtype() == at::kFloat;
  TORCH_CHECK(f32 || gate.dtype() == at::kBFloat16);
  auto stream = at::hip::getCurrentHIPStream();
  with_mode(mode, [&](auto md) {
    auto launch = [&](auto it, auto wt) {
      using W = decltype(wt);
      hipLaunchKernelGGL(
          (moe_norm_gate_route_kernel<decltype(md)::value, W,
                                      decltype(it)::value>),
          dim3(T), dim3(256), 0, stream, a, (short*)xn.data_ptr(),
          (short*)residual.data_ptr(), (const short*)x.data_ptr(),
          (const short*)norm_w.data_ptr(), (float)eps,
          (const W*)gate.data_ptr(), H);
    };
    auto sized = [&](auto wt) {
      if (H <= 2048) launch(std::integral_constant<int, 1>{}, wt);
      else if (H <= 4096) launch(std::integral_constant<int, 2>{}, wt);
      else launch(std::integral_constant<int, 4>{}, wt);
    };
    if (f32) sized(0.f); else sized((short)0);
  });
}

void moe_sort(at::Tensor sorted_tok, at::Tensor gates, at::Tensor offsets,
              at::Tensor pos, at::Tensor topi, at::Tensor topw) {
  KAITO_CHECK_I32(topi); KAITO_CHECK_F32(topw); KAITO_CHECK_I32(pos);
  KAITO_CHECK_I32(sorted_tok); KAITO_CHECK_F32(gates);
  KAITO_CHECK_I32(offsets);
  TORCH_CHECK(topi.dim() == 2 && topw.sizes() == topi.sizes());
  TORCH_CHECK(topi.numel() < (1ll << 31) - (1 << 20));
  const int TK = topi.numel(), top = topi.size(1);
  const int N = offsets.numel() - 1;
  TORCH_CHECK(sorted_tok.numel() == TK && gates.numel() == TK &&
              pos.numel() == TK && N >= 1 && N <= ROUTE_MAX);
  auto stream = at::hip::getCurrentHIPStream();
  // waves by the number of 64-pair rounds; their counters fit 64 KB
  const int nw = TK <= 256 ? 4 : (N <= 960 ? 16 : 8);
  const int blocks = TK <= 2048 ? 1 : (TK + SORT_BLOCK - 1) / SORT_BLOCK;
  at::Tensor hist;
  if (blocks > 1) {
    hist = at::empty({blocks, N}, topi.options());
    hipLaunchKernelGGL(moe_count_kernel, dim3(blocks), dim3(SORT_BLOCK),
        (size_t)N * 4, stream, hist.data_ptr<int>(), topi.data_ptr<int>(), TK,
        N);
  }
  int bits = 0;
  while ((1 << bits) < N) bits++;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(blocks), dim3(nw * 64),
      (size_t)(nw + 1) * N * 4, stream, sorted_tok.data_ptr<int>(),
      gates.data_ptr<float>(), offsets.data_ptr<int>(), pos.data_ptr<int>(),
      topi.data_ptr<int>(), topw.data_ptr<float>(),
      blocks > 1 ? hist.data_ptr<int>() : nullptr, TK, top, N, bits);
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("moe_route(Tensor(a!) topi, Tensor(b!) topw, Tensor(c!) w_id, Tensor logits, Tensor correction, int n_real, int groups, int keep, bool renorm, float scale, int mode) -> ()");
  m.def("moe_gate_route(Tensor(a!) topi, Tensor(b!) topw, Tensor(c!) w_id, Tensor x, Tensor gate, Tensor correction, int n_real, int groups, int keep, bool renorm, float scale, int mode) -> ()");
  m.def("moe_norm_gate_route(Tensor(a!) topi, Tensor(b!) topw, Tensor(c!) w_id, Tensor(d!) xn, Tensor(e!) residual, Tensor x, Tensor norm_w, float eps, Tensor gate, Tensor correction, int n_real, int groups, int keep, bool renorm, float scale, int mode) -> ()");
  m.def("moe_sort(Tensor(a!) sorted_tok, Tensor(b!) gates, Tensor(c!) offsets, Tensor(d!) pos, Tensor topi, Tensor topw) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("moe_route", &kaito::moe_route);
  m.impl("moe_gate_route", &kaito::moe_gate_route);
  m.impl("moe_norm_gate_route", &kaito::moe_norm_gate_route);
  m.impl("moe_sort", &kaito::moe_sort);
}
