// Real-gated linear recurrent unit for batches of chunks.
//
// Per channel c (block blk = c / bw of the block-diagonal gates):
//     r = sigmoid(gates[blk, t, c % bw])        recurrence gate
//     i = sigmoid(gates[blk, t, bw + c % bw])   input gate
//     log a = -r * decay_rate[c];  a = exp(log a)
//     S <- a * S + sqrt(1 - a^2) * i * u[t, c]
//     out[t, c] = S * gelu_tanh(y[t, c])
// The gate pre-activations come from a batched f32 matrix product; the
// recurrence is diagonal, so one thread owns one channel of one chunk and
// walks its tokens in order (loads of later tokens do not depend on S and
// pipeline freely). sqrt(1 - a^2) is evaluated as sqrt(-expm1(2 log a)),
// which keeps its precision when a is close to 1. S is f32 in the state
// slot; a chunk starting at position 0 starts from S = 0.
//
// Prompts are bound by the vector unit, not by memory: the gates'
// exponentials and quotients. They are written to need few of both: 1 - a^2
// from the same expm1 as a, gelu_tanh by the logistic function it equals,
// quotients by the reciprocal and one Newton step. Error of f32 outputs over
// 2048 tokens against f64, relative to their rms: 2.1e-7 before, 1.3e-7 now;
// with slow decay 5.1e-6 and 7.5e-7.
#include "mix_common.h"

namespace kaito {

namespace {

// 1 / d for 1 <= d <= e^88: one Newton step on the hardware's reciprocal
KAITO_DEV float recip_f(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.0f), r, r);
}
KAITO_DEV float logistic_f(float x) {   // 0 below -80: 2e-35
  return x < -80.0f ? 0.0f : recip_f(1.0f + expf(-x));
}
// z / 2 (1 + tanh u) = z logistic(2 u)
KAITO_DEV float gelu_f(float z) {
  const float c = 0.7978845608028654f;   // sqrt(2/pi)
  return z * logistic_f(2.0f * c * (z + 0.044715f * z * z * z));
}
// a = exp(log_a) and sqrt(1 - a^2) for log_a <= 0
KAITO_DEV void decay_f(float log_a, float& a, float& mult) {
  const float e = expm1f(log_a);         // a - 1
  a = 1.0f + e;
  mult = sqrtf(-e * (1.0f + a));
}

// ---- gates: gates[blk, t] = u[t, blk] W[blk] + b[blk], f32 ------------------
// u is bf16 and W f32, which three bf16 terms hold to the last bit: three
// products on v_mfma_f32_32x32x16_bf16 have the exact terms of an f32 one. A wave
// keeps 32 columns of its block's W in registers (96 at BW = 128) and walks over
// the tokens, the next 32 rows under way; results leave as whole 128-byte lines.
// 8192 tokens of 16 blocks of 128: 55 us for 134 MB of results (rows wait for the
// stores of the tile before the last), where a cast, a transposing copy and a
// batched f32 GEMM took 162; 32 tokens 5.1 and 13.2. Error against f64, relative
// in the 2-norm: 6.8e-8, of the f32 GEMM 2.0e-7.
typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));
// rows of 36 bytes: no 16-byte alignment
typedef hbf16x8 hbf16x8u __attribute__((aligned(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

constexpr int GATE_WAVES = 4;       // 128 columns per workgroup

// column `wp` (row stride N, from dim 8 h on) in three terms: dims 16 k + 8 h + i
template <int KS>
KAITO_DEV void gate_column(hbf16x8 (&b)[3][KS], const float* wp, const int N) {
#pragma unroll
  for (int k = 0; k < KS; k++)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      __bf16 t[3];
      bf16_terms(wp[(16 * k + i) * N], t);
#pragma unroll
      for (int n = 0; n < 3; n++) b[n][k][i] = t[n];
    }
}

// acc[0] + acc[1]: 32 rows x times 32 columns b, + c0; row r / 4 * 8 + 4 h + r % 4
// of column lane % 32. x: infinities are gone afterwards.
template <int KS>
KAITO_DEV void gate_products(f32x16 (&acc)[2], hbf16x8 (&x)[KS],
                             const hbf16x8 (&b)[3][KS], const float c0) {
  // an infinity is multiplied once: its products with the smaller terms could
  // be of the other sign, or 0 times it
  u16x8 top = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < KS; k++) {
    const u16x8 e = __builtin_bit_cast(u16x8, x[k]) & (unsigned short)0x7fff;
    top = __builtin_elementwise_max(top, e);
  }
  bool wild = false;
#pragma unroll
  for (int i = 0; i < 8; i++) wild |= top[i] >= 0x7f80;
#pragma unroll
  for (int r = 0; r < 16; r++) {    // the largest terms, the rest
    acc[0][r] = c0;
    acc[1][r] = 0.f;
  }
#pragma unroll
  for (int k = 0; k < KS; k++)
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[k], b[0][k], acc[0], 0,
                                                     0, 0);
  if (__any(wild)) {
#pragma unroll
    for (int k = 0; k < KS; k++)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float f = (float)x[k][i];
        if (!(fabsf(f) < INFINITY)) x[k][i] = (__bf16)0.f;
      }
  }
#pragma unroll
  for (int n = 2; n > 0; n--)
#pragma unroll
    for (int k = 0; k < KS; k++)
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[k], b[n][k], acc[1],
                                                       0, 0, 0);
}

template <int KS>                   // bw = 16 KS
__global__ __launch_bounds__(64 * GATE_WAVES, 2) void rglru_gates_kernel(
    float* __restrict__ gates, const short* __restrict__ u,
    const int64_t u_s0, const float* __restrict__ w,
    const float* __restrict__ bias, const int T_total) {
  constexpr int BW = 16 * KS, N = 2 * BW;
  const int lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x, n0 = (blockIdx.y * GATE_WAVES + wave) * 32;
  if (n0 >= N) return;              // no barriers below
  const short* ub = u + blk * BW + 8 * h;
  const int tiles = (T_total + 31) / 32;
  hbf16x8 a[KS];
  auto fetch = [&](const int tile) {
    const short* p = ub + min(tile * 32 + lr, T_total - 1) * u_s0;
#pragma unroll
    for (int k = 0; k < KS; k++)
      a[k] = *reinterpret_cast<const hbf16x8*>(p + 16 * k);
  };
  fetch(min((int)blockIdx.z, tiles - 1));
  hbf16x8 b[3][KS];
  gate_column<KS>(b, w + ((int64_t)blk * BW + 8 * h) * N + n0 + lr, N);
  const float c0 = bias[blk * N + n0 + lr];
  for (int t = blockIdx.z; t < tiles; t += gridDim.z) {
    hbf16x8 x[KS];
#pragma unroll
    for (int k = 0; k < KS; k++) x[k] = a[k];
    fetch(min(t + (int)gridDim.z, tiles - 1));
    f32x16 acc[2];
    gate_products<KS>(acc, x, b, c0);
    float* o = gates + ((int64_t)blk * T_total + t * 32) * N + n0 + lr;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int row = r / 4 * 8 + 4 * h + r % 4;
      if (t * 32 + row < T_total)
        o[row * N] = acc[0][r] + acc[1][r];
    }
  }
}

// ---- the same, and what the recurrence makes of the gates -------------------
// A wave's 32 columns are the recurrence and the input gates of 16 channels, so
// that after one exchange between lanes 16 apart a lane has both gates of 8 rows
// of a channel. It leaves the step S -> a S + b of every row instead of them
// (whole lines of (a, b)), in which a chunk's first row has a = 0 and its initial
// state in b and a padding row is 0, and the product of a segment's steps: two of
// the scan's three passes over 134 MB (8192 tokens, 2048 channels) and their
// exponentials are gone. The rows' own channels come from the operand by way of
// LDS (a wave's own 1 KB: no barrier), what is special about rows a tile ahead.
// Bound by the vector unit (some 90 instructions a row and lane) beside the
// stores. Gates and recurrence, 2048 channels: 8192 tokens 173 -> 132 us (this
// kernel 85), 2048 tokens 84 -> 52, 128 tokens 65 -> 32; 65536 tokens 1328 ->
// 1186. States against f64, relative in the 2-norm: 1.2e-7
// -> 1.1e-7, with slow decay 6.5e-7 -> 4.4e-7. For steps of one token a chunk the
// two launches stay: with 32 rows to a wave this one took 14.5 us, they 8.
struct TermsArgs {
  float2* ab;                       // [T, W]
  float *seg_p, *seg_e;             // [segments, W]
  const short* u;
  int64_t u_s0;
  const float *w, *bias, *rate, *state;
  const int *cu, *slots, *starts, *token_seq;
  int T, W;
};

constexpr int SEG = 64;             // rows of a segment of the scan

// (P, E): S -> P S + E, then S -> p S + e
KAITO_DEV void join(float& P, float& E, const float p, const float e) {
  E = p == 0.f ? e : p * E + e;
  P = p == 0.f ? 0.f : P * p;
}

template <int KS>                   // bw = 16 KS
__global__ __launch_bounds__(64 * GATE_WAVES, 2) void rglru_terms_kernel(
    const TermsArgs args) {
  constexpr int BW = 16 * KS, N = 2 * BW;
  __shared__ short own[GATE_WAVES][32][16 + 2];
  const int lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x, kc = blockIdx.y * GATE_WAVES + wave;
  const int ch = kc * 16;
  const bool second = lr >= 16;     // has the input gates, and later rows
  const int T = args.T, tiles = (T + 31) / 32;
  const int c = blk * BW + ch + (lr & 15);
  const short* ub = args.u + blk * BW + 8 * h;
  hbf16x8 a[KS];
  uint32_t next;                    // rows that are not a step like the others
  auto fetch = [&](const int tile) {
    const int row = min(tile * 32 + lr, T - 1);
    const short* p = ub + row * args.u_s0;
#pragma unroll
    for (int k = 0; k < KS; k++)
      a[k] = *reinterpret_cast<const hbf16x8*>(p + 16 * k);
  };
  auto look = [&](const int tile) {
    const int row = tile * 32 + lr;
    const int of = row < T ? args.token_seq[row] : -1;
    next = (uint32_t)__ballot(of < 0 || args.slots[max(of, 0)] < 0 ||
                              args.cu[max(of, 0)] == row);
  };
  constexpr int PER = SEG / 32;     // tiles of a segment
  fetch(min((int)blockIdx.z * PER, tiles - 1));
  hbf16x8 b[3][KS];
  const int n = ch + (lr & 15) + (second ? BW : 0);
  gate_column<KS>(b, args.w + ((int64_t)blk * BW + 8 * h) * N + n, N);
  const float c0 = args.bias[blk * N + n], rate = args.rate[c];
  look(blockIdx.z * PER);
  for (int seg = blockIdx.z; seg * PER < tiles; seg += gridDim.z) {
    float P = 1.f, E = 0.f;
#pragma unroll 1
    for (int half = 0; half < PER; half++) {
      const int tile = seg * PER + half;
      if (tile >= tiles) break;     // uniform
      hbf16x8 x[KS];
#pragma unroll
      for (int k = 0; k < KS; k++) {
        x[k] = a[k];
        if (k == kc)                // uniform
          *reinterpret_cast<hbf16x8u*>(&own[wave][lr][8 * h]) = x[k];
      }
      const uint32_t special = next;
      const int then =
          half + 1 < PER ? tile + 1 : (seg + (int)gridDim.z) * PER;
      fetch(min(then, tiles - 1));
      f32x16 acc[2];
      gate_products<KS>(acc, x, b, c0);
      look(then);
      // this lane's rows: 8 (j / 4) + j % 4 on from here
      const int r0 = (second ? 16 : 0) + 4 * h, t0 = tile * 32 + r0;
      float A[8], B[8];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        // lanes of recurrence gates keep row j and get its input gate, the
        // others give that and get the recurrence gate of row j + 8
        const float lo = acc[0][j] + acc[1][j];
        const float hi = acc[0][j + 8] + acc[1][j + 8];
        const float got = __shfl_xor(second ? lo : hi, 16, 64);
        const float rg = second ? got : lo, ig = second ? hi : got;
        float mult;
        decay_f(-logistic_f(rg) * rate, A[j], mult);
        B[j] = mult * logistic_f(ig) *
               bf16_to_f32(own[wave][r0 + j / 4 * 8 + j % 4][lr & 15]);
      }
      float2* to = args.ab + (int64_t)t0 * args.W + c;
      float p[2], e[2];             // of rows j < 4 and the other four
      if (special == 0) {           // uniform; and no row is past the last
#pragma unroll
        for (int j = 0; j < 8; j++) {
          to[(j / 4 * 8 + j % 4) * args.W] = {A[j], B[j]};
          p[j / 4] = j % 4 == 0 ? A[j] : p[j / 4] * A[j];
          e[j / 4] = j % 4 == 0 ? B[j] : A[j] * e[j / 4] + B[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const int r = j / 4 * 8 + j % 4, t = t0 + r;
          const bool cut = special >> (r0 + r) & 1;
          if (cut) {
            const int q = t < T ? args.token_seq[t] : -1;
            const int slot = q >= 0 ? args.slots[q] : -1;
            const float S0 = slot >= 0 && args.starts[q] > 0
                ? args.state[(int64_t)slot * args.W + c] : 0.f;
            B[j] = slot >= 0 ? A[j] * S0 + B[j] : 0.f;
            A[j] = 0.f;
          }
          if (t < T) to[r * args.W] = {A[j], B[j]};
          // nothing before such a row can reach past it
          p[j / 4] = j % 4 == 0 || cut ? A[j] : p[j / 4] * A[j];
          e[j / 4] = j % 4 == 0 || cut ? B[j] : A[j] * e[j / 4] + B[j];
        }
      }
      // groups of four rows in the order (half lane, j / 4, h)
      float tp = 1.f, te = 0.f;
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const float op = __shfl_xor(p[g], 32, 64);
        const float oe = __shfl_xor(e[g], 32, 64);
        join(tp, te, h ? op : p[g], h ? oe : e[g]);
        join(tp, te, h ? p[g] : op, h ? e[g] : oe);
      }
      const float op = __shfl_xor(tp, 16, 64);
      const float oe = __shfl_xor(te, 16, 64);
      join(P, E, second ? op : tp, second ? oe : te);
      join(P, E, second ? tp : op, second ? te : oe);
    }
    if (h == 0 && !second) {
      args.seg_p[(int64_t)seg * args.W + c] = P;
      args.seg_e[(int64_t)seg * args.W + c] = E;
    }
  }
}

template <typename T>
__global__ void rglru_scan_kernel(
    T* __restrict__ out, const T* __restrict__ u, const int64_t u_s0,
    const float* __restrict__ gates,        // [NB, T, 2*bw]
    const T* __restrict__ y, const int64_t y_s0,
    const float* __restrict__ decay_rate, float* __restrict__ state,
    const int* __restrict__ cu, const int* __restrict__ slots,
    const int* __restrict__ starts, const int T_total, const int W,
    const int bw) {
  const int b = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= W) return;
  const int slot = slots[b];
  const int r0 = cu[b], r1 = cu[b + 1];
  if (slot < 0 || r1 <= r0) return;
  const int blk = c / bw, cc = c % bw;
  const float rate = decay_rate[c];
  float S = starts[b] > 0 ? state[(int64_t)slot * W + c] : 0.0f;
  const float* gp = gates + ((int64_t)blk * T_total) * (2 * bw) + cc;
#pragma unroll 4
  for (int t = r0; t < r1; t++) {
    const float rg = sigmoid_f(gp[(int64_t)t * (2 * bw)]);
    const float ig = sigmoid_f(gp[(int64_t)t * (2 * bw) + bw]);
    float a, mult;
    decay_f(-rg * rate, a, mult);
    const float uv = act_ld(u + (int64_t)t * u_s0 + c);
    S = a * S + mult * ig * uv;
    act_st(out + (int64_t)t * W + c,
           S * gelu_tanh_f(act_ld(y + (int64_t)t * y_s0 + c)));
  }
  state[(int64_t)slot * W + c] = S;
}

// ---- segment-parallel scan for prompt-sized steps --------------------------
// The recurrence is linear, S_t = a_t S_(t-1) + b_t, so the rows of a step
// are cut into fixed segments of SEG rows (chunk borders may fall anywhere
// inside one) and scanned in three launches:
//   1. per (segment, channel): walk the rows from a zero carry with the
//      running product P of a's; a row that starts a chunk replaces the
//      running state by that chunk's initial state and sets P = 0 (nothing
//      before it can reach past it). Emit (P, E = state at segment end).
//   2. per (segment, channel): fold the (P, E) before it into the true
//      carry, back to where the product is 0 (a chunk's start, or decayed
//      away), walk again, write the outputs, and park the state at every
//      chunk's last row;
//   3. the parked states go to the slots, whose old ones 2 still reads.
// The fold costs every segment a walk over those before it, unless they have
// decayed away. Beyond FOLD_FROM segments that is more than one walk over all
// of them in a launch of its own (2048 channels: 131072 rows without decay 3090
// us and 1567, with fast decay 1501 and 1569; 65536 rows in walks 1128 and 762,
// 65600 with the launch 801 and 798).
// Rows are loaded 8 ahead of the walk. Measured on one MI355X, 4 prompts of
// 2048 tokens, 2048 channels: 230 us with the fold and the last segments'
// walk in launches of their own, one row's loads at a time, 126 now.
constexpr int AHEAD = 8;
constexpr int FOLD_FROM = 1024;

// the true carry into segment s: (P, E) of those before it, back to where the
// product is 0
KAITO_DEV float fold_carry(const float* __restrict__ seg_p,
                           const float* __restrict__ seg_e, const int s,
                           const int W, const int c) {
  float S = 0.0f, P = 1.0f;
  for (int e = s - 1; e >= 0 && P != 0.0f; e -= AHEAD) {
    float p[AHEAD], v[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      p[i] = seg_p[(int64_t)max(e - i, 0) * W + c];
      v[i] = seg_e[(int64_t)max(e - i, 0) * W + c];
    }
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      if (e - i < 0 || P == 0.0f) continue;
      S += P * v[i];
      P *= p[i];
    }
  }
  return S;
}

// PHASE 1, 2: see above. 3: 2 with the carry already in seg_e
template <typename T, int PHASE>
__global__ __launch_bounds__(256)
void rglru_segment_kernel(
    T* __restrict__ out, const T* __restrict__ u, const int64_t u_s0,
    const float* __restrict__ gates, const T* __restrict__ y,
    const int64_t y_s0, const float* __restrict__ decay_rate,
    const float* __restrict__ state, float* __restrict__ seg_p,
    float* __restrict__ seg_e, float* __restrict__ last,    // [B, W]
    const int* __restrict__ cu, const int* __restrict__ slots,
    const int* __restrict__ starts, const int* __restrict__ token_seq,
    const int T_total, const int W, const int bw) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= W) return;
  const int blk = c / bw, cc = c % bw;
  const float rate = decay_rate[c];
  const float* gp = gates + ((int64_t)blk * T_total) * (2 * bw) + cc;
  const int t0 = s * SEG, t1 = min(T_total, t0 + SEG);
  float S = 0.0f, P = 1.0f;
  if (PHASE == 3) S = seg_e[(int64_t)s * W + c];
  if (PHASE == 2) S = fold_carry(seg_p, seg_e, s, W, c);
  int seq = -1, slot = -1, first = -1, final = -1;
  for (int tb = t0; tb < t1; tb += AHEAD) {
    float rg[AHEAD], ig[AHEAD], uv[AHEAD], yv[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int64_t t = min(tb + i, t1 - 1);
      rg[i] = gp[t * (2 * bw)];
      ig[i] = gp[t * (2 * bw) + bw];
      uv[i] = act_ld(u + t * u_s0 + c);
      if (PHASE > 1) yv[i] = act_ld(y + t * y_s0 + c);
    }
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int t = tb + i;
      if (t >= t1) break;
      const int b = token_seq[t];
      if (b != seq || t == t0) {                       // uniform
        seq = b;
        slot = b >= 0 ? slots[b] : -1;
        first = b >= 0 ? cu[b] : -1;
        final = b >= 0 ? cu[b + 1] - 1 : -1;
      }
      if (slot < 0) { S = 0.0f; P = 0.0f; continue; }  // padding row
      if (t == first) {                                // chunk starts here
        S = starts[b] > 0 ? state[(int64_t)slot * W + c] : 0.0f;
        P = 0.0f;
      }
      float a, mult;
      decay_f(-logistic_f(rg[i]) * rate, a, mult);
      S = a * S + mult * logistic_f(ig[i]) * uv[i];
      if (PHASE == 1) {
        P *= a;
      } else {
        act_st(out + (int64_t)t * W + c, S * gelu_f(yv[i]));
        if (t == final) last[(int64_t)b * W + c] = S;
      }
    }
  }
  if (PHASE == 1) {
    seg_p[(int64_t)s * W + c] = P;
    seg_e[(int64_t)s * W + c] = S;
  }
}

// phase 2 of the scan (3 with CARRIED) over the steps of rglru_terms
template <bool CARRIED>
__global__ __launch_bounds__(256) void rglru_apply_kernel(
    short* __restrict__ out, const float2* __restrict__ ab,
    const short* __restrict__ y, const int64_t y_s0,
    const float* __restrict__ seg_p, const float* __restrict__ seg_e,
    float* __restrict__ last, const int* __restrict__ cu,
    const int* __restrict__ slots, const int* __restrict__ token_seq,
    const int T_total, const int W) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= W) return;
  const int t0 = s * SEG, t1 = min(T_total, t0 + SEG);
  float S = CARRIED ? seg_e[(int64_t)s * W + c]
                    : fold_carry(seg_p, seg_e, s, W, c);
  int seq = -1, slot = -1, first = -1, final = -1;
  for (int tb = t0; tb < t1; tb += AHEAD) {
    float2 v[AHEAD];
    float yv[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int64_t t = min(tb + i, t1 - 1);
      v[i] = ab[t * W + c];
      yv[i] = bf16_to_f32(y[t * y_s0 + c]);
    }
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const int t = tb + i;
      if (t >= t1) break;
      const int b = token_seq[t];
      if (b != seq || t == t0) {                       // uniform
        seq = b;
        slot = b >= 0 ? slots[b] : -1;
        first = b >= 0 ? cu[b] : -1;
        final = b >= 0 ? cu[b + 1] - 1 : -1;
      }
      S = t == first ? v[i].y : v[i].x * S + v[i].y;
      if (slot < 0) continue;                          // padding row
      out[(int64_t)t * W + c] = f32_to_bf16(S * gelu_f(yv[i]));
      if (t == final) last[(int64_t)b * W + c] = S;
    }
  }
}

// seg_e[s]: the state at segment s's end from a zero carry -> its carry
__global__ __launch_bounds__(64) void rglru_fold_kernel(
    const float* __restrict__ seg_p, float* __restrict__ seg_e, const int nseg,
    const int W) {
  const int c = blockIdx.x * 64 + threadIdx.x;
  if (c >= W) return;
  constexpr int N = 32;             // a batch, and the next one under way
  float p[2][N], v[2][N], S = 0.0f;
  auto fetch = [&](const int s, const int b) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      const int64_t at = (int64_t)min(s + i, nseg - 1) * W + c;
      p[b][i] = seg_p[at];
      v[b][i] = seg_e[at];
    }
  };
  auto fold = [&](const int s, const int b) {
    fetch(s + N, b ^ 1);            // ahead of the stores, which are to other rows
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (s + i < nseg) seg_e[(int64_t)(s + i) * W + c] = S;
      // a product of 0: a chunk starts here
      S = p[b][i] == 0.0f ? v[b][i] : p[b][i] * S + v[b][i];
    }
  };
  fetch(0, 0);
  for (int s = 0; s < nseg; s += 2 * N) {
    fold(s, 0);
    fold(s + N, 1);
  }
}

__global__ void rglru_store_kernel(float* __restrict__ state,
                                   const float* __restrict__ last,
                                   const int* __restrict__ cu,
                                   const int* __restrict__ slots,
                                   const int W) {
  const int b = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c < W && slots[b] >= 0 && cu[b + 1] > cu[b])
    state[(int64_t)slots[b] * W + c] = last[(int64_t)b * W + c];
}

template <typename T>
void run_rglru_segments(hipStream_t stream, at::Tensor& out,
                        const at::Tensor& u, const at::Tensor& gates,
                        const at::Tensor& y, const at::Tensor& decay_rate,
                        at::Tensor& state, const at::Tensor& cu,
                        const at::Tensor& slots, const at::Tensor& starts,
                        const at::Tensor& token_seq, int cblocks, int threads,
                        int bw) {
  const int T_total = u.size(0), W = u.size(1), B = slots.size(0);
  const int nseg = (T_total + SEG - 1) / SEG;
  at::Tensor seg_p = at::empty({nseg, W}, state.options());
  at::Tensor seg_e = at::empty({nseg, W}, state.options());
  at::Tensor last = at::empty({B, W}, state.options());
#define KAITO_RGLRU_SEG(PHASE_)                                              \
  hipLaunchKernelGGL((rglru_segment_kernel<T, PHASE_>),                      \
      dim3(nseg, cblocks), dim3(threads), 0, stream, (T*)out.data_ptr(),     \
      (const T*)u.data_ptr(), u.stride(0), gates.data_ptr<float>(),          \
      (const T*)y.data_ptr(), y.stride(0), decay_rate.data_ptr<float>(),     \
      state.data_ptr<float>(), seg_p.data_ptr<float>(),                      \
      seg_e.data_ptr<float>(), last.data_ptr<float>(), cu.data_ptr<int>(),   \
      slots.data_ptr<int>(), starts.data_ptr<int>(),                         \
      token_seq.data_ptr<int>(), T_total, W, bw)
  KAITO_RGLRU_SEG(1);
  if (nseg <= FOLD_FROM) {
    KAITO_RGLRU_SEG(2);
  } else {
    hipLaunchKernelGGL(rglru_fold_kernel, dim3((W + 63) / 64), dim3(64), 0,
        stream, seg_p.data_ptr<float>(), seg_e.data_ptr<float>(), nseg, W);
    KAITO_RGLRU_SEG(3);
  }
#undef KAITO_RGLRU_SEG
  hipLaunchKernelGGL(rglru_store_kernel, dim3(B, cblocks), dim3(threads), 0,
      stream, state.data_ptr<float>(), last.data_ptr<float>(),
      cu.data_ptr<int>(), slots.data_ptr<int>(), W);
}

}  // namespace

void rglru_gates(at::Tensor gates, at::Tensor u, at::Tensor w,
                 at::Tensor bias) {
  TORCH_CHECK(u.is_cuda() && u.dim() == 2 && u.dtype() == at::kBFloat16 &&
              u.stride(1) == 1 && u.stride(0) % 8 == 0 &&
              (uintptr_t)u.data_ptr() % 16 == 0);
  KAITO_CHECK_F32(gates); KAITO_CHECK_F32(w); KAITO_CHECK_F32(bias);
  TORCH_CHECK(w.dim() == 3 && w.size(2) == 2 * w.size(1) &&
              gates.dim() == 3);
  const int64_t NB = w.size(0), bw = w.size(1), T = u.size(0);
  TORCH_CHECK(u.size(1) == NB * bw && bias.numel() == NB * 2 * bw &&
              gates.size(0) == NB && gates.size(1) == T &&
              gates.size(2) == 2 * bw);
  TORCH_CHECK(bw == 64 || bw == 128, "blocks of 64 or 128 channels");
  TORCH_CHECK(T < (1ll << 31) - 32);
  if (T == 0 || NB == 0) return;
  const int cols = (int)((2 * bw + 32 * GATE_WAVES - 1) / (32 * GATE_WAVES));
  // two workgroups per CU: each reads and splits its columns of W first
  const int64_t tiles = (T + 31) / 32;
  const int64_t z = std::max<int64_t>(
      1, std::min<int64_t>(tiles, std::max<int64_t>(512 / (NB * cols), 1)));
  const dim3 grid(NB, cols, z), block(64 * GATE_WAVES);
  auto stream = at::hip::getCurrentHIPStream();
#define KAITO_GATES(KS_)                                                     \
  hipLaunchKernelGGL((rglru_gates_kernel<KS_>), grid, block, 0, stream,      \
      gates.data_ptr<float>(), (const short*)u.data_ptr(), u.stride(0),      \
      w.data_ptr<float>(), bias.data_ptr<float>(), (int)T)
  if (bw == 64) KAITO_GATES(4); else KAITO_GATES(8);
#undef KAITO_GATES
}

// rglru_gates and rglru_scan of bf16 rows, for steps of prompts
void rglru_rows(at::Tensor out, at::Tensor u, at::Tensor w, at::Tensor bias,
                at::Tensor y, at::Tensor decay_rate, at::Tensor state,
                at::Tensor cu_seqlens, at::Tensor state_slots,
                at::Tensor seq_starts, at::Tensor token_seq) {
  for (const auto& t : {u, y})
    TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.dtype() == at::kBFloat16 &&
                t.stride(1) == 1);
  TORCH_CHECK(u.stride(0) % 8 == 0 && (uintptr_t)u.data_ptr() % 16 == 0 &&
              y.sizes() == u.sizes() && out.sizes() == u.sizes() &&
              out.is_contiguous() && out.dtype() == at::kBFloat16);
  KAITO_CHECK_F32(w); KAITO_CHECK_F32(bias); KAITO_CHECK_F32(decay_rate);
  KAITO_CHECK_F32(state);
  KAITO_CHECK_I32(cu_seqlens); KAITO_CHECK_I32(state_slots);
  KAITO_CHECK_I32(seq_starts); KAITO_CHECK_I32(token_seq);
  const int64_t T = u.size(0), W = u.size(1), B = state_slots.size(0);
  TORCH_CHECK(w.dim() == 3 && w.size(2) == 2 * w.size(1) &&
              w.size(0) * w.size(1) == W && bias.numel() == 2 * W &&
              decay_rate.numel() == W && state.dim() == 2 &&
              state.size(1) == W && cu_seqlens.size(0) == B + 1 &&
              seq_starts.size(0) == B && token_seq.size(0) == T);
  const int64_t NB = w.size(0), bw = w.size(1);
  TORCH_CHECK(bw == 64 || bw == 128, "blocks of 64 or 128 channels");
  TORCH_CHECK(T < (1ll << 31) - 64);
  if (T == 0 || B == 0 || W == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const int nseg = (int)((T + SEG - 1) / SEG);
  const int cols = (int)(bw / (16 * GATE_WAVES));
  // two workgroups per CU, as for the gates alone
  const int z = (int)std::max<int64_t>(
      1, std::min<int64_t>(nseg, 512 / (NB * cols)));
  at::Tensor ab = at::empty({T, W, 2}, state.options());
  at::Tensor seg_p = at::empty({nseg, W}, state.options());
  at::Tensor seg_e = at::empty({nseg, W}, state.options());
  at::Tensor last = at::empty({B, W}, state.options());
  const TermsArgs a = {
      (float2*)ab.data_ptr(), seg_p.data_ptr<float>(), seg_e.data_ptr<float>(),
      (const short*)u.data_ptr(), u.stride(0), w.data_ptr<float>(),
      bias.data_ptr<float>(), decay_rate.data_ptr<float>(),
      state.data_ptr<float>(), cu_seqlens.data_ptr<int>(),
      state_slots.data_ptr<int>(), seq_starts.data_ptr<int>(),
      token_seq.data_ptr<int>(), (int)T, (int)W};
  const dim3 grid(NB, cols, z), block(64 * GATE_WAVES);
  hipLaunchKernelGGL(bw == 64 ? &rglru_terms_kernel<4> : &rglru_terms_kernel<8>,
      grid, block, 0, stream, a);
  const int threads = W >= 256 ? 256 : 64;
  const int cblocks = (int)((W + threads - 1) / threads);
  auto apply = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nseg, cblocks), dim3(threads), 0, stream,
        (short*)out.data_ptr(), a.ab, (const short*)y.data_ptr(), y.stride(0),
        a.seg_p, a.seg_e, last.data_ptr<float>(),
        a.cu, a.slots, a.token_seq, a.T, a.W);
  };
  if (nseg <= FOLD_FROM) {
    apply(&rglru_apply_kernel<false>);
  } else {
    hipLaunchKernelGGL(rglru_fold_kernel, dim3((W + 63) / 64), dim3(64), 0,
        stream, a.seg_p, a.seg_e, nseg, (int)W);
    apply(&rglru_apply_kernel<true>);
  }
  hipLaunchKernelGGL(rglru_store_kernel, dim3(B, cblocks), dim3(threads), 0,
      stream, state.data_ptr<float>(), last.data_ptr<float>(), a.cu, a.slots, (int)W);
}

void rglru_scan(at::Tensor out, at::Tensor u, at::Tensor gates, at::Tensor y,
                at::Tensor decay_rate, at::Tensor state,
                at::Tensor cu_seqlens, at::Tensor state_slots,
                at::Tensor seq_starts, at::Tensor token_seq) {
  TORCH_CHECK(u.is_cuda() && u.dim() == 2 && y.dim() == 2 &&
              u.stride(1) == 1 && y.stride(1) == 1 && u.dtype() == y.dtype());
  const int T = u.size(0), W = u.size(1);
  TORCH_CHECK(y.size(0) == T && y.size(1) == W);
  TORCH_CHECK(out.is_contiguous() && out.dtype() == u.dtype() &&
              out.size(0) == T && out.size(1) == W);
  KAITO_CHECK_F32(gates); KAITO_CHECK_F32(decay_rate); KAITO_CHECK_F32(state);
  TORCH_CHECK(gates.dim() == 3 && gates.size(1) == T);
  const int NB = gates.size(0);
  TORCH_CHECK(NB > 0 && W % NB == 0 && gates.size(2) == 2 * (W / NB));
  TORCH_CHECK(decay_rate.numel() == W && state.dim() == 2 &&
              state.size(1) == W);
  KAITO_CHECK_I32(cu_seqlens); KAITO_CHECK_I32(state_slots);
  KAITO_CHECK_I32(seq_starts);
  const int B = state_slots.size(0);
  TORCH_CHECK(cu_seqlens.size(0) == B + 1 && seq_starts.size(0) == B);
  if (T == 0 || B == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  const int threads = W >= 256 ? 256 : 64;
  const int cblocks = (W + threads - 1) / threads;
  if (token_seq.numel() > 0 && T >= 4 * B && T >= 2 * SEG) {
    // prompt-sized step: segment-parallel scan
    KAITO_CHECK_I32(token_seq);
    TORCH_CHECK(token_seq.size(0) == T);
    KAITO_DISPATCH_ACT(u, {
      run_rglru_segments<act_t>(stream, out, u, gates, y, decay_rate, state,
                                cu_seqlens, state_slots, seq_starts,
                                token_seq, cblocks, threads, W / NB);
    });
    return;
  }
  KAITO_DISPATCH_ACT(u, {
    hipLaunchKernelGGL((rglru_scan_kernel<act_t>),
        dim3(B, (W + threads - 1) / threads), dim3(threads), 0, stream,
        (act_t*)out.data_ptr(), (const act_t*)u.data_ptr(), u.stride(0),
        gates.data_ptr<float>(), (const act_t*)y.data_ptr(), y.stride(0),
        decay_rate.data_ptr<float>(), state.data_ptr<float>(),
        cu_seqlens.data_ptr<int>(), state_slots.data_ptr<int>(),
        seq_starts.data_ptr<int>(), T, W, W / NB);
  });
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("rglru_gates(Tensor(a!) gates, Tensor u, Tensor w, Tensor bias) -> ()");
  m.def("rglru_rows(Tensor(a!) out, Tensor u, Tensor w, Tensor bias, Tensor y, Tensor decay_rate, Tensor(b!) state, Tensor cu_seqlens, Tensor state_slots, Tensor seq_starts, Tensor token_seq) -> ()");
  m.def("rglru_scan(Tensor(a!) out, Tensor u, Tensor gates, Tensor y, Tensor decay_rate, Tensor(b!) state, Tensor cu_seqlens, Tensor state_slots, Tensor seq_starts, Tensor token_seq) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("rglru_gates", &kaito::rglru_gates);
  m.impl("rglru_rows", &kaito::rglru_rows);
  m.impl("rglru_scan", &kaito::rglru_scan);
}
