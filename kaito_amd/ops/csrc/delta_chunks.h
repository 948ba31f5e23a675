// Gated delta rule, sixteen tokens at a time on the f32 matrix instruction.
//
// With S0 the state before a chunk, d_i the decays, R_ij = d_(j+1) .. d_i and
// g_i = d_0 .. d_i, the tokens' writes u_i = beta_i (v_i - S^T k_i) solve
//     (I + A) U = diag(beta) (V - diag(g) K S0),  A_ij = beta_i R_ij k_i.k_j
// below the diagonal, and
//     O = diag(g) Q S0 + (R_ij q_i.k_j)_(j <= i) U
//     S = g_15 S0 + sum over i of R_15,i k_i u_i^T.
// R is multiplied up and never divided out, so that no decay is too small; row
// j of (I + A)^-1 is what a write leaves for later tokens, products of
// contractions, so no entry is large.
//
// delta_chunk_prep_kernel: one wave per (chunk, qk head) normalises q and k,
// forms both 16 x 16 products, and per head the inverse (forward substitution,
// a lane per column), decays and read-out matrix.
// delta_chunk_kernel: NW waves per (sequence, head, 16 columns of S), each with
// every NW-th row tile of S. A lane's accumulators of a row tile are at once
// the operands of the next chunk's products with S (the dims of K are taken in
// that order), and the results of one product those of the next: S, U and the
// right-hand side never change lanes. The next chunk's operands are under way
// while one is multiplied.
//
// S and its products are f32. What is 16 x 16 is f64, from K K^T to U and the
// read-out: an error there is every dim's at once, and the loop has no such sums.
// All in f32, states came out up to 1.25 times as far from 64 bits as the loop's
// and read-outs 1.19 times (f32 inputs, keys of one direction, cosine 0.9, decays
// from 0.5 to 0.9; both 0.93 to 1.07 elsewhere). Now states 0.78 to 1.01 times
// (1.07 with those keys at 0.5), read-outs 0.72 to 0.95 (1.04). It costs a tenth:
// 4 prompts of 2048 tokens, 294 -> 328 us.
//
// The token-by-token loop is bound by its chain of sums, 830 cycles a token;
// here it is instruction issue beside the matrix unit. 64-bit addresses and
// clamps for every load cost a fifth more than buffers that end with their
// sequence. Times beside the loop's: run_chunks.
#pragma once
#include "mix_common.h"

namespace kaito {
namespace delta_chunks {

constexpr int C = 16;               // tokens of a chunk
// floats per (chunk, head): inverse times beta, read-out matrix, g, R_15
constexpr int REC = 2 * C * C + 2 * C;

typedef double f64x4 __attribute__((ext_vector_type(4)));

KAITO_DEV f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Sequence b's chunks are numbered from cu[b] / C + b: disjoint, in order and
// below T / C + B, without a scan over the lengths.
template <typename T, int NJ>       // dim = 16 NJ
__global__ __launch_bounds__(64) void delta_chunk_prep_kernel(
    float* __restrict__ qn, float* __restrict__ kn,       // [T, G, D]
    float* __restrict__ rec,                               // [.., H, REC]
    const T* __restrict__ q, const int64_t q_s0, const int64_t q_s1,
    const T* __restrict__ k, const int64_t k_s0, const int64_t k_s1,
    const T* __restrict__ a, const int64_t a_s0,
    const T* __restrict__ b, const int64_t b_s0,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const int* __restrict__ cu, const int* __restrict__ slots, const int B,
    const int G, const int H, const float qk_eps) {
  constexpr int D = 16 * NJ, P = C + 4;
  __shared__ __attribute__((aligned(16))) float qk[C][P];
  __shared__ double kk[C][P];
  __shared__ __attribute__((aligned(16))) double A[4][C][C + 2];
  __shared__ __attribute__((aligned(16))) float dl[4][C], bl[4][C];
  const int id = blockIdx.x, g = blockIdx.y;
  const int lane = threadIdx.x, lo = lane & 15, hi = lane >> 4;
  int seq = -1;
  for (int s = 0; s < B; s += 64)
    seq += __builtin_popcountll(__ballot(
        s + lane < B && cu[min(s + lane, B - 1)] / C + s + lane <= id));
  if (seq < 0 || slots[seq] < 0) return;
  const int r0 = cu[seq], r1 = cu[seq + 1];
  const int t0 = r0 + (id - r0 / C - seq) * C;
  if (t0 >= r1) return;
  const int n = min(C, r1 - t0);

  float4_t kv[NJ], qv[NJ];
  const int64_t t = t0 + min(lo, n - 1);
  float4_t q2{0.f, 0.f, 0.f, 0.f}, k2 = q2;
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    kv[j] = act_ld4(k + t * k_s0 + g * k_s1 + 16 * j + 4 * hi);
    qv[j] = act_ld4(q + t * q_s0 + g * q_s1 + 16 * j + 4 * hi);
  }
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      q2[e] += qv[j][e] * qv[j][e];
      k2[e] += kv[j][e] * kv[j][e];
    }
  float sq = (q2[0] + q2[1]) + (q2[2] + q2[3]);
  float sk = (k2[0] + k2[1]) + (k2[2] + k2[3]);
#pragma unroll
  for (int off = 16; off < 64; off <<= 1) {
    sq += __shfl_xor(sq, off, 64);
    sk += __shfl_xor(sk, off, 64);
  }
  const float iq = (1.0f / sqrtf(sq + qk_eps)) * (1.0f / sqrtf((float)D));
  const float ik = 1.0f / sqrtf(sk + qk_eps);
  // k.k of the unit vectors, as the state has them; q.k of the rows, rounded last.
  // Sums in trees of one instruction's, for their rounding.
  const f32x4 zero{0.f, 0.f, 0.f, 0.f};
  f32x4 cq[NJ];
  f64x4 ck{0., 0., 0., 0.};
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int64_t at = (t * G + g) * D + 16 * j + 4 * hi;
    const float4_t ku = kv[j] * ik;
    if (lo < n) {
      *reinterpret_cast<float4_t*>(kn + at) = ku;
      *reinterpret_cast<float4_t*>(qn + at) = qv[j] * iq;
    }
    f32x4 pq[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      ck = __builtin_amdgcn_mfma_f64_16x16x4f64(ku[e], ku[e], ck, 0, 0, 0);
      pq[e] = mfma4(qv[j][e], kv[j][e], zero);
    }
    cq[j] = (pq[0] + pq[1]) + (pq[2] + pq[3]);
  }
#pragma unroll
  for (int w = 1; w < NJ; w *= 2)
#pragma unroll
    for (int j = 0; j < NJ; j += 2 * w) cq[j] += cq[j + w];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    kk[4 * r + hi][lo] = ck[r];
    // a row whose square is beyond f32 has a unit vector of 0
    const float ir = __shfl(iq, 4 * hi + r, 64);
    qk[4 * hi + r][lo] = ir == 0.f || ik == 0.f ? 0.f : cq[0][r] * ir * ik;
  }

  // four heads at a time, a quarter wave each
  const int per = H / G;
  for (int hb = 0; hb < per; hb += 4) {
    const bool live = hb + hi < per;
    const int h = g * per + min(hb + hi, per - 1);
    const float av = act_ld(a + t * a_s0 + h), bv = act_ld(b + t * b_s0 + h);
    dl[hi][lo] = lo < n
        ? expf(-expf(a_log[h]) * softplus_f(av + dt_bias[h])) : 1.0f;
    const float beta = lo < n ? sigmoid_f(bv) : 0.0f;
    bl[hi][lo] = beta;
    __syncthreads();
    float* out = rec + ((int64_t)id * H + h) * REC;
    // in 64 bits: an error here is every dim's at once, where those of S differ
    // from row to row
    double R = 1., gam = 1.;
#pragma unroll
    for (int i = 0; i < C; i++) {
      const double d = dl[hi][i];
      if (i > lo) R *= d;
      if (i <= lo) gam *= d;
      A[hi][i][lo] = i > lo ? bl[hi][i] * (R * kk[i][lo]) : 0.;
      const double ro = i >= lo ? R * qk[i][lo] : 0.;
      if (live) out[C * C + i * C + lo] = (float)ro;
    }
    if (live) {
      out[2 * C * C + lo] = (float)gam;
      out[2 * C * C + C + lo] = (float)R;
    }
    __syncthreads();
    double x[C];                    // column lo of the inverse
#pragma unroll
    for (int i = 0; i < C; i++) {
      double s = i == lo ? 1. : 0.;
#pragma unroll
      for (int m = 0; m < i; m++) s -= A[hi][i][m] * x[m];
      // what stands above the diagonal is 0 also where A or beta is not finite
      x[i] = i < lo ? 0. : s;
      if (live) out[i * C + lo] = i < lo ? 0.f : (float)(x[i] * beta);
    }
    __syncthreads();
  }
}

KAITO_DEV __amdgpu_buffer_rsrc_t rows(const void* p, const int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x27000);
}
KAITO_DEV float4_t load4(__amdgpu_buffer_rsrc_t r, const int at) {
  return __builtin_bit_cast(
      float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
}
template <typename T>
KAITO_DEV T load1(__amdgpu_buffer_rsrc_t r, const int at) {
  if constexpr (sizeof(T) == 4) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
  } else {
    return T{(short)__builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0)};
  }
}

// Rows of a sequence are read and written as buffers that end with it: rows past
// its last are 0, and not written.
template <typename T, int NJ, int NW>
__global__ __launch_bounds__(64 * NW, 2) void delta_chunk_kernel(
    float* __restrict__ o,                                 // [T, H, V]
    const float* __restrict__ qn, const float* __restrict__ kn,
    const float* __restrict__ rec, const T* __restrict__ v,
    const int64_t v_s0, const int64_t v_s1,
    float* __restrict__ state,                             // [slots, H, D, V]
    const int* __restrict__ cu, const int* __restrict__ slots,
    const int* __restrict__ starts, const int G, const int H, const int V) {
  constexpr int D = 16 * NJ, J = NJ / NW;
  __shared__ f32x4 meet[2][NW][2][64];
  const int b = blockIdx.x, h = blockIdx.y;
  const int slot = slots[b];
  const int r0 = cu[b], r1 = cu[b + 1];
  if (slot < 0 || r1 <= r0) return;
  const int g = h / (H / G);
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int v0 = blockIdx.z * 16, d0 = wave * J * 16;

  f32x4 S[J];                       // rows d0 + 16 j + 4 hi + e, column lo
  float* sp = state + (((int64_t)slot * H + h) * D + d0 + 4 * hi) * V + v0 + lo;
  const bool carried = starts[b] > 0;
#pragma unroll
  for (int j = 0; j < J; j++)
#pragma unroll
    for (int e = 0; e < 4; e++)
      S[j][e] = carried ? sp[(int64_t)(16 * j + e) * V] : 0.f;

  struct Operands {
    float4_t k[J], q[J];            // token lo, dims 16 j + 4 hi ..
    float4_t kt[J];                 // dim 16 j + lo, tokens 4 hi ..
    float4_t inv, ro, gam, rest;
    T v[4];
  };
  const int n = r1 - r0, nc = (n + C - 1) / C;
  const int krow = G * D * 4, vrow = (int)v_s0 * (int)sizeof(T);
  const int orow = H * V * 4;
  const int64_t k0 = ((int64_t)r0 * G + g) * D;
  const auto kb = rows(kn + k0, (n - 1) * krow + D * 4);
  const auto qb = rows(qn + k0, (n - 1) * krow + D * 4);
  const auto vb = rows(v + r0 * v_s0 + h * v_s1,
                       (n - 1) * vrow + V * (int)sizeof(T));
  const auto ob = rows(o + ((int64_t)r0 * H + h) * V,
                       (n - 1) * orow + V * 4);
  const float* rp = rec + ((int64_t)(r0 / C + b) * H + h) * REC;
  // offsets in a chunk
  const int kat = lo * krow + (d0 + 4 * hi) * 4;
  const int tat = 4 * hi * krow + (d0 + lo) * 4;
  const int vat = 4 * hi * vrow + (v0 + lo) * (int)sizeof(T);
  const int oat = 4 * hi * orow + (v0 + lo) * 4;
  // the f64 product's row 4 e + hi is the other's 4 hi + e
  const int irow = lo % 4 * 4 + lo / 4;
  auto fetch = [&](Operands& x, const int c) {
    const float* p = rp + (int64_t)c * H * REC;
    const int kc = kat + c * C * krow, tc = tat + c * C * krow;
    const int vc = vat + c * C * vrow;
#pragma unroll
    for (int j = 0; j < J; j++) {
      x.k[j] = load4(kb, kc + j * 64);
      x.q[j] = load4(qb, kc + j * 64);
    }
    x.inv = *reinterpret_cast<const float4_t*>(p + irow * C + 4 * hi);
    x.ro = *reinterpret_cast<const float4_t*>(p + C * C + irow * C + 4 * hi);
    x.gam = *reinterpret_cast<const float4_t*>(p + 2 * C * C + 4 * hi);
    x.rest = *reinterpret_cast<const float4_t*>(p + 2 * C * C + C + 4 * hi);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      x.v[e] = load1<T>(vb, vc + e * vrow);
#pragma unroll
      for (int j = 0; j < J; j++)
        x.kt[j][e] = load1<float>(kb, tc + e * krow + j * 64);
    }
  };
  // 16 x 16 matrix times 16 rows, on top of u
  auto times = [&](const float4_t m, const f64x4 y, f64x4 u) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      u = __builtin_amdgcn_mfma_f64_16x16x4f64((double)m[e], y[e], u, 0, 0, 0);
    return u;
  };
  auto chunk = [&](const Operands& x, const int c) {
    f32x4 ks[4], qs[4];             // short chains, for their rounding
#pragma unroll
    for (int i = 0; i < 4; i++)
      ks[i] = qs[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        ks[e] = mfma4(x.k[j][e], S[j][e], ks[e]);
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        qs[e] = mfma4(x.q[j][e], S[j][e], qs[e]);
    f32x4 sk = (ks[0] + ks[1]) + (ks[2] + ks[3]);
    f32x4 sq = (qs[0] + qs[1]) + (qs[2] + qs[3]);
    if constexpr (NW > 1) {
      f32x4 (*m)[2][64] = meet[c & 1];
      m[wave][0][lane] = sk;
      m[wave][1][lane] = sq;
      __syncthreads();              // the other half is free until the next
      sk = m[0][0][lane];
      sq = m[0][1][lane];
#pragma unroll
      for (int w = 1; w < NW; w++) {
        sk += m[w][0][lane];
        sq += m[w][1][lane];
      }
    }
    const f32x4 zero{0.f, 0.f, 0.f, 0.f};
    const f64x4 none{0., 0., 0., 0.};
    f64x4 rhs, out;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      rhs[e] = (double)act_ld(&x.v[e]) - (double)x.gam[e] * (double)sk[e];
      out[e] = (double)x.gam[e] * (double)sq[e];
    }
    f64x4 u = times(x.inv, rhs, none);
    bool finite = true;
#pragma unroll
    for (int e = 0; e < 4; e++) finite &= fabs(u[e]) < (double)INFINITY;
    const bool mine = c % NW == wave;       // writes the chunk's output
    if (__all(finite)) {
      if (mine) out = times(x.ro, u, out);
    } else {
      // A value that is not finite reaches the tokens before its own as 0
      // times it: token by token, later ones as 0.
      const f64x4 base = out;
      for (int i = 0; i < C; i++) {
        f64x4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = 4 * hi + e <= i ? rhs[e] : 0.;
        y = times(x.inv, y, none);
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (4 * hi + e == i) u[e] = y[e];
      }
      for (int i = 0; i < C; i++) {
        f64x4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = 4 * hi + e <= i ? u[e] : 0.;
        y = times(x.ro, y, base);
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (4 * hi + e == i) out[e] = y[e];
      }
    }
    const float all = __int_as_float(
        __builtin_amdgcn_readlane(__float_as_int(x.gam[3]), 48));   // g_15
    f32x4 w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = (float)(u[e] * (double)x.rest[e]);
    // the chunk's own sum first: S is rounded once, not with every term
    constexpr int HALF = J > 4 ? 4 : J;     // registers
#pragma unroll
    for (int j0 = 0; j0 < J; j0 += HALF) {
      f32x4 add[HALF];
#pragma unroll
      for (int j = 0; j < HALF; j++) add[j] = zero;
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int j = 0; j < HALF; j++)
          add[j] = mfma4(x.kt[j0 + j][e], w[e], add[j]);
#pragma unroll
      for (int j = 0; j < HALF; j++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          S[j0 + j][e] = fmaf(S[j0 + j][e], all, add[j][e]);
    }
    if (mine)
#pragma unroll
      for (int e = 0; e < 4; e++)
        __builtin_amdgcn_raw_buffer_store_b32(
            __float_as_uint((float)out[e]), ob, oat + c * C * orow + e * orow, 0,
            0);
  };

  Operands x0, x1;
  fetch(x0, 0);
  for (int c = 0; c < nc; c += 2) {
    fetch(x1, min(c + 1, nc - 1));
    chunk(x0, c);
    if (c + 1 >= nc) break;
    fetch(x0, min(c + 2, nc - 1));
    chunk(x1, c + 1);
  }
#pragma unroll
  for (int j = 0; j < J; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) sp[(int64_t)(16 * j + e) * V] = S[j][e];
}

}  // namespace delta_chunks
}  // namespace kaito
