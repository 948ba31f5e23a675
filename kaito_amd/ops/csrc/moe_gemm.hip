// Grouped GEMMs of prompt-sized MoE steps: rows sorted by expert, one launch
// per projection, tile bounds from the device's offsets (no host read).
//
//   moe_grouped_up    act[s] = act(x[tok_s] Wg[e]^T, x[tok_s] Wu[e]^T)
//   moe_grouped_down  y[s] = act[s] Wd[e]^T (+ bias), bf16 or f32
//   moe_combine       out[t] = sum over t's pairs of weight * y[row], f32
//                     sums in the order of the choice, plus identity and
//                     shared experts
//
// The products' main loop is that of tile_gemm.h; every workgroup stays and takes
// tile after tile, of the shape that the step's rows need fewest rounds of. Measured
// on one MI355X, us, 8 waves of 128 x 64 on 32x32x16 products with a workgroup per
// tile, now: 8 experts of 2048 x 2048, top 2, 8192 tokens up 272 and 238 (1160
// TFLOP/s), down 131 and 112; 4096 170 and 148, 80 and 69; 2048 93 and 82, 53 and 49;
// 1000 56 and 53, 49 and 34; 300 33 and 30, 32 and 21; 100 31 and 24, 29 and 19. 8 of
// 4096 x 14336, 8192 tokens: 3117 and 2736 (1400 TFLOP/s), 1631 and 1438; 128: 383
// and 357, 297 and 185. 32 of 2048 x 1024, top 4, 2048 tokens 124 and 119, 62 and
// 50. 64 of 1024 x 512, top 4, weights from memory, 4096 tokens 64 and 54, 37 and 29;
// 256, where every row of weights is read for 16 tokens, 29.1 and 27.9, 15.0 and 14.7.
// A library GEMM per expert with its gathers, casts and index_add took 958 us behind
// a host read at the first of these.
#include "tile_gemm.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <type_traits>

namespace kaito {

namespace {

using tile::BK;
using tile::CUS;
using tile::NG;
using tile::GemmArgs;
using tile::Tile;
using tile::SILU;
using tile::CLAMPED;
using tile::RELU2;
using tile::PLAIN;
using tile::PLAIN_F32;

// inclusive sum over the lanes before
KAITO_DEV int lane_scan(int x) {
  auto add = [&](auto ctrl, auto rows) {
    x += __builtin_amdgcn_update_dpp(0, x, decltype(ctrl)::value,
                                     decltype(rows)::value, 0xf, false);
  };
  using std::integral_constant;
  add(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});  // row_shr
  add(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
  add(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // bcast15
  add(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});  // bcast31
  return x;
}

// rows of 64 experts from e0 on, one per lane
struct Rows {
  int o0, o1;
  KAITO_DEV Rows(const GemmArgs& a, const int e0) {
    const int lane = threadIdx.x & 63, e = a.e_base + e0 + lane;
    o0 = e0 + lane < a.E ? a.offsets[e] : 0;
    o1 = e0 + lane < a.E ? a.offsets[e + 1] : 0;
  }
  KAITO_DEV int tiles(const int BM) const { return (o1 - o0 + BM - 1) / BM; }
};

// Tiles of 32 FM x 32 FN of a launch, numbered expert by expert, in blocks of NG
// column tiles x all row tiles, column fastest; every XCD takes one contiguous
// eighth: the 32 in flight behind one L2 share rows and weights.
template <int FM, int FN, int KIND>
struct Tiles {
  static constexpr int BM = 32 * FM, COLS = tile::columns<FN, KIND>();
  const GemmArgs& a;
  const Rows& first;                // of 64 experts
  int scan;                         // of their row tiles
  int ntiles;                       // column tiles
  int share, at, here;              // of an XCD; this one's first and number

  KAITO_DEV Tiles(const GemmArgs& a, const Rows& first) : a(a), first(first) {
    ntiles = (a.N + COLS - 1) / COLS;
    scan = lane_scan(first.tiles(BM));
    int total = __builtin_amdgcn_readlane(scan, 63);
    for (int e0 = 64; e0 < a.E; e0 += 64)
      total += __builtin_amdgcn_readlane(lane_scan(Rows(a, e0).tiles(BM)), 63);
    total *= ntiles;
    share = (total + 7) / 8;
    at = blockIdx.x % 8 * share;
    here = max(min(share, total - at), 0);
  }
  KAITO_DEV Tile operator()(int t) const {
    Tile out{};
    int mtiles = 1;
    t += at;
    auto look = [&](const Rows& r, const int scan, const int e0) {
      const unsigned long long hit = __ballot(scan * ntiles > t);
      if (!hit) {
        t -= __builtin_amdgcn_readlane(scan, 63) * ntiles;
        return false;
      }
      const int src = __builtin_ctzll(hit);
      mtiles = __builtin_amdgcn_readlane(r.tiles(BM), src);
      t -= (__builtin_amdgcn_readlane(scan, src) - mtiles) * ntiles;
      out.expert = a.e_base + e0 + src;
      out.m0 = __builtin_amdgcn_readlane(r.o0, src);
      out.row_end = __builtin_amdgcn_readlane(r.o1, src);
      return true;
    };
    if (!look(first, scan, 0))
      for (int e0 = 64; e0 < a.E; e0 += 64) {
        const Rows r(a, e0);
        if (look(r, lane_scan(r.tiles(BM)), e0)) break;
      }
    const int blk = t / (NG * mtiles);
    const int wide = min(NG, ntiles - blk * NG);
    const int in_blk = t - blk * NG * mtiles;
    out.n0 = (blk * NG + in_blk % wide) * COLS;
    out.m0 += in_blk / wide * BM;
    return out;
  }
};

// What a round takes where the weights come from memory and serve one expert's rows:
// 128 x 256 tiles, which read as much of them as large ones, more than where rows and
// weights are shared, small ones, with four steps under way, a little less. us, weights
// from memory, large, 128 x 256, 256 x 128 and small: 64 experts of 1024 x 512, 1024
// pairs, up 33.5, 30.0, 38.7, 27.2; 32 of 2880 x 2880, 512 pairs, down 130, 126, 131,
// 97, 8192 pairs, up, 345, 423, 416, 398; 64 of 2048 x 1408, 18000 pairs, up, 252,
// 286, 286, 300; 8 of 2048 x 2048, 1400 pairs, up, 50, 44, 42, 47. With 5, 3, 3, 2
// (tile_linear.hip) 92 of 240 such products took 5 % or more longer than with the best
// shape, and the first four here were slower than with a workgroup per tile.
//   Two small tiles for one of 128 x 256 are ahead while rows are few and K is short
// (their rows of x are read twice as often): 64 of 2048 x 1408, up, 1.05 at 24 rows
// an expert, 1.01 at 48, 0.99 at 66; 128 of 4096 x 1536, up, 0.99 at 16, 0.94 at 64;
// 64 of 1024 x 512, down, 1.09 at 16, 1.08 at 64. Of fewer weights than 64 MB they are
// two chains of latencies for one: 24 of 1536 x 768, down, 0.94 to 0.97.
template <int KIND>
__global__ __launch_bounds__(256, 1) void moe_grouped_kernel(const GemmArgs a,
                                                             const int small) {
  __shared__ __attribute__((aligned(1024))) short lds[tile::LDS];
  const Rows rows(a, 0);
  tile::run<KIND>(a, lds, {50, 40, 30, small}, Tiles<8, 8, KIND>(a, rows),
                  Tiles<4, 8, KIND>(a, rows), Tiles<8, 4, KIND>(a, rows),
                  Tiles<4, 4, KIND>(a, rows));
}

// ---- keys and values of latent rows ----------------------------------------
// [k | v][t] = c[t] [Wk | Wv^T]^T, tiles of 256 x 256 over both: the tiles of
// Wk's N1 rows first. Behind one another, as a library product and a batched one
// of Wv as it is stored, they took 32 + 42 us (8192 rows of 512, 16 heads of 128 +
// 128; 34 GFLOP, 80 MB), here 41 with the transposition: 8 K steps a tile.
__global__ __launch_bounds__(256, 1) void latent_kv_kernel(const GemmArgs a,
                                                           const int T) {
  __shared__ __attribute__((aligned(1024))) short lds[tile::LDS];
  const int ntiles = (a.N + 255) / 256, mtiles = (T + 255) / 256;
  const int total = ntiles * mtiles, share = (total + 7) / 8;
  const int at = blockIdx.x % 8 * share, here = min(share, total - at);
  int i = blockIdx.x / 8;
  tile::stream<8, 8, PLAIN, true>(a, lds, [&](Tile& t) {
    if (i >= here) return false;
    const int blk = (at + i) / (NG * mtiles), in_blk = at + i - blk * NG * mtiles;
    const int wide = min(NG, ntiles - blk * NG);
    t = {0, in_blk / wide * 256, T, (blk * NG + in_blk % wide) * 256};
    i += CUS / 8;
    return true;
  });
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

// rows: of all experts, which `offsets` ends; w: this rank's
template <int KIND>
void launch_grouped(const GemmArgs& a, const int64_t rows,
                    const at::Tensor& offsets, const at::Tensor& w) {
  const int64_t of_one = rows / std::max<int64_t>(offsets.numel() - 1, 1);
  const bool few = a.K + 32 * of_one < 4096 && w.numel() >= 1 << 25;
  hipLaunchKernelGGL((moe_grouped_kernel<KIND>), dim3(CUS), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), a, few ? 19 : 20);
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
              w.size(2) == a.K && a.K % BK == 0 && a.N % 64 == 0 && a.K > 0 &&
              act.size(1) < tile::MOST_OUTPUTS);
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
  if (x.numel() * 2 > tile::MOST_BYTES) {       // beyond 32-bit offsets
    gathered = x.index_select(0, sorted_ids);
    a.x = (const short*)gathered.data_ptr();
    a.rows = nullptr;
  }
  a.offsets = offsets.data_ptr<int>();
  a.limit = (float)act_limit;
  if (act.size(0) == 0 || a.E == 0 || a.N == 0) return;
  if (plain) launch_grouped<RELU2>(a, act.size(0), offsets, w);
  else if (act_mode == 1) launch_grouped<CLAMPED>(a, act.size(0), offsets, w);
  else launch_grouped<SILU>(a, act.size(0), offsets, w);
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
              a.N % 64 == 0 && a.K > 0 && y.size(1) < tile::MOST_OUTPUTS);
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
  if (wide) launch_grouped<PLAIN_F32>(a, y.size(0), offsets, w);
  else launch_grouped<PLAIN>(a, y.size(0), offsets, w);
}

// kv [T, H D + H V]: c [T, K] times wk [H, D, K] (rows K long) and wv [H, K, V]
void latent_kv(at::Tensor kv, at::Tensor c, at::Tensor wk, at::Tensor wv) {
  check16(kv); check16(c); check16(wk); check16(wv);
  TORCH_CHECK(c.dim() == 2 && kv.dim() == 2 && wk.dim() == 3 && wv.dim() == 3);
  const int64_t T = c.size(0), K = c.size(1), H = wk.size(0), V = wv.size(2);
  const int64_t N1 = H * wk.size(1);
  TORCH_CHECK(wk.size(2) == K && wv.size(0) == H && wv.size(1) == K &&
              kv.size(0) == T && kv.size(1) == N1 + H * V &&
              K % 64 == 0 && K > 0 && V % 64 == 0 && N1 % 256 == 0 &&
              T < (1ll << 22) && kv.size(1) < tile::MOST_OUTPUTS);
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
  a.x2 = a.x;
  a.w2 = (const short*)wt.data_ptr();
  a.n2 = (int)N1;
  hipLaunchKernelGGL(latent_kv_kernel, dim3(CUS), dim3(256), 0, stream, a,
                     (int)T);
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
