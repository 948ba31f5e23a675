// MLA (multi-head latent attention) for gfx950: DECODE over the paged cache
// and what precedes attention in a layer.
//
// Absorbed decode of DeepSeek V2/V3/R1 (models/mla.py): one latent row per
// cached token, c_kv[R = 512] | k_rope[P = 64], shared by every head. With
// q_c = W_uk^T q_nope, scores[h][t] = (q_c | q_rope)[h] . row[t] and
// out[h] = sum_t softmax * row[t][0:R]. Stands for the vLLM MLA backend that
// the reference hands the deepseek presets to (supported_models.yaml:
// deepseek-v3-0324, deepseek-r1-0528).
//
// mla_decode_kernel: a workgroup of 1 to 4 waves per (sequence, 16 heads, split of
// the keys); 16 heads fill the columns of v_mfma_f32_16x16x32_bf16. Every
// wave walks its own keys, 32 at a time, without a barrier:
//   - two pages (18 KB each, contiguous) go to the wave's LDS by 16-byte
//     direct loads, the chunk order of a row exclusive-ored with its number,
//     so that both ways to read it spread over the banks;
//   - S^T = C Q^T reads 16-byte chunks of rows; a head's scores sit in one
//     column, so maximum and rescale are per-lane scalars;
//   - O^T += C^T P^T takes P (bf16) from the score registers and reads the
//     same rows again, transposed, as columns: the cache row serves as key
//     and as value from one load.
// The waves' (max, sum, O) are folded through LDS, the splits' by
// mla_fold_kernel.
//
// What bounds it: bytes in flight. A tile costs a CU 68 KB of LDS reads (550
// cycles) and 70 matrix instructions on one of four SIMDs for 36 KB of cache,
// far less than HBM takes for it (2900 cycles at 13 B per CU and cycle), so
// LDS is spent on loads under way: 4 x 36 KB per CU. Measured on one MI355X
// against 16-token blocks staged by 256 threads through registers behind two
// barriers, with V transposed by scalar LDS stores (before -> now, 16 heads):
//   1 sequence of 512 tokens: 28 -> 14 us;  32 of 1800: 65 -> 26;
//   256 of 400: 77 -> 30;  2048 of 300: 351 -> 160 (4.4 TB/s);
//   128 heads, 250 of 300: 352 -> 82 us.
//
// Cache layout: [num_blocks, 16, R + P] bf16.
#include "flash_prefill.h"
#include <algorithm>
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

namespace {

using flash::hbf16x8;
using flash::LOG2E;

constexpr int R = 512, P = 64, DT = R + P;
constexpr int BS = 16;              // tokens per page
constexpr int KT = 32;              // keys per wave step: two pages
constexpr int WIDE = 4;             // waves whose rows fill the LDS
constexpr int HT = 16;              // heads per workgroup
constexpr int RS = R + 4;           // floats per head in the fold

struct MlaArgs {
  short* out;                       // [T, H, R]
  const short* qc;                  // q in the latent space: t, h strides
  const short* qr;                  // its rotated part
  int64_t qc_ts, qc_hs, qr_ts, qr_hs;
  const short* cache;
  const int* block_tables;          // [T, max_blocks]
  const int* seq_lens;              // [T]
  float scale;
  int T, H, max_blocks;
  float* part;                      // splits: [splits, T, H, R]
  float* ml;                        // splits: [splits, T, H, 2] max, sum
};

// Workgroup id -> (sequence, head tile). Ids go round the 8 dies, each with
// its own L2: the tiles of a sequence, which read the same rows, share one.
KAITO_DEV int seq_of(int id, int tiles) {
  return id / (8 * tiles) * 8 + id % 8;
}

template <int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64)
__attribute__((amdgpu_waves_per_eu(1, 1)))
void mla_decode_kernel(const MlaArgs a) {
  constexpr int LP = BS * DT / 8 / 64;      // loads per lane and page: 18
  constexpr int KK = DT / 32, OT = R / 16, KB = 3;
  __shared__ __attribute__((aligned(128))) short lds[NW][KT * DT];
  __shared__ float s_m[NW][HT], s_l[NW][HT];
  static_assert(sizeof(lds) >= NW * HT * RS * sizeof(float), "fold");
  const int tiles_h = (a.H + HT - 1) / HT;
  const int seq = seq_of(blockIdx.x, tiles_h);
  const int h0 = blockIdx.x / 8 % tiles_h * HT;
  if (seq >= a.T) return;           // the last 8 sequences may be fewer
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int seq_len = a.seq_lens[seq];
  const int* bt = a.block_tables + (int64_t)seq * a.max_blocks;

  const int tiles = (seq_len + KT - 1) / KT;
  const int nsplit = SPLIT ? gridDim.y : 1, split = SPLIT ? blockIdx.y : 0;
  const int per = (tiles + nsplit * NW - 1) / (nsplit * NW);
  const int t0 = min(tiles, (split * NW + wave) * per);
  const int t1 = min(tiles, t0 + per);
  const int last_page = (seq_len - 1) / BS;
  if constexpr (SPLIT) {
    if (split * NW * per >= tiles) {        // nothing for any of the waves
      if (threadIdx.x < HT && h0 + (int)threadIdx.x < a.H) {
        float* ml = a.ml +
            (((int64_t)split * a.T + seq) * a.H + h0 + threadIdx.x) * 2;
        ml[0] = -1e30f;
        ml[1] = 0.f;
      }
      return;
    }
  }

  hbf16x8 qf[KK];
  {
    const int h = min(h0 + lo, a.H - 1);
    const short* qc = a.qc + seq * a.qc_ts + h * a.qc_hs + hi * 8;
    const short* qr = a.qr + seq * a.qr_ts + h * a.qr_hs + hi * 8;
#pragma unroll
    for (int kk = 0; kk < KK; kk++)
      qf[kk] = *reinterpret_cast<const hbf16x8*>(
          kk < R / 32 ? qc + kk * 32 : qr + (kk - R / 32) * 32);
  }
  float m = -1e30f, l = 0.f;
  f32x4 o[OT];
#pragma unroll
  for (int i = 0; i < OT; i++) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  short* const st = lds[wave];
  // chunk c of row r lies at place c ^ (r / 2 % 8); 72 chunks a row, so the
  // low three bits stay in the row
  uint32_t off[LP / 2];             // the other 8 rows of a page: off ^ 32
#pragma unroll
  for (int j = 0; j < LP / 2; j++) {
    const uint32_t s = j * 64 + lane;
    off[j] = (s ^ (s / (DT / 8) >> 1 & 7)) * 8;
  }
  const short* kp[2];                       // even and odd 32-dim steps
#pragma unroll
  for (int e = 0; e < 2; e++)
    kp[e] = st + lo * DT + ((e * 4 + hi) ^ (lo >> 1 & 7)) * 8;
  const int vrow = 4 * hi + (lo >> 2), vc = (lo & 3) >> 1, ve = (lo & 1) * 4;
  const short* vp[4];
#pragma unroll
  for (int e = 0; e < 4; e++)
    vp[e] = st + vrow * DT + ((e * 2 + vc) ^ (vrow >> 1 & 7)) * 8 + ve;
  const float c = a.scale * LOG2E;

  int pages = 0, pages_at = -64;    // lane i: page pages_at + i of the table
  for (int t = t0; t < t1; t++) {
    // the pages of a tile are even and odd: one test serves both
    if (t * 2 >= pages_at + 64) {           // uniform; spans move forward
      pages_at = t * 2;
      pages = bt[min(t * 2 + lane, last_page)];
    }
    const short* src[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
      src[i] = a.cache + (int64_t)__builtin_amdgcn_readlane(
          pages, t * 2 + i - pages_at) * BS * DT;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < LP; j++)
        flash::lds_copy16(
            src[i] + (j < LP / 2 ? off[j] : (off[j - LP / 2] ^ 32) + 8 * DT),
            st + (i * LP + j) * 512);
    __builtin_amdgcn_s_waitcnt(0x0f70);     // vmcnt(0): this wave's own rows
    __builtin_amdgcn_wave_barrier();
    // ---- S^T: keys 16 i + 4 hi + r of head lo
    f32x4 s[2][2];
    hbf16x8 kf[2][KB][2];           // a batch of steps and the next one's
    auto read_k = [&](const int b) {
#pragma unroll
      for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int i = 0; i < 2; i++)
          kf[b & 1][kk][i] = *reinterpret_cast<const hbf16x8*>(
              kp[(b * KB + kk) & 1] + i * BS * DT + (b * KB + kk) / 2 * 64);
      __builtin_amdgcn_sched_barrier(0);    // all under way before products
    };
    read_k(0);
#pragma unroll
    for (int i = 0; i < 2; i++)
      s[i][0] = s[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < KK / KB; b++) {
      if (b + 1 < KK / KB) read_k(b + 1);
#pragma unroll
      for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int i = 0; i < 2; i++)
          s[i][kk & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              kf[b & 1][kk][i], qf[b * KB + kk], s[i][kk & 1], 0, 0, 0);
    }
    s[0][0] += s[0][1];
    s[1][0] += s[1][1];
    // ---- softmax
    const int key0 = t * KT;
    const bool whole = key0 + KT <= seq_len;
    float mx = -1e30f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s[i][0][r] *= c;
        if (!whole && key0 + 16 * i + 4 * hi + r >= seq_len)
          s[i][0][r] = -1e30f;
        mx = fmaxf(mx, s[i][0][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float corr = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= corr;
#pragma unroll
      for (int i = 0; i < OT; i++) o[i] *= corr;
    }
    hbf16x8 p;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float w = s[i][0][r] > -1e29f
            ? __builtin_amdgcn_exp2f(s[i][0][r] - m) : 0.f;
        l += w;
        p[i * 4 + r] = (__bf16)w;
      }
    // ---- O^T: dims 16 i + 4 hi + r of head lo
#pragma unroll
    for (int i = 0; i < OT; i++) {
      const short* at = vp[i & 3] + i / 4 * 64;
      const short4_t a4 = flash::read_tr(at), b4 = flash::read_tr(at + BS * DT);
      const hbf16x8 vf = __builtin_bit_cast(
          hbf16x8, __builtin_shufflevector(a4, b4, 0, 1, 2, 3, 4, 5, 6, 7));
      o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, p, o[i], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 16, 1);
#pragma unroll
    for (int i = 0; i < OT - 8; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 1);
    __builtin_amdgcn_wave_barrier();        // rows read before the next ones
  }

  // ---- fold the waves through LDS
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float* const acc = reinterpret_cast<float*>(&lds[0][0]);
  __syncthreads();                  // every wave is done with its rows
#pragma unroll
  for (int i = 0; i < OT; i++)
    *reinterpret_cast<f32x4*>(acc + (wave * HT + lo) * RS + i * 16 + hi * 4) =
        o[i];
  if (hi == 0) { s_m[wave][lo] = m; s_l[wave][lo] = l; }
  __syncthreads();
#pragma unroll 2
  for (int idx = threadIdx.x; idx < HT * R / 4; idx += NW * 64) {
    const int g = idx / (R / 4), d = idx % (R / 4) * 4;
    if (h0 + g >= a.H) break;
    float gm = -1e30f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) gm = fmaxf(gm, s_m[w][g]);
    f32x4 num{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float e = __builtin_amdgcn_exp2f(s_m[w][g] - gm);
      num += e * *reinterpret_cast<const f32x4*>(acc + (w * HT + g) * RS + d);
      den += e * s_l[w][g];
    }
    const int64_t row = ((int64_t)split * a.T + seq) * a.H + h0 + g;
    if constexpr (SPLIT) {
      *reinterpret_cast<f32x4*>(a.part + row * R + d) = num;
      if (d == 0) { a.ml[row * 2] = gm; a.ml[row * 2 + 1] = den; }
    } else {
      const float inv = 1.f / fmaxf(den, 1e-20f);
      short4_t v;
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] = f32_to_bf16(num[r] * inv);
      *reinterpret_cast<short4_t*>(a.out + row * R + d) = v;
    }
  }
}

// One workgroup per (sequence, head) folds the splits, up to 64; empty ones
// (no key) hold a maximum and no row. A chain of loads, so short ones: lane s
// of every wave has split s's weight, 4 groups of 2 waves take every 4th row.
__global__ __launch_bounds__(R)
void mla_fold_kernel(short* __restrict__ out, const float* __restrict__ part,
                     const float* __restrict__ ml, const int splits) {
  __shared__ f32x4 red[4][R / 4];
  const int64_t row = blockIdx.x, rows = gridDim.x;
  const int lane = threadIdx.x & 63;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / (R / 4));
  const int col = threadIdx.x % (R / 4);
  float m = -1e30f, l = 0.f;
  if (lane < splits) {
    const float2 v = reinterpret_cast<const float2*>(ml)[lane * rows + row];
    m = v.x;
    l = v.y;
  }
  float gm = m;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) gm = fmaxf(gm, __shfl_xor(gm, d, 64));
  const float e = m > -1e29f ? __builtin_amdgcn_exp2f(m - gm) : 0.f;
  float den = e * l;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) den += __shfl_xor(den, d, 64);
  f32x4 num{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = group; s < splits; s += 4) {
    const float w = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e), s));
    if (w == 0.f) continue;
    num += w * *reinterpret_cast<const f32x4*>(part + (s * rows + row) * R +
                                               col * 4);
  }
  red[group][col] = num;
  __syncthreads();
  if (group > 0) return;
  num += red[1][col] + red[2][col] + red[3][col];
  const float inv = 1.f / fmaxf(den, 1e-20f);
  short4_t v;
#pragma unroll
  for (int r = 0; r < 4; r++) v[r] = f32_to_bf16(num[r] * inv);
  *reinterpret_cast<short4_t*>(out + row * R + col * 4) = v;
}

}  // namespace

// qc [T, H, R] and qr [T, H, P] of any token and head stride
void mla_decode(at::Tensor out, at::Tensor qc, at::Tensor qr, at::Tensor cache,
                at::Tensor block_tables, at::Tensor seq_lens, double scale) {
  auto ok = [](const at::Tensor& t) {
    return t.is_cuda() && t.dtype() == at::kBFloat16 && t.stride(-1) == 1;
  };
  TORCH_CHECK(ok(qc) && ok(qr) && qc.dim() == 3 && qr.dim() == 3);
  TORCH_CHECK(cache.dtype() == at::kBFloat16 && cache.is_contiguous());
  TORCH_CHECK(out.is_contiguous() && out.dtype() == at::kBFloat16);
  TORCH_CHECK(block_tables.dtype() == at::kInt
              && seq_lens.dtype() == at::kInt);
  const int T = qc.size(0), H = qc.size(1);
  TORCH_CHECK(qc.size(2) == R && qr.size(2) == P && out.size(2) == R &&
              cache.size(2) == DT, "unsupported MLA dims r=", out.size(2),
              " r+rope=", cache.size(2), " (deepseek family is 512/576)");
  TORCH_CHECK(qr.size(0) == T && qr.size(1) == H && out.size(0) == T &&
              out.size(1) == H);
  TORCH_CHECK(cache.size(1) == BS, "block_size must be 16");
  if (T == 0 || H == 0) return;
  MlaArgs a{};
  a.out = (short*)out.data_ptr();
  a.qc = (const short*)qc.data_ptr();
  a.qr = (const short*)qr.data_ptr();
  a.qc_ts = qc.stride(0); a.qc_hs = qc.stride(1);
  a.qr_ts = qr.stride(0); a.qr_hs = qr.stride(1);
  a.cache = (const short*)cache.data_ptr();
  a.block_tables = block_tables.data_ptr<int>();
  a.seq_lens = seq_lens.data_ptr<int>();
  a.scale = (float)scale;
  a.T = T; a.H = H;
  a.max_blocks = block_tables.size(1);
  auto stream = at::hip::getCurrentHIPStream();
  // 4 waves have a CU to themselves: splits until 256 workgroups, as long as
  // every wave keeps a tile of the longest context that the table can hold
  // (the lengths are on the device). With more workgroups than CUs, smaller
  // ones start and fold behind the others' loads: 768 sequences of 300
  // tokens 72 us with 4 waves, 68 with 2; 2048 193, 169 and 160 with 1.
  const int tiles_h = (H + HT - 1) / HT;
  const int64_t grid = (int64_t)(T + 7) / 8 * 8 * tiles_h;
  const int64_t splits = std::min<int64_t>(
      {(256 + (int64_t)T * tiles_h - 1) / ((int64_t)T * tiles_h),
       (int64_t)a.max_blocks * BS / (WIDE * KT), 64});
  if (splits > 1) {
    auto opts = out.options().dtype(at::kFloat);
    at::Tensor part = at::empty({splits, T, H, R}, opts);
    at::Tensor ml = at::empty({splits, T, H, 2}, opts);
    a.part = part.data_ptr<float>();
    a.ml = ml.data_ptr<float>();
    hipLaunchKernelGGL((mla_decode_kernel<WIDE, true>), dim3(grid, splits),
                       dim3(WIDE * 64), 0, stream, a);
    hipLaunchKernelGGL(mla_fold_kernel, dim3(T * H), dim3(R), 0, stream,
                       a.out, a.part, a.ml, (int)splits);
  } else if ((int64_t)T * tiles_h <= 512) {
    hipLaunchKernelGGL((mla_decode_kernel<WIDE, false>), dim3(grid),
                       dim3(WIDE * 64), 0, stream, a);
  } else if ((int64_t)T * tiles_h > 1024) {
    hipLaunchKernelGGL((mla_decode_kernel<1, false>), dim3(grid),
                       dim3(64), 0, stream, a);
  } else {
    hipLaunchKernelGGL((mla_decode_kernel<WIDE / 2, false>), dim3(grid),
                       dim3(WIDE / 2 * 64), 0, stream, a);
  }
}

namespace {

// What a layer needs before attention, in one launch per step instead of
// seven (three copies of strided parts, norm, rotation, cache write; about
// 4 us each): RMS norm of the latent, rotation of the shared key part and of
// the queries' rotated parts, scatter into the cache. Bound by the launch for
// decode steps. Wave 0 of a token's workgroup has the latent (8 dims a lane),
// the others rotate 8 pairs a lane; norm and rotation round as the single
// kernels do.
struct PrepareArgs {
  short* q_out;                     // [T, H, P]
  short* c_out;                     // [T, R]
  short* k_out;                     // [T, P]
  short* cache;                     // [NB, BS, DT] or nullptr
  const short* q;
  int64_t q_ts, q_hs;
  const short* kv_a;
  int64_t kv_ts;
  const short* w;
  float eps;
  const int64_t* positions;
  const float* cos_sin;             // [max_pos, P]
  const int64_t* slots;
  int H;
};

KAITO_DEV void prepare_token(const PrepareArgs& a, const int64_t t) {
  short* __restrict__ q_out = a.q_out;
  short* __restrict__ c_out = a.c_out;
  short* __restrict__ k_out = a.k_out;
  short* __restrict__ cache = a.cache;
  const short* __restrict__ q = a.q;
  const short* __restrict__ kv_a = a.kv_a;
  const short* __restrict__ w = a.w;
  const float* __restrict__ cos_sin = a.cos_sin;
  const int64_t* __restrict__ positions = a.positions;
  const int64_t* __restrict__ slots = a.slots;
  const int64_t q_ts = a.q_ts, q_hs = a.q_hs, kv_ts = a.kv_ts;
  const float eps = a.eps;
  const int H = a.H;
  const int tid = threadIdx.x;
  const int64_t slot = cache ? slots[t] : -1;
  if (tid < 64) {
    const short8_t v =
        *reinterpret_cast<const short8_t*>(kv_a + t * kv_ts + tid * 8);
    const short8_t g = *reinterpret_cast<const short8_t*>(w + tid * 8);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float f = bf16_to_f32(v[j]);
      ss += f * f;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) ss += __shfl_xor(ss, d, 64);
    const float inv = rsqrtf(ss / (float)R + eps);
    short8_t o;
#pragma unroll
    for (int j = 0; j < 8; j++)
      o[j] = f32_to_bf16(bf16_to_f32(v[j]) * inv * bf16_to_f32(g[j]));
    *reinterpret_cast<short8_t*>(c_out + t * R + tid * 8) = o;
    if (slot >= 0)
      *reinterpret_cast<short8_t*>(cache + slot * DT + tid * 8) = o;
    return;
  }
  const float* cs = cos_sin + positions[t] * P;
  // (head, 8 pairs); head H is the key
  for (int i = tid - 64; i < (H + 1) * (P / 16); i += 192) {
    const int h = i / (P / 16), d = i % (P / 16) * 8;
    const short* src = h < H ? q + t * q_ts + h * q_hs
                             : kv_a + t * kv_ts + R;
    short* dst = h < H ? q_out + (t * H + h) * P : k_out + t * P;
    const short8_t xa = *reinterpret_cast<const short8_t*>(src + d);
    const short8_t xb = *reinterpret_cast<const short8_t*>(src + P / 2 + d);
    short8_t oa, ob;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float co = cs[d + j], si = cs[P / 2 + d + j];
      const float x = bf16_to_f32(xa[j]), y = bf16_to_f32(xb[j]);
      oa[j] = f32_to_bf16(x * co - y * si);
      ob[j] = f32_to_bf16(y * co + x * si);
    }
    *reinterpret_cast<short8_t*>(dst + d) = oa;
    *reinterpret_cast<short8_t*>(dst + P / 2 + d) = ob;
    if (h == H && slot >= 0) {
      short* row = cache + slot * DT + R;
      *reinterpret_cast<short8_t*>(row + d) = oa;
      *reinterpret_cast<short8_t*>(row + P / 2 + d) = ob;
    }
  }
}

__global__ __launch_bounds__(256)
void mla_prepare_kernel(const PrepareArgs a) { prepare_token(a, blockIdx.x); }

}  // namespace

// q [T, H, P] of any token and head stride; an empty cache: nothing cached
static PrepareArgs prepare_args(
    const at::Tensor& q_out, const at::Tensor& c_out, const at::Tensor& k_out,
    const at::Tensor& cache, const at::Tensor& q, const at::Tensor& kv_a,
    const at::Tensor& w, double eps, const at::Tensor& positions,
    const at::Tensor& cos_sin, const at::Tensor& slots) {
  auto ok = [](const at::Tensor& t) {
    bool fine = t.is_cuda() && t.dtype() == at::kBFloat16 &&
                t.stride(-1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0;
    for (int i = 0; i + 1 < t.dim(); i++)
      fine = fine && (t.size(i) == 1 || t.stride(i) % 8 == 0);
    return fine;
  };
  const int64_t T = q.size(0), H = q.size(1);
  TORCH_CHECK(ok(q) && ok(kv_a) && ok(w) && q.dim() == 3 && kv_a.dim() == 2);
  TORCH_CHECK(q.size(2) == P && kv_a.size(0) == T && kv_a.size(1) == DT &&
              w.numel() == R);
  TORCH_CHECK(ok(q_out) && ok(c_out) && ok(k_out) && q_out.is_contiguous() &&
              c_out.is_contiguous() && k_out.is_contiguous() &&
              q_out.numel() == T * H * P && c_out.numel() == T * R &&
              k_out.numel() == T * P);
  TORCH_CHECK(positions.dtype() == at::kLong && positions.numel() >= T &&
              positions.is_contiguous() && cos_sin.dtype() == at::kFloat &&
              cos_sin.size(1) == P && cos_sin.is_contiguous());
  const bool cached = cache.numel() > 0;
  if (cached) {
    TORCH_CHECK(cache.dtype() == at::kBFloat16 && cache.is_contiguous() &&
                cache.size(2) == DT && slots.dtype() == at::kLong &&
                slots.numel() == T && slots.is_contiguous());
  }
  return {(short*)q_out.data_ptr(), (short*)c_out.data_ptr(),
          (short*)k_out.data_ptr(),
          cached ? (short*)cache.data_ptr() : nullptr,
          (const short*)q.data_ptr(), q.stride(0), q.stride(1),
          (const short*)kv_a.data_ptr(), kv_a.stride(0),
          (const short*)w.data_ptr(), (float)eps,
          positions.data_ptr<int64_t>(), cos_sin.data_ptr<float>(),
          cached ? slots.data_ptr<int64_t>() : nullptr, (int)H};
}

void mla_prepare(at::Tensor q_out, at::Tensor c_out, at::Tensor k_out,
                 at::Tensor cache, at::Tensor q, at::Tensor kv_a, at::Tensor w,
                 double eps, at::Tensor positions, at::Tensor cos_sin,
                 at::Tensor slots) {
  const PrepareArgs a = prepare_args(q_out, c_out, k_out, cache, q, kv_a, w,
                                     eps, positions, cos_sin, slots);
  if (q.size(0) == 0) return;
  hipLaunchKernelGGL(mla_prepare_kernel, dim3(q.size(0)), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), a);
}

namespace {

// y[t, h] = x[t, h] W[h] for the two small products around absorbed decode
// (W_uk [nope, R] and W_uv [R, v] per head), up to 32 rows: a workgroup per
// (32 columns, head) holds its [K, 32] of W in LDS, every byte on its way at
// once, and reads it transposed (C^T = W^T X^T); two waves per 16 columns take
// half of K each. Bound by the chain launch -> load -> products; the batched
// library products took 12.3 (K = 128) and 4.7 us (K = 512) of which the
// second needed a copy of 4.7 us to transpose its result, these
// 5.9 each (32 rows of 16 heads, with the launch).
struct HeadArgs {
  short* y;                         // [T, H, N]
  const short* x;
  int64_t x_ts, x_hs;
  const short* w;                   // [H, K, N]
  int T, H, K, N;
};

// wt: [K][32]
template <int MT>
KAITO_DEV void head_tile(const HeadArgs& a, short* wt, f32x4 (&red)[2][MT][64],
                         const int n0, const int head) {
  short* __restrict__ y = a.y;
  const short* __restrict__ x = a.x;
  const short* __restrict__ w = a.w;
  const int64_t x_ts = a.x_ts, x_hs = a.x_hs;
  const int T = a.T, H = a.H, K = a.K, N = a.N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const int half = wave >> 1, col = (wave & 1) * 16;
  const short* wh = w + (int64_t)head * K * N + n0;
  // slot s (16 bytes) is row s / 4, place s % 4
  for (int j = 0; j < K / 64; j++) {
    const int s = j * 256 + threadIdx.x, row = s / 4;
    const int c = s % 4 ^ (row >> 2 & 1) << 1;
    flash::lds_copy16(wh + (int64_t)row * N + c * 8,
                      wt + (j * 256 + wave * 64) * 8);
  }
  const short* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; m++)
    xp[m] = x + min(m * 16 + lo, T - 1) * x_ts + head * x_hs + hi * 4;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  // rows k + 4 hi + j and k + 16 + 4 hi + j: the order of a transposed read
  const int row = 4 * hi + (lo >> 2);
  const short* wp = wt + row * 32 +
      ((col / 8 + ((lo & 3) >> 1)) ^ (row >> 2 & 1) << 1) * 8 + (lo & 1) * 4;
#pragma unroll 4
  for (int k = half * (K / 2); k < (half + 1) * (K / 2); k += 32) {
    const short4_t a4 = flash::read_tr(wp + k * 32);
    const short4_t b4 = flash::read_tr(wp + (k + 16) * 32);
    const hbf16x8 wf = __builtin_bit_cast(
        hbf16x8, __builtin_shufflevector(a4, b4, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const short4_t u = *reinterpret_cast<const short4_t*>(xp[m] + k);
      const short4_t v = *reinterpret_cast<const short4_t*>(xp[m] + k + 16);
      const hbf16x8 xf = __builtin_bit_cast(
          hbf16x8, __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7));
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, acc[m], 0, 0, 0);
    }
  }
  if (half) {
#pragma unroll
    for (int m = 0; m < MT; m++) red[wave & 1][m][lane] = acc[m];
  }
  __syncthreads();
  if (half) return;
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int t = m * 16 + lo;
    if (t >= T) break;
    const f32x4 v = acc[m] + red[wave & 1][m][lane];
    *reinterpret_cast<short4_t*>(
        y + ((int64_t)t * H + head) * N + n0 + col + hi * 4) =
        short4_t{f32_to_bf16(v[0]), f32_to_bf16(v[1]), f32_to_bf16(v[2]),
                 f32_to_bf16(v[3])};
  }
}

template <int MT>
__global__ __launch_bounds__(256) void head_rows_kernel(const HeadArgs a) {
  extern __shared__ __attribute__((aligned(128))) short wt[];
  __shared__ f32x4 red[2][MT][64];
  head_tile<MT>(a, wt, red, blockIdx.x * 32, blockIdx.y);
}

// mla_prepare's workgroups and behind them those of head_rows: neither reads what
// the other writes, and both are little more than a launch (one MI355X, 32 rows of
// 16 heads: 2.5 and 3.6 us, together 3.7).
template <int MT>
__global__ __launch_bounds__(256)
void mla_prepare_rows_kernel(const PrepareArgs p, const HeadArgs a) {
  extern __shared__ __attribute__((aligned(128))) short wt[];
  __shared__ f32x4 red[2][MT][64];
  if ((int)blockIdx.x < a.T) {
    prepare_token(p, blockIdx.x);
  } else {
    const int b = blockIdx.x - a.T, tiles = a.N / 32;
    head_tile<MT>(a, wt, red, b % tiles * 32, b / tiles);
  }
}

}  // namespace

// y [T, H, N], x [T, H, K] of any token and head stride, w [H, K, N]
static HeadArgs head_args(const at::Tensor& y, const at::Tensor& x,
                          const at::Tensor& w) {
  for (const at::Tensor* t : {&y, &x, &w})
    TORCH_CHECK(t->is_cuda() && t->dtype() == at::kBFloat16 && t->dim() == 3);
  const int64_t T = x.size(0), H = x.size(1), K = x.size(2), N = w.size(2);
  TORCH_CHECK(y.is_contiguous() && w.is_contiguous() && x.stride(2) == 1 &&
              y.size(0) == T && y.size(1) == H && y.size(2) == N &&
              w.size(0) == H && w.size(1) == K);
  TORCH_CHECK(T <= 32 && K % 64 == 0 && K > 0 && K <= 512 && N % 32 == 0 &&
              x.stride(0) % 4 == 0 && x.stride(1) % 4 == 0 &&
              (uintptr_t)x.data_ptr() % 8 == 0 &&
              (uintptr_t)w.data_ptr() % 16 == 0);
  return {(short*)y.data_ptr(), (const short*)x.data_ptr(), x.stride(0),
          x.stride(1), (const short*)w.data_ptr(), (int)T, (int)H, (int)K,
          (int)N};
}

void head_rows(at::Tensor y, at::Tensor x, at::Tensor w) {
  const HeadArgs a = head_args(y, x, w);
  if (a.T == 0 || a.H == 0 || a.N == 0) return;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(a.N / 32, a.H), dim3(256), a.K * 64,
                       at::hip::getCurrentHIPStream(), a);
  };
  if (a.T <= 16) launch(&head_rows_kernel<1>);
  else launch(&head_rows_kernel<2>);
}

// mla_prepare and head_rows of the same up to 32 rows
void mla_prepare_rows(at::Tensor q_out, at::Tensor c_out, at::Tensor k_out,
                      at::Tensor cache, at::Tensor q, at::Tensor kv_a,
                      at::Tensor w, double eps, at::Tensor positions,
                      at::Tensor cos_sin, at::Tensor slots, at::Tensor y,
                      at::Tensor x, at::Tensor wx) {
  const PrepareArgs p = prepare_args(q_out, c_out, k_out, cache, q, kv_a, w,
                                     eps, positions, cos_sin, slots);
  const HeadArgs a = head_args(y, x, wx);
  TORCH_CHECK(q.size(0) == a.T);
  if (a.T == 0) return;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(a.T + a.N / 32 * a.H), dim3(256),
                       a.K * 64, at::hip::getCurrentHIPStream(), p, a);
  };
  if (a.T <= 16) launch(&mla_prepare_rows_kernel<1>);
  else launch(&mla_prepare_rows_kernel<2>);
}

// MLA cache write alone: latent row (c_kv ‖ k_rope) scattered to the paged
// cache. One wave per token: 64 lanes x 16 B covers the 512-dim c_kv; lanes
// 0-7 append the 64 rope dims.
__global__ __launch_bounds__(64, 8)
void mla_cache_write_kernel(
    short* __restrict__ cache,          // [NB, BS, R+P] bf16
    const short* __restrict__ c_kv,     // [T, R]
    const short* __restrict__ k_pe,     // [T, P] (row stride pe_stride)
    const int64_t* __restrict__ slots,  // [T]; <0 = skip (padding)
    const int64_t pe_stride) {
  const int t = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t slot = slots[t];
  if (slot < 0) return;
  short* dst = cache + slot * DT;
  static_assert(R == 64 * 8 && P == 8 * 8);
  *reinterpret_cast<short8_t*>(dst + lane * 8) =
      *reinterpret_cast<const short8_t*>(c_kv + (int64_t)t * R + lane * 8);
  if (lane < P / 8)
    *reinterpret_cast<short8_t*>(dst + R + lane * 8) =
        *reinterpret_cast<const short8_t*>(k_pe + t * pe_stride + lane * 8);
}

void mla_cache_write(at::Tensor cache, at::Tensor c_kv, at::Tensor k_pe,
                     at::Tensor slots) {
  TORCH_CHECK(cache.is_cuda() && cache.dtype() == at::kBFloat16
              && cache.is_contiguous());
  TORCH_CHECK(c_kv.is_contiguous() && c_kv.dtype() == at::kBFloat16);
  TORCH_CHECK(k_pe.stride(-1) == 1 && k_pe.dtype() == at::kBFloat16);
  TORCH_CHECK(slots.dtype() == at::kLong);
  const int T = c_kv.size(0);
  TORCH_CHECK(c_kv.size(1) == R && k_pe.size(1) == P,
              "unsupported MLA cache dims ", c_kv.size(1), "+", k_pe.size(1));
  TORCH_CHECK(cache.size(2) == DT && k_pe.size(0) == T
              && slots.size(0) == T);
  auto stream = at::hip::getCurrentHIPStream();
  if (T == 0) return;
  hipLaunchKernelGGL((mla_cache_write_kernel), dim3(T), dim3(64), 0, stream,
                     (short*)cache.data_ptr(), (const short*)c_kv.data_ptr(),
                     (const short*)k_pe.data_ptr(),
                     slots.data_ptr<int64_t>(), k_pe.stride(0));
}

}  // namespace kaito
