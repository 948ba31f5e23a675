// Tiles of large products C = X W^T for gfx950 (bf16, f32 sums): the main loop
// behind grouped expert products, SwiGLU products of prompts and latent keys and
// values.
//
// A workgroup of 4 waves (2 over rows x 2 over weight rows), one per SIMD, stays
// and takes one tile after another: 256 x 256, 128 x 128 per wave (FM = FN = 8), 256
// x 128 or 128 x 128. Products are transposed (C^T = W X^T: a lane owns
// one row of X and 4 neighbouring outputs), on v_mfma_f32_16x16x32_bf16.
//
// What bounds large products here is power: the clock drops until the chip stays
// within its budget. Hence (one MI355X, 8192 x 4096 x 14336, where a library product
// reaches 1600 TFLOP/s; 8 waves of 128 x 64 on 32 x 32 tiles, as before: 1180):
//   - 16x16x32 instead of 32x32x16: alone, on random data, 1940 TFLOP/s at 2.0 GHz
//     and 1780 at 1.8 (on zeros 2330 and 2410, at 2.4 and 2.3);
//   - 128 x 128 per wave: a fragment that is read serves 8 products, of 128 x 64 some
//     5.3; LDS is busy 20 % of the time instead of 55;
//   - sums in accumulation registers through inline assembly, by name: with the
//     intrinsic the compiler moved 17 of 64 tiles of sums between the files in
//     every step;
//   - fragments and loads spread evenly between the products (1467 and 1537 with the
//     loads all behind the fragments and evenly), and one loop for all steps: the
//     loads behind the last tile's end have a resource of no bytes.
//
// K steps of 64 go through a ring in LDS, 16-byte chunk c of row r at c ^ (r >> 1 &
// 7): the 16 rows that LDS serves in a cycle lie in different banks. 8 x 8: five
// slots, x and w by turns: when step s begins x(s), w(s), x(s + 1) and w(s + 1) are
// there or under way, x(s + 2) and, behind the barrier that frees a slot, w(s + 2)
// are asked for. Smaller tiles: three or five whole steps. The steps of the next
// tile follow those of the present one: its first are in LDS when its turn comes,
// and the sums of the present one leave through the part that is free then.
#pragma once
#include "common.h"

// The accumulation registers, as a clobber list: see `products`
#define KAITO_SUMS \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", \
  "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", \
  "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", \
  "a30", "a31", "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", \
  "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48", "a49", \
  "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", \
  "a60", "a61", "a62", "a63", "a64", "a65", "a66", "a67", "a68", "a69", \
  "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
  "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", \
  "a90", "a91", "a92", "a93", "a94", "a95", "a96", "a97", "a98", "a99", \
  "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", \
  "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", \
  "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", "a128", "a129", \
  "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", \
  "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", \
  "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
  "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", \
  "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", \
  "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", \
  "a190", "a191", "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", \
  "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", \
  "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", \
  "a220", "a221", "a222", "a223", "a224", "a225", "a226", "a227", "a228", "a229", \
  "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
  "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", \
  "a250", "a251", "a252", "a253", "a254", "a255"

namespace kaito {
namespace tile {

typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));

constexpr int BK = 64;              // K step

struct GemmArgs {
  short* out;                       // [rows, N]
  float* out32;                     // PLAIN_F32: [rows, N] in place of out
  const short* x;                   // [.., K]
  const short* w;                   // [E, rows, K]
  // TWO: outputs from n2 on, of rows x2 (no `rows`) and weights w2, which go to
  // out2 [rows, N - n2]
  const short *x2, *w2, *bias2;
  short* out2;                      // nullptr: to out as the others
  int n2;
  const short* bias;                // [E, rows] or nullptr
  const int* rows;                  // x row of an output row; none: the same
  const int* offsets;               // [.., E + 1]
  int e_base, E, N, K;
  float limit;
};

// rows of a weight: gate and up (SILU, CLAMPED), or one per output
enum Kind { SILU, CLAMPED, RELU2, PLAIN, PLAIN_F32 };
constexpr bool is_gated(int kind) { return kind <= CLAMPED; }

// CLAMPED: min(g, limit) sigmoid(1.702 min(g, limit)) (clamp(u) + 1)
template <int KIND>
KAITO_DEV float gated(float g, float u, float limit) {
  if constexpr (KIND == CLAMPED) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return (u + 1.f) * swish_f32(g, 1.702f);
  }
  return silu_f32(g) * u;
}

// bytes of x behind gathered rows, of weights behind a tile's first
constexpr uint32_t MOST_BYTES = 0xffff0000;
// outputs of a row are fewer: a wave's 128 rows of them, in f32, end below 2^31
constexpr int64_t MOST_OUTPUTS = 1 << 22;

struct Tile {
  int expert, m0, row_end, n0;      // first row, rows' end, first output
};

// 16 bytes per lane from r + lane offset + uniform offset to dst + 16 * lane
KAITO_DEV void buffer_copy16(__amdgpu_buffer_rsrc_t r, short* dst,
                             const uint32_t lane_off, const int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)dst, 16, lane_off, off, 0, 0);
}

// bytes: 0 for a resource from which nothing is read and to which nothing goes
KAITO_DEV __amdgpu_buffer_rsrc_t resource(const void* p, const uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes,
                                           0x27000);
}

constexpr int LDS = 5 * 256 * BK;
// K steps of 32 FM rows and 32 FN weight rows in LDS; 8 x 8: two and a half
template <int FM, int FN> constexpr int stages() {
  return LDS / ((FM + FN) * 32 * BK);
}
// steps that loads are ahead of products; a tile has more than these, if need be
// of zeros
template <int FM, int FN> constexpr int ahead() {
  return FM + FN == 16 ? 2 : stages<FM, FN>() - 1;
}
template <int FN, int KIND> constexpr int columns() {
  return is_gated(KIND) ? 16 * FN : 32 * FN;
}

// Tiles of 32 FM rows x 32 FN weight rows, as next(Tile&) names them until it
// returns false; the same ones for all waves. TWO: n2 is a multiple of 32 FN.
template <int FM, int FN, int KIND, bool TWO, class Next>
KAITO_DEV void stream(const GemmArgs& a, short* lds, Next&& next) {
  constexpr int D = ahead<FM, FN>(), P = FM * FN / 2;   // pairs of products
  constexpr bool GATED = is_gated(KIND);
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int steps = max(a.K / BK, D + 1);
  const int wrows = GATED ? 2 * a.N : a.N;

  // ---- loads. Copy j of a thread fills 16 bytes of row 32 j + its eighth
  const int eighth = threadIdx.x / 8;
  const int chunk = ((threadIdx.x % 8) ^ (eighth >> 1 & 7)) * 8;
  struct {                          // where the loads are; x and w by themselves
    const short *x, *w;
    uint32_t xs[FM], ws[FN];
    int k, bytes;                   // 0 bytes: nothing is read, LDS gets zeros
  } at;
  // rows that do not exist are beyond the resource's end: zeros, unread
  constexpr int BYTES = (int)MOST_BYTES;
  constexpr uint32_t NOWHERE = 0xffffff00;
  // dims from k on, or, from the tile's end on, none
  auto seek = [&](const int k, const int some) {
    at.bytes = __builtin_amdgcn_readfirstlane(some & (k - a.K) >> 31 & BYTES);
    at.k = k & at.bytes >> 31;
  };
  auto row_of = [&](const Tile& t, const int j) {
    return min(j * 32 + eighth, t.row_end - 1 - t.m0);
  };
  auto aim_w = [&](const Tile& t) {
    at.w = TWO && t.n0 >= a.n2
        ? a.w2 + (int64_t)(t.n0 - a.n2) * a.K
        : a.w + ((int64_t)t.expert * wrows + t.n0) * a.K;
#pragma unroll
    for (int j = 0; j < FN; j++) {
      // gated: every 32 tile rows are 16 gate rows, then their up rows
      const int n = GATED ? j * 16 + eighth % 16 : j * 32 + eighth;
      const uint32_t row = n + (GATED && eighth >= 16 ? a.N : 0);
      at.ws[j] = t.n0 + n < a.N ? (row * a.K + chunk) * 2 : NOWHERE;
    }
  };
  auto aim_x = [&](const Tile& t, const int (&src)[FM]) {
    at.x = a.rows ? a.x
        : (TWO && t.n0 >= a.n2 ? a.x2 : a.x) + (int64_t)t.m0 * a.K;
#pragma unroll
    for (int j = 0; j < FM; j++)
      at.xs[j] = j * 32 + eighth < t.row_end - t.m0
          ? ((uint32_t)src[j] * a.K + chunk) * 2 : NOWHERE;
  };
  auto rows_of = [&](const Tile& t, int (&src)[FM]) {
#pragma unroll
    for (int j = 0; j < FM; j++) src[j] = row_of(t, j);
    if (a.rows) {
#pragma unroll
      for (int j = 0; j < FM; j++) src[j] = a.rows[t.m0 + src[j]];
    }
  };
  auto load = [&](const bool is_x, short* slot, const int j) {
    buffer_copy16(resource(is_x ? at.x : at.w, (uint32_t)at.bytes),
                  slot + (j * 256 + wave * 64) * 8,
                  is_x ? at.xs[j] : at.ws[j], at.k * 2);
  };

  // ---- fragments: rows 16 n of x or w, dims 32 kk + 8 hi of K
  hbf16x8 wf[2][FN], xf[2][FM];
  const int place0 = (hi ^ (lo >> 1 & 7)) * 8, place1 = place0 ^ 32;
  const int x_at = (wm * FM * 16 + lo) * BK, w_at = (wn * FN * 16 + lo) * BK;
  // in the order in which products need them: x's first, all of w, the rest
  auto read = [&](const short* xs, const short* ws, const int kk, const int n) {
    const int c = kk ? place1 : place0;
    if (n >= 1 && n <= FN)
      wf[kk][n - 1] = *reinterpret_cast<const hbf16x8*>(
          ws + w_at + c + (n - 1) * 16 * BK);
    else
      xf[kk][n ? n - FN : 0] = *reinterpret_cast<const hbf16x8*>(
          xs + x_at + c + (n ? n - FN : 0) * 16 * BK);
  };
  // Sums of weight rows 16 i and x rows 16 j are a[4 (FN j + i)] to the third
  // behind, by name: left to the compiler, they moved. Every statement that names
  // one clobbers all, so that no value of the compiler's outlives a statement there;
  // that none lives between two either is looked at in what was built
  // (tests/test_tile_linear.py). Fragments come from LDS alone, so that no product
  // follows a vector instruction that writes its operands.
  auto fence = [&] { asm volatile("" ::: KAITO_SUMS); };
  auto products = [&](const int kk, const int j, const int i0, const int i1,
                      const bool first) {
    const int a0 = 4 * (FN * j + i0), a1 = 4 * (FN * j + i1);
    if (first)                      // known where this is inlined
      asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %4, %6, 0\n\t"
                   "v_mfma_f32_16x16x32_bf16 a[%2:%3], %5, %6, 0"
                   :: "n"(a0), "n"(a0 + 3), "n"(a1), "n"(a1 + 3),
                      "v"(wf[kk][i0]), "v"(wf[kk][i1]), "v"(xf[kk][j])
                   : KAITO_SUMS);
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %4, %6, a[%0:%1]\n\t"
                   "v_mfma_f32_16x16x32_bf16 a[%2:%3], %5, %6, a[%2:%3]"
                   :: "n"(a0), "n"(a0 + 3), "n"(a1), "n"(a1 + 3),
                      "v"(wf[kk][i0]), "v"(wf[kk][i1]), "v"(xf[kk][j])
                   : KAITO_SUMS);
  };
  auto settle = [&] {               // the last products' results are there
    asm volatile("s_nop 15\n\ts_nop 15" ::: KAITO_SUMS);
  };
  auto sum = [&](const int i, const int j, const int e) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]"
                 : "=v"(v) : "n"(4 * (FN * j + i) + e) : KAITO_SUMS);
    return v;
  };

  // where x and w of the step i behind the present one are. 8 x 8: five slots, x
  // and w by turns; else whole steps
  constexpr bool TURNS = FM + FN == 16;
  constexpr int RING = TURNS ? 5 : stages<FM, FN>(), STRIDE = TURNS ? 2 : 1;
  constexpr int SLOT = TURNS ? 256 * BK : (FM + FN) * 32 * BK;
  static_assert(!TURNS || FM == FN);
  int slot = 0;
  auto nth = [&](const int i) {
    return lds + (slot + i < RING ? slot + i : slot + i - RING) * SLOT;
  };
  auto x_of = [&](const int i) { return nth(STRIDE * i); };
  auto w_of = [&](const int i) {
    return TURNS ? nth(STRIDE * i + 1) : nth(STRIDE * i) + FM * 32 * BK;
  };
  // products of one half of a step; beside them the fragments of the next half
  // and the loads of one operand of one step
  auto half = [&](const int kk, const short* xs, const short* ws, short* to,
                  const bool first) {
    constexpr int R = FM + FN;
    const int L = kk == 0 ? FM : FN;
    fence();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < P; p++) {
      const int j = p / (FN / 2), q = p % (FN / 2);
      const int i = j & 1 ? FN - 1 - 2 * q : 2 * q;
      products(kk, j, i, j & 1 ? i - 1 : i + 1, first);
      // early ahead of the barrier, which waits for them
      const int per = kk == 0 && 2 * R <= P ? P / 2 : P;
#pragma unroll
      for (int n = 0; n < R; n++)
        if (n * per / R == p) read(xs, ws, kk ^ 1, n);
      if (p % (P / L) == (P / L > 1)) load(kk == 0, to, p / (P / L));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // own reads done and own loads landed but for the newest, of x D - 1 steps and
  // of w D - 2: all's. A tile's first step does not wait for the stores of the one before,
  // as many for any rows, that lie between.
  constexpr int NO = GATED ? FN / 2 : FN;           // 16-output blocks of a wave
  constexpr int WC = NO * 16, CH = WC / 8;          // outputs, chunks of a row
  constexpr int NR = 16 * CH / 64;                  // 16-byte reads per 16 rows
  constexpr bool F32 = KIND == PLAIN_F32;
  auto meet = [&](const bool behind_stores) {
    constexpr int N = (D - 1) * FM + (D - 2) * FN;
    constexpr int M = N + (F32 ? 0 : FM * NR);
    static_assert(M < 64);
    if (behind_stores)
      __builtin_amdgcn_s_waitcnt(0x0070 | (M & 15) | ((M >> 4) << 14));
    else
      __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  auto follow = [&](Tile& t) {
    Tile u{};
    const bool some = next(u);
    t.expert = __builtin_amdgcn_readfirstlane(u.expert);
    t.m0 = __builtin_amdgcn_readfirstlane(u.m0);
    t.row_end = __builtin_amdgcn_readfirstlane(u.row_end);
    t.n0 = __builtin_amdgcn_readfirstlane(u.n0);
    return (bool)__builtin_amdgcn_readfirstlane(some);
  };
  Tile cur, nxt;
  if (!follow(cur)) return;
  int src[FM];
  rows_of(cur, src);
  auto load_x = [&](const int s) {
    seek(s * BK, -1);
#pragma unroll
    for (int j = 0; j < FM; j++) load(true, x_of(s), j);
  };
  auto load_w = [&](const int s) {
    seek(s * BK, -1);
#pragma unroll
    for (int j = 0; j < FN; j++) load(false, w_of(s), j);
  };
  // weights while the numbers of the rows are on their way
  aim_w(cur);
  load_w(0);
  load_w(1);
  aim_x(cur, src);
  load_x(0);
  load_x(1);
#pragma unroll
  for (int s = 2; s < D; s++) {
    load_w(s);
    load_x(s);
  }
  seek(D * BK, -1);
  {
    constexpr int N = FM + (D - 2) * (FM + FN);     // behind x(0)
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int n = 0; n < FM + FN; n++) read(x_of(0), w_of(0), 0, n);

  for (bool stored = false;; stored = true) {
    const bool more = follow(nxt);
    if (more) rows_of(nxt, src);
    auto step = [&](const int s, const bool first) {
      half(0, x_of(0), w_of(0), x_of(D), first);
      meet(first && stored);
      slot = slot + STRIDE < RING ? slot + STRIDE : slot + STRIDE - RING;
      half(1, x_of(0), w_of(0), w_of(D - 1), false);
      seek(at.k + BK, at.bytes);
      if (s == steps - 1 - D && more) {   // the rest of this tile is on its way
        aim_w(nxt);
        aim_x(nxt, src);
        seek(0, -1);
      }
    };
    step(0, true);
    for (int s = 1; s < steps; s++) step(s, false);
    settle();

    // ---- outputs 16 i + 4 hi + e of x row 16 j + lo. bf16 rows pass through
    // this wave's part of the slot that the next step's loads fill first: the
    // same kilobytes that its own copies go to
    constexpr int RPP = 512 / WC;                   // rows in a kilobyte
    const bool apart = TWO && a.out2 && cur.n0 >= a.n2;
    // columns of the rows written, this wave's first one of them
    const int N = apart ? a.N - a.n2 : TWO && a.out2 ? a.n2 : a.N;
    const int c0 = cur.n0 + wn * WC - (apart ? a.n2 : 0);
    const int64_t first_row = cur.m0 + wm * FM * 16;
    // rows of this wave that exist: their bytes, and not all that follow, have to
    // stay below BEYOND
    const int live = min(cur.row_end - (int)first_row, FM * 16);
    constexpr int SIZE = F32 ? 4 : 2;
    // rows and columns that do not exist lie beyond the resource's end
    const auto ro = resource(
        F32 ? (void*)(a.out32 + first_row * N + c0)
            : (void*)((apart ? a.out2 : a.out) + first_row * N + c0),
        live > 0 && c0 < N ? ((live - 1) * N + min(WC, N - c0)) * SIZE : 0);
    constexpr int BEYOND = 0x80000000;
    char* slab = (char*)(x_of(D) + wave * 512);
    auto slab_at = [&](const int row, const int c) {
      return row / RPP * 4096 + row % RPP * WC * 2 +
          (c ^ (CH == 16 ? row : row >> (CH == 8 ? 1 : 2)) % CH) * 16;
    };
    const int write0 = slab_at(lo, hi / 2) + hi % 2 * 8;
    int from[NR], to[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int row = (r * 64 + lane) / CH, c = lane % CH;
      from[r] = slab_at(row, c);
      to[r] = c0 + c * 8 < N ? (row * N + c * 8) * 2 : BEYOND;
    }
    typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
    const short* bias = apart ? a.bias2
        : a.bias ? a.bias + (int64_t)cur.expert * wrows : nullptr;
    auto outputs = [&](const bool biased) {
      const short* be = bias + c0 + 4 * hi;
      short4_t b[GATED ? 2 : 1][NO];
      if (biased) {
#pragma unroll
        for (int i = 0; i < NO; i++)
#pragma unroll
          for (int g = 0; g < (GATED ? 2 : 1); g++) {
            b[g][i] = short4_t{0, 0, 0, 0};
            if (c0 + i * 16 < N)
              b[g][i] =
                  *reinterpret_cast<const short4_t*>(be + g * a.N + i * 16);
          }
      }
      u32x4 rows[NR];
      auto store = [&](const int j) {
#pragma unroll
        for (int r = 0; r < NR; r++)
          __builtin_amdgcn_raw_buffer_store_b128(
              rows[r], ro, to[r] + j * 32 * N, 0, 0);
      };
#pragma unroll
      for (int j = 0; j < FM; j++) {
        // one row block's sums at a time are in vector registers
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NO; i++) {
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            v[e] = sum(GATED ? 2 * i : i, j, e);
            if (biased) v[e] += bf16_to_f32(b[0][i][e]);
            if constexpr (GATED) {
              float u = sum(2 * i + 1, j, e);
              if (biased) u += bf16_to_f32(b[1][i][e]);
              v[e] = gated<KIND>(v[e], u, a.limit);
            } else if constexpr (KIND == RELU2) {
              v[e] = fmaxf(v[e], 0.f);
              v[e] *= v[e];
            }
          }
          if constexpr (F32) {
            __builtin_amdgcn_raw_buffer_store_b128(
                __builtin_bit_cast(u32x4, v), ro,
                c0 + i * 16 < N
                    ? ((j * 16 + lo) * N + i * 16 + 4 * hi) * 4 : BEYOND,
                0, 0);
          } else {
            *reinterpret_cast<short4_t*>(slab + (write0 ^ i * 32)) =
                short4_t{f32_to_bf16(v[0]), f32_to_bf16(v[1]),
                         f32_to_bf16(v[2]), f32_to_bf16(v[3])};
          }
        }
        if constexpr (F32) continue;
        // LDS serves a wave in order: no wait between writes and reads; rows
        // leave when the next ones are on their way there
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
        if (j > 0) store(j - 1);
#pragma unroll
        for (int r = 0; r < NR; r++)
          rows[r] = *reinterpret_cast<const u32x4*>(slab + from[r]);
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (!F32) store(FM - 1);
    };
    if (bias) outputs(true);
    else outputs(false);
    if (!more) break;
    cur = nxt;
    // this wave's reads of the slab are done before its copies overwrite it
    __builtin_amdgcn_s_waitcnt(0xc07f);             // lgkmcnt(0)
  }
  // no copy is left under way for what uses LDS next
  __builtin_amdgcn_s_waitcnt(0x0070);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

constexpr int NG = 4;               // column tiles that share row tiles
constexpr int CUS = 256;            // 8 XCDs of 32

// What a round of tiles of a shape takes, beside those of the others; quarters are
// small tiles
struct Rounds {
  int large, wide, tall, small;
};

// A launch of CUS workgroups, one per CU: all tiles of a product, of the shape that
// takes least time. Of each shape: `share` tiles per XCD, `here` on this one, tile
// i of those by number. Tiles of 256 x 256, those of a small last round in quarters,
// or of 128 x 256, 256 x 128 or 128 x 128.
template <int KIND, bool TWO = false, class Large, class Wide, class Tall,
          class Small>
KAITO_DEV void run(const GemmArgs& a, short* lds, const Rounds takes,
                   const Large& large, const Wide& wide, const Tall& tall,
                   const Small& small) {
  constexpr int workers = CUS / 8;
  enum { LARGE, WIDE, TALL, SMALL };
  auto rounds = [&](const int n) { return (n + workers - 1) / workers; };
  // of n tiles, those that are cut in quarters
  auto last = [&](const int n) {
    const int rest = n % workers;
    return 4 * rest > workers * (n < workers ? 2 : 1) ? 0 : rest;
  };
  // the same answer on all XCDs, whose tiles are numbered through
  const int over = last(large.share);
  int best = takes.large * rounds(large.share - over) +
             takes.small * rounds(4 * over);
  int mode = LARGE;
  auto other = [&](const int m, const int cost) {
    if (cost < best) best = cost, mode = m;
  };
  other(WIDE, takes.wide * rounds(wide.share));
  other(TALL, takes.tall * rounds(tall.share));
  other(SMALL, takes.small * rounds(small.share));
  const int rest = last(large.here);
  int i = blockIdx.x / 8;
  auto all = [&](const auto& tiles, const int end) {
    return [&, end](Tile& t) {
      if (i >= end) return false;
      t = tiles(i);
      i += workers;
      return true;
    };
  };
  if (mode == LARGE) stream<8, 8, KIND, TWO>(a, lds, all(large, large.here - rest));
  if (mode == WIDE) {
    stream<4, 8, KIND, TWO>(a, lds, all(wide, wide.here));
  } else if (mode == TALL) {
    stream<8, 4, KIND, TWO>(a, lds, all(tall, tall.here));
  } else {
    i = blockIdx.x / 8;
    const int end = mode == LARGE ? 4 * rest : small.here;
    stream<4, 4, KIND, TWO>(a, lds, [&](Tile& t) {
      for (; i < end; i += workers) {
        if (mode == LARGE) {
          t = large(large.here - rest + i / 4);
          t.m0 += i % 4 / 2 * (large.BM / 2);
          t.n0 += i % 2 * (large.COLS / 2);
          if (t.m0 >= t.row_end || t.n0 >= a.N) continue;
        } else {
          t = small(i);
        }
        i += workers;
        return true;
      }
      return false;
    });
  }
}

}  // namespace tile
}  // namespace kaito
