// Linear layers of prompts on the tiles of tile_gemm.h:
//
//   tile_linear   out = x W^T, for vocabularies and for products whose large tiles
//                 fill no whole number of rounds
//   tile_swiglu   out = silu(x Wg^T) (x Wu^T) of W = [Wg | Wu]
//   tile_pair     out = x W^T (+ bias), out2 = x2 W2^T (+ bias2): one launch, whose
//                 last round of tiles is not each product's own
//
// A SwiGLU pair as a library product and a pass over its rows moves 6 bytes per
// output more, and rounds gate and up to bf16 on the way.
#include "tile_gemm.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPFunctions.h>

namespace kaito {

namespace {

using tile::GemmArgs;
using tile::Tile;

// Tiles of 32 FM x 32 FN, in blocks of NG column tiles x all row tiles, column
// fastest; every XCD takes one contiguous eighth
template <int FM, int FN, int KIND>
struct Tiles {
  static constexpr int BM = 32 * FM, COLS = tile::columns<FN, KIND>();
  int T, ntiles, mtiles, share, at, here;

  KAITO_DEV Tiles(const GemmArgs& a, const int T)
      : T(T), ntiles((a.N + COLS - 1) / COLS), mtiles((T + BM - 1) / BM) {
    const int total = ntiles * mtiles;
    share = (total + 7) / 8;
    at = blockIdx.x % 8 * share;
    here = max(min(share, total - at), 0);
  }
  KAITO_DEV Tile operator()(int t) const {
    t += at;
    const int blk = t / (tile::NG * mtiles);
    const int wide = min(tile::NG, ntiles - blk * tile::NG);
    const int in_blk = t - blk * tile::NG * mtiles;
    return {0, in_blk / wide * BM, T,
            (blk * tile::NG + in_blk % wide) * COLS};
  }
};

// where weights and rows come from the caches (K = 2048: 50 us for a large one, 18
// for a small one); ops/__init__.py `_tile_plan` counts with the same
constexpr tile::Rounds TAKES = {5, 3, 3, 2};

template <int KIND, bool TWO>
__global__ __launch_bounds__(256, 1) void tile_linear_kernel(const GemmArgs a,
                                                             const int T) {
  __shared__ __attribute__((aligned(1024))) short lds[tile::LDS];
  tile::run<KIND, TWO>(a, lds, TAKES, Tiles<8, 8, KIND>(a, T),
                       Tiles<4, 8, KIND>(a, T), Tiles<8, 4, KIND>(a, T),
                       Tiles<4, 4, KIND>(a, T));
}

}  // namespace

static void check(const at::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.is_contiguous() &&
              t.get_device() == c10::hip::current_device() &&
              t.dtype() == at::kBFloat16 && (uintptr_t)t.data_ptr() % 16 == 0);
}

// what all take: out [T, N], x [T, K], w [rows, K]
static GemmArgs tile_args(const at::Tensor& out, const at::Tensor& x,
                          const at::Tensor& w, int64_t rows) {
  check(out); check(x); check(w);
  const int64_t T = x.size(0), K = x.size(1);
  TORCH_CHECK(out.size(0) == T && w.size(0) == rows && w.size(1) == K &&
              K % tile::BK == 0 && out.size(1) % 64 == 0 && K > 0 &&
              K < (1 << 22) && T < (1 << 24) && rows < tile::MOST_OUTPUTS &&
              w.numel() * 2 <= tile::MOST_BYTES);
  GemmArgs a{};
  a.out = (short*)out.data_ptr();
  a.x = (const short*)x.data_ptr();
  a.w = (const short*)w.data_ptr();
  a.E = 1;
  a.N = (int)out.size(1);
  a.K = (int)K;
  return a;
}

static const short* bias_of(const at::Tensor& bias, int64_t N) {
  if (bias.numel() == 0) return nullptr;
  TORCH_CHECK(bias.is_cuda() && bias.is_contiguous() && bias.numel() == N &&
              bias.dtype() == at::kBFloat16 &&
              (uintptr_t)bias.data_ptr() % 8 == 0);
  return (const short*)bias.data_ptr();
}

template <int KIND, bool TWO>
static void launch(const GemmArgs& a, int64_t T) {
  if (T == 0 || a.N == 0) return;
  hipLaunchKernelGGL((tile_linear_kernel<KIND, TWO>), dim3(tile::CUS), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), a, (int)T);
}

void tile_linear(at::Tensor out, at::Tensor x, at::Tensor w) {
  GemmArgs a = tile_args(out, x, w, out.size(1));
  a.n2 = a.N;                       // no second product
  launch<tile::PLAIN, true>(a, x.size(0));
}

// w [2 N, K]
void tile_swiglu(at::Tensor out, at::Tensor x, at::Tensor w) {
  launch<tile::SILU, false>(tile_args(out, x, w, 2 * out.size(1)), x.size(0));
}

// the first product's outputs in multiples of 256
void tile_pair(at::Tensor out, at::Tensor x, at::Tensor w, at::Tensor bias,
               at::Tensor out2, at::Tensor x2, at::Tensor w2,
               at::Tensor bias2) {
  GemmArgs a = tile_args(out, x, w, out.size(1));
  const GemmArgs b = tile_args(out2, x2, w2, out2.size(1));
  TORCH_CHECK(a.N % 256 == 0 && a.N > 0 && b.N > 0 &&
              x2.sizes() == x.sizes());
  a.bias = bias_of(bias, a.N);
  a.bias2 = bias_of(bias2, b.N);
  a.x2 = b.x;
  a.w2 = b.w;
  a.out2 = b.out;
  a.n2 = a.N;
  a.N += b.N;
  launch<tile::PLAIN, true>(a, x.size(0));
}

}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("tile_linear(Tensor(a!) out, Tensor x, Tensor w) -> ()");
  m.def("tile_swiglu(Tensor(a!) out, Tensor x, Tensor w) -> ()");
  m.def("tile_pair(Tensor(a!) out, Tensor x, Tensor w, Tensor bias, Tensor(b!) out2, Tensor x2, Tensor w2, Tensor bias2) -> ()");
}
TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("tile_linear", &kaito::tile_linear);
  m.impl("tile_swiglu", &kaito::tile_swiglu);
  m.impl("tile_pair", &kaito::tile_pair);
}
