// Entry of the paged-attention decode kernel (paged_decode.h) for rotary models:
// one row per sequence, lengths on the device.
#include "paged_decode.h"
#include <torch/library.h>

namespace kaito {

namespace {

// what every call has; false: there are no rows
bool decode_args(DecodeArgs& a, const at::Tensor& out, const at::Tensor& query,
                 const at::Tensor& k_cache, const at::Tensor& v_cache,
                 const at::Tensor& block_tables, const at::Tensor& seq_lens,
                 double scale, int64_t window, const at::Tensor& sinks) {
  if (sinks.numel() > 0) {
    TORCH_CHECK(sinks.dtype() == at::kFloat && sinks.is_cuda() &&
                sinks.numel() == query.size(1));
    a.sinks = sinks.data_ptr<float>();
  }
  TORCH_CHECK(query.is_cuda() && query.dtype() == at::kBFloat16);
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(query.stride(-1) == 1 && query.stride(1) == query.size(2),
              "query must be [T, QH, D] with contiguous heads");
  TORCH_CHECK(block_tables.dtype() == at::kInt && seq_lens.dtype() == at::kInt);
  const int D = query.size(2);
  a.KH = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == BS, "block_size must be 16");
  TORCH_CHECK(query.size(1) % a.KH == 0);
  a.G = query.size(1) / a.KH;
  a.max_blocks = block_tables.size(1);
  if (query.size(0) == 0) return false;
  const bool group_ok = D == 128 ? a.G >= 1 && a.G <= 8
      : D == 64 ? a.G == 1 || a.G == 2 || a.G == 4 || a.G == 8
                : a.G == 1 || a.G == 2 || a.G == 4;
  TORCH_CHECK(D == 64 || D == 128 || D == 256, "unsupported head_dim ", D);
  TORCH_CHECK(group_ok, "unsupported GQA group ", a.G);
  a.out = (short*)out.data_ptr();
  a.q = (const short*)query.data_ptr();
  a.k = k_cache.data_ptr();
  a.v = v_cache.data_ptr();
  a.block_tables = block_tables.data_ptr<int>();
  a.seq_lens = seq_lens.data_ptr<int>();
  a.scale = (float)scale;
  a.q_stride = query.stride(0);
  a.window = (int)window;
  return true;
}

template <bool ROPE>
void launch(const DecodeArgs& a, const at::Tensor& out, int T, int D, bool fp8) {
#define PA_DIM(D_)                                                            \
  if (D == D_) {                                                              \
    if (fp8) launch_paged_decode<D_, true, false, ROPE>(a, out, T);           \
    else launch_paged_decode<D_, false, false, ROPE>(a, out, T);              \
    return;                                                                   \
  }
  PA_DIM(64) PA_DIM(128) PA_DIM(256)
#undef PA_DIM
}

}  // namespace

void paged_attention_sp(at::Tensor out, at::Tensor query, at::Tensor k_cache,
                        at::Tensor v_cache, at::Tensor block_tables,
                        at::Tensor seq_lens, double scale, int64_t window,
                        at::Tensor sinks) {
  DecodeArgs a{};
  if (decode_args(a, out, query, k_cache, v_cache, block_tables, seq_lens,
                  scale, window, sinks))
    launch<false>(a, out, query.size(0), query.size(2),
                  k_cache.dtype() == at::kByte);    // OCP e4m3 pages
}

// rope_and_cache and paged_attention_sp in one launch: rows of one sequence each,
// whose own key is the last of seq_lens. q, k and v stay as they are.
void rope_paged_attention(at::Tensor out, at::Tensor positions,
                          at::Tensor query, at::Tensor k, at::Tensor v,
                          at::Tensor cos_sin, at::Tensor k_cache,
                          at::Tensor v_cache, at::Tensor slots,
                          at::Tensor block_tables, at::Tensor seq_lens,
                          double scale, int64_t window, at::Tensor sinks) {
  DecodeArgs a{};
  if (!decode_args(a, out, query, k_cache, v_cache, block_tables, seq_lens,
                   scale, window, sinks))
    return;
  const int64_t T = query.size(0), D = query.size(2);
  for (const auto& t : {k, v})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 && t.dim() == 2 &&
                t.stride(1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0 &&
                (T == 1 || t.stride(0) % 8 == 0) && t.size(0) == T &&
                t.size(1) == a.KH * D);
  TORCH_CHECK(out.sizes() == query.sizes() && (T == 1 || a.q_stride % 8 == 0) &&
              (uintptr_t)query.data_ptr() % 16 == 0);
  TORCH_CHECK(positions.dtype() == at::kLong && positions.numel() == T &&
              positions.is_contiguous() && slots.dtype() == at::kLong &&
              slots.numel() == T && slots.is_contiguous());
  TORCH_CHECK(cos_sin.dtype() == at::kFloat && cos_sin.is_contiguous() &&
              cos_sin.size(1) == D && (uintptr_t)cos_sin.data_ptr() % 16 == 0);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              k_cache.dtype() == v_cache.dtype() && k_cache.size(3) == D &&
              k_cache.sizes() == v_cache.sizes());
  const bool fp8 = k_cache.dtype() == at::kByte;
  TORCH_CHECK(fp8 || k_cache.dtype() == at::kBFloat16);
  a.positions = positions.data_ptr<int64_t>();
  a.k_row = (const short*)k.data_ptr();
  a.v_row = (const short*)v.data_ptr();
  a.k_stride = k.stride(0);
  a.v_stride = v.stride(0);
  a.cos_sin = cos_sin.data_ptr<float>();
  a.slots = slots.data_ptr<int64_t>();
  launch<true>(a, out, (int)T, (int)D, fp8);
}

}  // namespace kaito
