// Entry of the paged-attention decode kernel (paged_decode.h) for rotary models:
// one row per sequence, lengths on the device.
#include "paged_decode.h"
#include <torch/library.h>

namespace kaito {

void paged_attention_sp(at::Tensor out, at::Tensor query, at::Tensor k_cache,
                        at::Tensor v_cache, at::Tensor block_tables,
                        at::Tensor seq_lens, double scale, int64_t window,
                        at::Tensor sinks) {
  DecodeArgs a{};
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
  const bool fp8 = k_cache.dtype() == at::kByte;   // OCP e4m3 KV cache
  const int T = query.size(0);
  const int D = query.size(2);
  a.KH = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == BS, "block_size must be 16");
  TORCH_CHECK(query.size(1) % a.KH == 0);
  a.G = query.size(1) / a.KH;
  a.max_blocks = block_tables.size(1);
  if (T == 0) return;
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
#define PA_DIM(D_)                                                            \
  if (D == D_) {                                                              \
    if (fp8) launch_paged_decode<D_, true, false>(a, out, T);                 \
    else launch_paged_decode<D_, false, false>(a, out, T);                    \
    return;                                                                   \
  }
  PA_DIM(64) PA_DIM(128) PA_DIM(256)
#undef PA_DIM
}

}  // namespace kaito
