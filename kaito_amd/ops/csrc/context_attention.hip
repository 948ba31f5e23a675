// Paged CONTEXT prefill attention: varlen causal attention where Q covers
// only the SUFFIX tokens of each sequence and K/V are read from the paged
// cache (which already holds the full context including the suffix).
// Enables chunked prefill and partial prefix-cache restore. Causal rule: q
// row qi (0-based within the suffix) has absolute position kv_len - q_len +
// qi and attends kv positions <= it. The kernel is flash_prefill.h's, its
// tiles gathered through the block table.
#include "flash_prefill.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

void context_attention(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor tile_seq,
                       at::Tensor tile_qbase, at::Tensor cu_seqlens_q,
                       at::Tensor kv_lens, at::Tensor block_tables,
                       double scale, int64_t window, at::Tensor sinks) {
  flash::Args a{};
  if (sinks.numel() > 0) {
    TORCH_CHECK(sinks.dtype() == at::kFloat && sinks.is_cuda() &&
                sinks.numel() == q.size(1));
    a.sinks = sinks.data_ptr<float>();
  }
  TORCH_CHECK(q.is_cuda() && q.dtype() == at::kBFloat16);
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.stride(-1) == 1 && q.stride(1) == q.size(2));
  const int D = q.size(2);
  const int ntiles = tile_seq.size(0);
  a.QH = q.size(1);
  a.KH = k_cache.size(1);
  a.BS = k_cache.size(2);
  a.max_blocks = block_tables.size(1);
  TORCH_CHECK(a.BS == 16 && (D == 128 || D == 64 || D == 256),
              "context attn: D 64/128/256");
  if (ntiles == 0) return;
  a.out = (short*)out.data_ptr();
  a.q = (const short*)q.data_ptr();
  a.k = k_cache.data_ptr();
  a.v = v_cache.data_ptr();
  a.q_ts = q.stride(0); a.q_hs = D;
  a.tile_seq = tile_seq.data_ptr<int>();
  a.tile_qbase = tile_qbase.data_ptr<int>();
  a.cu = cu_seqlens_q.data_ptr<int>();
  a.kv_lens = kv_lens.data_ptr<int>();
  a.block_tables = block_tables.data_ptr<int>();
  a.gs = flash::group_shift(a.QH, a.KH);
  a.scale = (float)scale;
  a.window = (int)window;
  const bool fp8 = k_cache.dtype() == at::kByte;
  const dim3 grid(flash::grid_size(a, ntiles));
  auto stream = at::hip::getCurrentHIPStream();
#define CTX_LAUNCH(D_)                                                        \
  do {                                                                        \
    if (fp8)                                                                  \
      hipLaunchKernelGGL((flash::flash_prefill_kernel<D_, D_,                 \
                              flash::PAGED_FP8, false>),                      \
                         grid, dim3(256), 0, stream, a);                      \
    else                                                                      \
      hipLaunchKernelGGL((flash::flash_prefill_kernel<D_, D_,                 \
                              flash::PAGED_BF16, false>),                     \
                         grid, dim3(256), 0, stream, a);                      \
  } while (0)
  if (D == 128) CTX_LAUNCH(128);
  else if (D == 256) CTX_LAUNCH(256);
  else CTX_LAUNCH(64);
#undef CTX_LAUNCH
}

}  // namespace kaito
