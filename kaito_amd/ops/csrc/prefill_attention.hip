// Varlen causal attention of whole prompts: queries, keys and values are the
// step's own rows (flash_prefill.h). Replaces vLLM's prefill attention.
#include "flash_prefill.h"
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>

namespace kaito {

namespace {

void check_tiles(const at::Tensor& tile_seq, const at::Tensor& tile_qbase,
                 const at::Tensor& cu) {
  TORCH_CHECK(tile_seq.dtype() == at::kInt && cu.dtype() == at::kInt &&
              tile_qbase.dtype() == at::kInt);
  TORCH_CHECK(tile_seq.is_contiguous() && tile_qbase.is_contiguous() &&
              cu.is_contiguous() && tile_qbase.numel() == tile_seq.numel());
}

}  // namespace

void prefill_attention(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v,
                       at::Tensor tile_seq, at::Tensor tile_qbase,
                       at::Tensor cu_seqlens, double scale, int64_t window,
                       at::Tensor sinks, int64_t longest) {
  flash::Args a{};
  if (sinks.numel() > 0) {
    TORCH_CHECK(sinks.dtype() == at::kFloat && sinks.is_cuda() &&
                sinks.numel() == q.size(1));
    a.sinks = sinks.data_ptr<float>();
  }
  TORCH_CHECK(q.is_cuda() && q.dtype() == at::kBFloat16);
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(q.stride(-1) == 1 && q.stride(1) == q.size(2));
  TORCH_CHECK(k.stride(-1) == 1 && k.stride(1) == k.size(2));
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share row stride");
  check_tiles(tile_seq, tile_qbase, cu_seqlens);
  const int D = q.size(2);
  const int ntiles = tile_seq.size(0);
  a.QH = q.size(1);
  a.KH = k.size(1);
  TORCH_CHECK(a.QH % a.KH == 0);
  if (ntiles == 0) return;
  // keys and values go straight to LDS in 16-byte pieces of their rows
  auto aligned = [](const at::Tensor& t) {
    return (uintptr_t)t.data_ptr() % 16 == 0 && t.stride(0) % 8 == 0;
  };
  if (!aligned(k) || !aligned(v)) {
    k = k.clone(at::MemoryFormat::Contiguous);
    v = v.clone(at::MemoryFormat::Contiguous);
  }
  a.out = (short*)out.data_ptr();
  a.q = (const short*)q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.q_ts = q.stride(0); a.q_hs = D;
  a.k_ts = a.v_ts = k.stride(0); a.k_hs = a.v_hs = D;
  a.tile_seq = tile_seq.data_ptr<int>();
  a.tile_qbase = tile_qbase.data_ptr<int>();
  a.cu = cu_seqlens.data_ptr<int>();
  // Short prompts leave most of a workgroup's 128 rows and 64 keys empty. Up to
  // 32 rows (`longest`, or 0 where it is not known: few rows, and few per
  // tile), a wave per head and 32 keys: one prompt of 32 rows, 32/8 heads of 128,
  // 7.2 -> 4.7 us, 64 of 30 19.5 -> 18.0, 32/32 heads 24.6 -> 18.1. Up to 64,
  // where no heads are flattened and there are more than two workgroups for every
  // CU, two waves (64 of 50, 32/32 heads, 30.1 -> 26.6; one of 50 5.8, 6.2 in
  // two). Heads of 256 are too large for more workgroups per CU; while CUs
  // are idle each gets its own (one of 32 rows, 8/4 heads, 9.2 -> 8.0).
  const int64_t T = q.size(0), pairs = (int64_t)ntiles * a.QH;
  const int gs = flash::group_shift(a.QH, a.KH);
  const bool brief = longest > 0 ? longest <= 32
      : T <= 512 && T <= 32 * (int64_t)ntiles;
  const bool half = longest > 0 && longest <= 64 && gs == 0 && pairs > 512;
  const int waves = D > 128 ? 4 : brief ? 1 : half ? 2 : 4;
  a.gs = brief && (D <= 128 || pairs <= 256) ? 0 : gs;
  a.scale = (float)scale;
  a.window = (int)window;
  auto stream = at::hip::getCurrentHIPStream();
#define PF_LAUNCH(D_, KVT_, NW_)                                              \
  hipLaunchKernelGGL((flash::flash_prefill_kernel<D_, D_, flash::ROWS_BF16,   \
                                                  false, false, false, D_,    \
                                                  KVT_, NW_>),                \
                     dim3(flash::grid_size(a, ntiles, NW_)), dim3(NW_ * 64),  \
                     0, stream, a)
#define PF_CASE(D_)                                                           \
  case D_: if (waves == 1) PF_LAUNCH(D_, 32, 1);                              \
           else if (waves == 2) PF_LAUNCH(D_, 32, 2);                         \
           else PF_LAUNCH(D_, 64, 4);                                         \
           break
  switch (D) {
    case 256: PF_LAUNCH(256, 32, 4); break;
    PF_CASE(128);
    PF_CASE(96);
    PF_CASE(64);
    default: TORCH_CHECK(false, "prefill: unsupported head_dim ", D);
  }
#undef PF_CASE
#undef PF_LAUNCH
}

// Latent attention's whole prompts: keys are 128 dims per head beside 64
// rotated dims that all heads share, values 128 dims per head; each part is
// read where its projection left it.
void mla_prefill_attention(at::Tensor out, at::Tensor q, at::Tensor q_pe,
                           at::Tensor k, at::Tensor k_pe, at::Tensor v,
                           at::Tensor tile_seq, at::Tensor tile_qbase,
                           at::Tensor cu_seqlens, double scale) {
  for (const auto& t : {out, q, q_pe, k, k_pe, v})
    TORCH_CHECK(t.is_cuda() && t.dtype() == at::kBFloat16 &&
                t.stride(-1) == 1 && (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(q.dim() == 3 && q_pe.dim() == 3 && k.dim() == 3 &&
              k_pe.dim() == 2 && v.dim() == 3 && out.is_contiguous());
  const int64_t T = q.size(0), H = q.size(1);
  TORCH_CHECK(q.size(2) == 128 && k.size(2) == 128 && v.size(2) == 128 &&
              q_pe.size(2) == 64 && k_pe.size(1) == 64);
  for (const auto& t : {q_pe, k, v, out})
    TORCH_CHECK(t.size(0) == T && t.size(1) == H);
  TORCH_CHECK(k_pe.size(0) == T && out.size(2) == 128);
  for (const auto& t : {q, q_pe, k, v})
    TORCH_CHECK(t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0);
  TORCH_CHECK(k_pe.stride(0) % 8 == 0);
  check_tiles(tile_seq, tile_qbase, cu_seqlens);
  if (tile_seq.numel() == 0) return;
  flash::Args a{};
  a.QH = a.KH = (int)H;
  a.out = (short*)out.data_ptr();
  a.q = (const short*)q.data_ptr();
  a.q2 = (const short*)q_pe.data_ptr();
  a.k = k.data_ptr();
  a.k2 = (const short*)k_pe.data_ptr();
  a.v = v.data_ptr();
  a.q_ts = q.stride(0); a.q_hs = q.stride(1);
  a.q2_ts = q_pe.stride(0); a.q2_hs = q_pe.stride(1);
  a.k_ts = k.stride(0); a.k_hs = k.stride(1); a.k2_ts = k_pe.stride(0);
  a.v_ts = v.stride(0); a.v_hs = v.stride(1);
  a.tile_seq = tile_seq.data_ptr<int>();
  a.tile_qbase = tile_qbase.data_ptr<int>();
  a.cu = cu_seqlens.data_ptr<int>();
  a.scale = (float)scale;
  hipLaunchKernelGGL((flash::flash_prefill_kernel<192, 128, flash::ROWS_BF16,
                                                  false, false, false, 128>),
                     dim3(flash::grid_size(a, tile_seq.numel())), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), a);
}

}  // namespace kaito
