// torch op registration for the "mla" kernel group of kaito_amd's gfx950
// extension (one shared library per group, loaded on first use).
#include <torch/library.h>
#include <ATen/ATen.h>

namespace kaito {
void mla_decode(at::Tensor out, at::Tensor qc, at::Tensor qr, at::Tensor cache,
                at::Tensor block_tables, at::Tensor seq_lens, double scale);
void mla_prepare(at::Tensor q_out, at::Tensor c_out, at::Tensor k_out,
                 at::Tensor cache, at::Tensor q, at::Tensor kv_a, at::Tensor w,
                 double eps, at::Tensor positions, at::Tensor cos_sin,
                 at::Tensor slots);
void mla_prepare_rows(at::Tensor q_out, at::Tensor c_out, at::Tensor k_out,
                      at::Tensor cache, at::Tensor q, at::Tensor kv_a,
                      at::Tensor w, double eps, at::Tensor positions,
                      at::Tensor cos_sin, at::Tensor slots, at::Tensor y,
                      at::Tensor x, at::Tensor wx);
void head_rows(at::Tensor y, at::Tensor x, at::Tensor w);
void mla_cache_write(at::Tensor cache, at::Tensor c_kv, at::Tensor k_pe,
                     at::Tensor slots);
}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("mla_decode(Tensor(a!) out, Tensor qc, Tensor qr, Tensor cache, Tensor block_tables, Tensor seq_lens, float scale) -> ()");
  m.def("mla_prepare(Tensor(a!) q_out, Tensor(b!) c_out, Tensor(c!) k_out, Tensor(d!) cache, Tensor q, Tensor kv_a, Tensor w, float eps, Tensor positions, Tensor cos_sin, Tensor slots) -> ()");
  m.def("mla_prepare_rows(Tensor(a!) q_out, Tensor(b!) c_out, Tensor(c!) k_out, Tensor(d!) cache, Tensor q, Tensor kv_a, Tensor w, float eps, Tensor positions, Tensor cos_sin, Tensor slots, Tensor(e!) y, Tensor x, Tensor wx) -> ()");
  m.def("head_rows(Tensor(a!) y, Tensor x, Tensor w) -> ()");
  m.def("mla_cache_write(Tensor(a!) cache, Tensor c_kv, Tensor k_pe, Tensor slots) -> ()");
}

TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("mla_decode", &kaito::mla_decode);
  m.impl("mla_prepare", &kaito::mla_prepare);
  m.impl("mla_prepare_rows", &kaito::mla_prepare_rows);
  m.impl("head_rows", &kaito::head_rows);
  m.impl("mla_cache_write", &kaito::mla_cache_write);
}
