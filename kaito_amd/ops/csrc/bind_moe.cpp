// torch op registration for the "moe" kernel group of kaito_amd's gfx950
// extension (one shared library per group, loaded on first use).
#include <torch/library.h>
#include <ATen/ATen.h>

namespace kaito {
void moe_gate_silu(at::Tensor act, at::Tensor x, at::Tensor w_gate_up,
                   at::Tensor sorted_ids, at::Tensor offsets, at::Tensor bias,
                   int64_t act_mode, int64_t e_base, int64_t n_local_experts,
                   double act_limit);
void moe_down_rows(at::Tensor y, at::Tensor act, at::Tensor w_down,
                   at::Tensor offsets, at::Tensor bias, int64_t e_base,
                   int64_t n_local_experts);
void moe_up_pairs(at::Tensor act, at::Tensor x, at::Tensor w_gate_up,
                  at::Tensor topi, at::Tensor bias, int64_t act_mode,
                  int64_t n_experts, int64_t e_base, int64_t n_local_experts,
                  double act_limit, at::Tensor all_w, at::Tensor all_act);
void moe_down_pairs(at::Tensor y, at::Tensor act, at::Tensor w_down,
                    at::Tensor topi, at::Tensor bias, int64_t n_experts,
                    int64_t e_base, int64_t n_local_experts, at::Tensor all_w,
                    at::Tensor all_act, at::Tensor all_y);
}  // namespace kaito

TORCH_LIBRARY_FRAGMENT(kaito, m) {
  m.def("moe_gate_silu(Tensor(a!) act, Tensor x, Tensor w_gate_up, Tensor sorted_ids, Tensor offsets, Tensor bias, int act_mode, int e_base, int n_local_experts, float act_limit) -> ()");
  m.def("moe_down_rows(Tensor(a!) y, Tensor act, Tensor w_down, Tensor offsets, Tensor bias, int e_base, int n_local_experts) -> ()");
  m.def("moe_up_pairs(Tensor(a!) act, Tensor x, Tensor w_gate_up, Tensor topi, Tensor bias, int act_mode, int n_experts, int e_base, int n_local_experts, float act_limit, Tensor all_w, Tensor(b!) all_act) -> ()");
  m.def("moe_down_pairs(Tensor(a!) y, Tensor act, Tensor w_down, Tensor topi, Tensor bias, int n_experts, int e_base, int n_local_experts, Tensor all_w, Tensor all_act, Tensor(b!) all_y) -> ()");
}

TORCH_LIBRARY_IMPL(kaito, CUDA, m) {
  m.impl("moe_gate_silu", &kaito::moe_gate_silu);
  m.impl("moe_down_rows", &kaito::moe_down_rows);
  m.impl("moe_up_pairs", &kaito::moe_up_pairs);
  m.impl("moe_down_pairs", &kaito::moe_down_pairs);
}
