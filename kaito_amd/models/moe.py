"""Mixture-of-experts FFN (Mixtral / Qwen-MoE / gpt-oss class).

Replaces vLLM's fused-MoE CUDA path for the MoE presets in the reference
catalog (gpt-oss-120b / Qwen MoE presets in
supported_models.yaml).

The GPU path needs no host read: two launches choose the experts and, beyond
small steps of few experts, sort the (token, expert) pairs by expert
(ops/csrc/moe_route.hip), grouped products gather the rows, apply the activation
and go down again behind the device's offsets (ops/csrc/moe.hip for decode-sized
steps, moe_gemm.hip for prompts), and one launch sums every token's rows with
their weights, the identity experts' share and the shared expert. Worst-case tile grids make every shape
static, so MoE decode steps capture into hipGraphs.

Parallelism at tp>1:
  * EP (expert parallel) when num_experts % tp == 0: each rank owns
    E/tp experts; non-local tokens contribute nothing locally and the
    rank outputs are summed by the existing TP all-reduce.
  * TP fallback (IE sharding) otherwise: every rank runs all experts on
    an intermediate-dim shard, same all-reduce.
"""
from __future__ import annotations

import torch
import torch.nn as nn

from .. import ops
from ..engine.config import ModelConfig
from ..parallel.layers import taken_apart, untouched
from ..parallel.state import get_state, tp_all_reduce


class MoERows:
    """A layer's output before its sum over the experts: whoever normalises
    it next sums it in the same launch."""

    def __init__(self, shape, dtype, *sum_args):
        self.shape, self.dtype, self.sum_args = shape, dtype, sum_args

    def tensor(self) -> torch.Tensor:
        y = self.sum_args[0]
        out = torch.empty(self.shape, device=y.device, dtype=self.dtype)
        ops.moe_combine(out, *self.sum_args)
        return out

    def _fits(self, residual, weight) -> bool:
        return self.dtype == torch.bfloat16 and self.shape[1] <= 8192 \
            and residual.dtype == weight.dtype \
            and all(t.is_contiguous() and t.data_ptr() % 16 == 0
                    for t in (residual, weight))

    def add_rms_norm(self, residual, weight, eps: float):
        """ops.fused_add_rms_norm of it."""
        if residual.dtype == torch.bfloat16 and self._fits(residual, weight):
            return ops.moe_combine_norm(residual, weight, eps,
                                        *self.sum_args), residual
        return ops.fused_add_rms_norm(self.tensor(), residual, weight, eps)

    def post_norm(self, x32, weight, eps: float, out_dtype):
        """ops.post_norm_residual of it."""
        if out_dtype == torch.bfloat16 and x32.dtype == torch.float32 \
                and self._fits(x32, weight):
            return ops.moe_combine_norm(x32, weight, eps, *self.sum_args)
        return ops.post_norm_residual(x32, self.tensor(), weight, eps,
                                      out_dtype)


@taken_apart
class MoEMLP(nn.Module):
    def __init__(self, cfg: ModelConfig):
        super().__init__()
        st = get_state()
        tp = st.tp_size
        self.cfg = cfg
        h = cfg.hidden_size
        ie = cfg.moe_intermediate_size or cfg.intermediate_size
        e = cfg.num_experts
        self.top_k = cfg.num_experts_per_tok
        self.num_experts = e
        # router outputs: the experts, then those that hand x through
        self.n_identity = cfg.moe_identity_experts
        self.n_route = e + self.n_identity
        if tp > 1 and e % tp == 0:
            # expert parallelism: contiguous expert slice per rank
            self.e_local = e // tp
            self.e_base = st.tp_rank * self.e_local
            self.ie_local = ie
        else:
            assert tp == 1 or ie % tp == 0, (ie, tp)
            self.e_local = e
            self.e_base = 0
            self.ie_local = ie // tp
        # f32 router option: the matrix is held in f32 and x is widened
        # before the product, so no logit is rounded to the activation
        # dtype before top-k
        self.gate = nn.Parameter(
            torch.empty(self.n_route, h, dtype=torch.float32
                        if cfg.moe_router_fp32 else cfg.dtype),
            requires_grad=False)
        # "relu2": ungated experts down(relu(up x)^2); everything else is
        # gated (act(gate x) * up x)
        self.gated = cfg.moe_act != "relu2"
        rows = 2 if self.gated else 1
        # stacked expert weights (local shard):
        # [E_l, 2*IE_l, h] (gate|up; ungated: [E_l, IE_l, h], up only)
        # and [E_l, h, IE_l]
        self.w_gate_up = nn.Parameter(
            torch.empty(self.e_local, rows * self.ie_local, h,
                        dtype=cfg.dtype),
            requires_grad=False)
        self.w_down = nn.Parameter(
            torch.empty(self.e_local, h, self.ie_local, dtype=cfg.dtype),
            requires_grad=False)
        if cfg.moe_bias:   # gpt-oss per-expert biases
            self.b_gate_up = nn.Parameter(
                torch.empty(self.e_local, 2 * self.ie_local, dtype=cfg.dtype),
                requires_grad=False)
            self.b_down = nn.Parameter(
                torch.empty(self.e_local, h, dtype=cfg.dtype),
                requires_grad=False)
        else:
            self.b_gate_up = None
            self.b_down = None
        self.act_mode = {"swiglu_oai": 1, "clamped_glu": 1,
                         "relu2": 2}.get(cfg.moe_act, 0)
        self.act_limit = float(cfg.moe_act_limit) \
            if cfg.moe_act == "clamped_glu" else 7.0
        # per-expert selection bias (deepseek-v3 noaux_tc; softmax_bias)
        self.e_score_correction_bias = None
        if cfg.moe_routing == "noaux_tc" or (
                cfg.moe_routing == "softmax_bias"
                and cfg.moe_choice_correction):
            self.e_score_correction_bias = nn.Parameter(
                torch.empty(self.n_route, dtype=torch.float32),
                requires_grad=False)
        if self.n_identity:
            if cfg.moe_routing != "softmax_bias" or tp > 1:
                raise NotImplementedError(
                    "identity experts: softmax_bias routing, one rank")
        # deepseek shared experts: always-on dense SwiGLU of width
        # n_shared * moe_ie, IE-sharded over TP; its down output is a
        # TP-partial like the routed output, so both ride ONE all-reduce
        if cfg.n_shared_experts > 0 or cfg.moe_shared_intermediate_size > 0:
            sie = cfg.moe_shared_intermediate_size \
                or cfg.n_shared_experts * ie
            assert tp == 1 or sie % tp == 0, (sie, tp)
            self.sie_local = sie // tp
            self.w_shared_gate_up = nn.Parameter(
                torch.empty(rows * self.sie_local, h, dtype=cfg.dtype),
                requires_grad=False)
            self.w_shared_down = nn.Parameter(
                torch.empty(h, self.sie_local, dtype=cfg.dtype),
                requires_grad=False)
        else:
            self.w_shared_gate_up = None

    def _choice(self):
        """The router's arguments behind the rows it reads."""
        cfg = self.cfg
        bias, groups, keep = None, 1, 1
        renorm, scale = cfg.moe_norm_topk, cfg.routed_scaling_factor
        if cfg.moe_routing in ("noaux_tc", "sigmoid_groups"):
            # deepseek-v3: sigmoid scores; SELECTION uses scores+bias with
            # group-limited top-k; WEIGHTS are the original sigmoid scores.
            # "sigmoid_groups" is the same without a selection bias.
            mode = "sigmoid"
            groups, keep = cfg.n_group, cfg.topk_group
            if cfg.moe_routing == "noaux_tc":
                bias = self.e_score_correction_bias
        elif cfg.moe_routing == "softmax_bias":
            # softmax over all outputs; the choice adds the correction
            # (and is group-limited), the weights are the chosen scores
            mode = "softmax"
            groups, keep = cfg.n_group, cfg.topk_group
            bias = self.e_score_correction_bias
        elif cfg.moe_routing == "topk_softmax":
            # gpt-oss: top-k on raw logits, softmax over the selected k
            mode, renorm, scale = "logits", False, 1.0
        else:
            mode = "softmax"
        if groups <= 1:             # no limit, whatever the number kept says
            groups = keep = 1
        # f32 router: x is widened before the product
        return (self.gate, bias, self.top_k, self.num_experts, groups, keep,
                renorm, scale, mode)

    def _choose(self, x: torch.Tensor):
        """Top-k choice, device-only: (experts int32 [T, K], weights f32
        [T, K], summed weight f32 [T] on identity experts)."""
        return ops.moe_gate_route(x, *self._choice())

    # Pairs up to which the weight-streaming kernels run, beyond it the tiled
    # grouped GEMMs: 16 rows per expert, 12 with many experts. A layer streamed
    # and tiled, in us, at 8, 16 and 32 rows per expert: 8 experts of 2048 x
    # 2048 58 and 73, 70 and 72, 101 and 74; 8 of 4096 x 14336 469 and 650, 615
    # and 641, 1102 and 660; 32 of 2880 x 2880 293 and 373, 375 and 373, 627
    # and 384; 128 of 2048 x 768 280 and 293, 352 and 309, 538 and 318; 64 of
    # 2048 x 1408 at 12 rows 270 and 272, at 16 288 and 271. (Beyond 4096 pairs
    # tiled rows are bf16, hence 16 for more than 256 experts.)
    # KAITO_MOE_FUSED_MAX overrides.
    import os as _os
    _most = _os.environ.get("KAITO_MOE_FUSED_MAX")
    FUSED_MAX_TOKENS = None if _most is None else int(_most)

    def _kernels_for(self, x: torch.Tensor) -> str:
        """"streamed", "tiled" (both free of host reads) or "loop": one
        library GEMM per expert, for f32 and odd widths. (Where an expert's
        rows and width keep the library's tiles full, 8 experts of 4096 x
        14336 and 8192 tokens, it takes 5.72 ms against 5.28 tiled.)"""
        E, H, TK = self.num_experts, x.size(1), x.size(0) * self.top_k
        if not (x.is_cuda and x.dtype == torch.bfloat16 and H % 64 == 0
                and self.ie_local % 64 == 0):
            return "loop"
        most = self.FUSED_MAX_TOKENS
        if most is None:
            most = E * (12 if 32 < E <= 256 else 16)
        return "streamed" if TK <= most else "tiled"

    def forward_add_norm(self, x, residual, weight, eps: float,
                         defer: bool = False):
        """fused_add_rms_norm(x, residual, weight), then forward of its rows:
        (output, residual)."""
        xn, residual, *chosen = ops.moe_norm_gate_route(
            x, residual, weight, eps, *self._choice())
        return self(xn, defer=defer and untouched(self, MoEMLP),
                    chosen=chosen), residual

    def forward(self, x: torch.Tensor, keep_f32: bool = False,
                split_shared: bool = False, defer: bool = False,
                chosen=None):
        """keep_f32: the routed sum is returned as accumulated, in f32.
        split_shared: returns (routed sum, the shared expert's output or
        None) for a caller that adds them itself. defer: the output may be
        MoERows. chosen: the result of _choose, if it is there already."""
        T, H = x.shape
        topi, topw, w_id = chosen if chosen is not None else self._choose(x)
        kernels = self._kernels_for(x)
        # decode-sized steps: every expert finds its rows by itself
        pairs = kernels == "streamed" and ops.moe_pairs_pay(
            topi.numel(), self.e_local, self.w_gate_up.size(1), x.size(1))
        pos = None
        if not pairs:
            # identity outputs sort behind every expert's rows
            sorted_tok, gates, offsets, pos = ops.moe_plan(topi, topw,
                                                           self.n_route)
        if not self.n_identity:
            w_id = None
        shared = None
        # deepseek shared experts; beside the routed ones where they fit
        beside = pairs and self._shared_fits(T)
        if self.w_shared_gate_up is not None and not beside:
            h1 = ops.linear_swiglu(x, self.w_shared_gate_up) if self.gated \
                else ops.relu2(ops.linear(x, self.w_shared_gate_up))
            shared = ops.linear(h1, self.w_shared_down)
        if kernels == "loop":
            out = self._routed_start(x, w_id)
            self._forward_loop(x, sorted_tok, gates, offsets, out)
            out = out if keep_f32 else out.to(x.dtype)
        else:
            x = x.contiguous()
            if x.data_ptr() % 16:
                x = x.clone()
            if pairs:
                y, beside_y = self._rows_pairs(x, topi, beside)
                shared = beside_y if beside else shared
            elif kernels == "streamed":
                y = self._rows_streamed(x, sorted_tok, offsets)
            else:
                y = self._rows_tiled(x, sorted_tok, offsets)
            rows = MoERows((T, H), torch.float32 if keep_f32 else x.dtype, y,
                           pos, topi, topw, self.e_base, self.e_local, x,
                           w_id, None if split_shared else shared)
            if defer and get_state().tp_size == 1:
                assert not split_shared
                return rows
            out = rows.tensor()
        if split_shared:
            assert get_state().tp_size == 1
            return out, shared
        if shared is not None and kernels == "loop":
            out = out + shared
        if get_state().tp_size > 1:
            out = tp_all_reduce(out)
        return out

    @staticmethod
    def _routed_start(x, w_id):
        """The routed sum starts from the identity experts' share."""
        return torch.zeros(x.shape, dtype=torch.float32, device=x.device) \
            if w_id is None else x * w_id[:, None]

    # All return the experts' outputs of the sorted rows (or of the pairs), to be
    # summed per token by moe_combine; static shapes, no host read.
    def _shared_fits(self, T: int) -> bool:
        """Whether the shared expert runs as one more of the routed ones: of
        their sizes, on few tokens."""
        w = self.w_shared_gate_up
        if w is None or not ops.moe_shared_pays(
                T, T * self.top_k, self.num_experts, w.size(1), w.size(0) // 2):
            return False
        d = self.w_shared_down
        return self.gated \
            and self.act_mode == 0 \
            and self.b_gate_up is None and self.b_down is None \
            and w.shape == self.w_gate_up.shape[1:] \
            and d.shape == self.w_down.shape[1:] \
            and w.dtype == d.dtype == torch.bfloat16 \
            and w.is_contiguous() and d.is_contiguous() \
            and w.data_ptr() % 16 == d.data_ptr() % 16 == 0

    def _rows_pairs(self, x, topi, beside: bool = False):
        """(rows of the pairs, the shared expert's [T, H] or None)"""
        def new(rows, cols, dtype):
            return torch.empty(rows, cols, dtype=dtype, device=x.device)

        T, H = x.shape
        act = new(topi.numel(), self.ie_local, x.dtype)
        up, down, all_y = {}, {}, None
        if beside:
            all_act, all_y = new(T, self.ie_local, x.dtype), new(T, H, x.dtype)
            up = dict(all_w=self.w_shared_gate_up, all_act=all_act)
            down = dict(all_w=self.w_shared_down, all_act=all_act,
                        all_y=all_y)
        ops.moe_up_pairs(act, x, self.w_gate_up, topi, self.n_route,
                         self.e_base, self.e_local, self.b_gate_up,
                         self.act_mode, self.act_limit, **up)
        y = new(topi.numel(), H, torch.float32)
        ops.moe_down_pairs(y, act, self.w_down, topi, self.n_route,
                           self.e_base, self.e_local, self.b_down, **down)
        return y, all_y

    def _rows_tiled(self, x, sorted_tok, offsets):
        TK, H = sorted_tok.numel(), x.size(1)
        act = torch.empty(TK, self.ie_local, dtype=x.dtype, device=x.device)
        ops.moe_grouped_up(act, x, self.w_gate_up, sorted_tok, offsets,
                           self.e_base, self.b_gate_up, self.act_mode,
                           self.act_limit)
        # rows keep f32 until their sum where they always did: in steps of
        # up to 4096 pairs and in captured ones
        y = torch.empty(TK, H, device=x.device, dtype=torch.float32
                        if TK <= 4096
                        or torch.cuda.is_current_stream_capturing()
                        else x.dtype)
        ops.moe_grouped_down(y, act, self.w_down, offsets, self.e_base,
                             self.b_down)
        return y

    def _rows_streamed(self, x, sorted_tok, offsets):
        act = torch.empty(sorted_tok.numel(), self.ie_local, dtype=x.dtype,
                          device=x.device)
        ops.moe_gate_silu(act, x, self.w_gate_up, sorted_tok, offsets,
                          self.e_base, self.e_local, self.b_gate_up,
                          self.act_mode, self.act_limit)
        y = torch.empty(sorted_tok.numel(), x.size(1), dtype=torch.float32,
                        device=x.device)
        ops.moe_down_rows(y, act, self.w_down, offsets, self.e_base,
                          self.e_local, self.b_down)
        return y

    def _forward_loop(self, x, sorted_tok, gates, offsets, out):
        """Per-expert torch GEMMs (_kernels_for). Host sync on the segment
        sizes."""
        off = offsets.tolist()
        idx64 = sorted_tok.long()
        for le in range(self.e_local):
            e = self.e_base + le
            s, t = off[e], off[e + 1]
            if s == t:
                continue
            rows = idx64[s:t]
            xs = x[rows]
            h1 = ops.linear(
                xs, self.w_gate_up[le],
                self.b_gate_up[le] if self.b_gate_up is not None else None)
            if self.act_mode == 2:
                act = ops.relu2(h1)
            elif self.act_mode == 1:
                act = ops.clamped_glu(h1, self.act_limit)
            else:
                act = ops.silu_and_mul(h1.contiguous())
            y = ops.linear(
                act, self.w_down[le],
                self.b_down[le] if self.b_down is not None else None)
            # f32 accumulation over a token's experts, like the fused path
            out.index_add_(0, rows, y.float() * gates[s:t, None])
