"""kaito_amd.ops — gfx950 HIP kernels with a CPU fp32 reference fallback.

Dispatch policy (engine contract):
  * CUDA/ROCm tensors → the in-tree HIP extension. If the extension is
    missing on a GPU machine this raises loudly — there is NO silent
    eager fallback on GPU.
  * CPU tensors → torch_ref reference implementations (tests / no-GPU dev).

The extension is split into kernel groups (ops/_build.py GROUPS), one
shared library each; a group is built (if absent) and loaded the first
time one of its ops is called.
"""
from __future__ import annotations

import functools

import numpy as np
import torch
import torch.autograd.forward_ad as _fwd_ad

from . import torch_ref
from ._build import GROUPS, SO_PATH, so_path

_LOADED: set = set()

# op name → kernel group that registers it
_OP_GROUP = {}
for _g, _names in {
    "core": ("rms_norm fused_add_rms_norm rotary_embedding silu_and_mul "
             "gelu_and_mul gelu layer_norm fused_add_layer_norm "
             "rope_and_cache reshape_and_cache topk skinny_linear skinny_norm skinny_swiglu "
             "skinny_linear_pair batch_linear batch_parts add_rms_norm_parts "
             "tile_linear tile_swiglu tile_pair"),
    "attn": ("paged_attention paged_attention_sp rope_paged_attention "
             "prefill_attention "
             "mla_prefill_attention context_attention mfma_tile_gemm paged_read_bw"),
    "mla": "mla_decode mla_prepare mla_prepare_rows head_rows mla_cache_write",
    "moe": ("moe_gate_silu moe_down_rows moe_up_pairs moe_down_pairs "
            "moe_grouped_up moe_grouped_down moe_combine moe_combine_norm "
            "latent_kv"),
    "route": "moe_route moe_gate_route moe_norm_gate_route moe_sort",
    "quant": ("w4a16_gemv w4a16_dequant w4a16_gemm w4a16_swiglu "
              "w4a16_norm_linear w4a16_norm_in_tiles "
              "w4a16_in_tiles lora_shrink lora_expand"),
    "comm": ("allreduce_rmsnorm one_shot_ar_rmsnorm ipc_handle ipc_open "
             "ipc_close"),
    "mix": ("causal_conv_update "
            "qk_norm_cache_write window_attention window_attention_tiles "
            "embed_positions "
            "post_norm_residual rms_norm_cast residual_add_norm "
            "scaled_residual_add_norm token_shift "
            "clamped_glu sigmoid_mul gelu_glu relu_glu relu2 "
            "scaled_softcap"),
    "latent": ("bigram_embed latent_rope_cache_write latent_attention "
               "latent_expand"),
    "delta": "gated_delta_rule rglru_gates rglru_scan rglru_rows",
    "diag": "diag_delta_rule hgrn2_scan gla_scan",
    "decay": "mlstm_scan ssd_scan",
    "streams": "stream_mix_norm stream_embed",
    "lnorm": "layer_norm_cast embed_layer_norm sandwich_norm_residual",
}.items():
    for _n in _names.split():
        _OP_GROUP[_n] = _g

# groups that predate the split: load_extension() without arguments loads
# these, so `ops.load_extension(); torch.ops.kaito.<op>` keeps working
_LEGACY_GROUPS = ("core", "attn", "mla", "moe", "quant", "comm")


def extension_available(group: str = "core") -> bool:
    return so_path(group).exists()


def load_extension(*groups: str) -> None:
    """Load (and build together, if absent) kernel groups; no arguments =
    every group except the lazily-loaded newer ones."""
    todo = [g for g in (groups or _LEGACY_GROUPS) if g not in _LOADED]
    absent = [g for g in todo if not so_path(g).exists()]
    if absent:
        from ._build import build
        build(groups=absent)
    for g in todo:
        torch.ops.load_library(str(so_path(g)))
        _LOADED.add(g)


class _Kernels:
    """`_K.<op>` = torch.ops.kaito.<op> with its group loaded first."""

    def __getattr__(self, name: str):
        group = _OP_GROUP[name]
        if group not in _LOADED:
            if not torch.cuda.is_available():
                raise RuntimeError(
                    "kaito_amd.ops: got a CUDA tensor but torch.cuda is "
                    "unavailable")
            load_extension(group)
        fn = getattr(torch.ops.kaito, name)
        setattr(self, name, fn)
        return fn


_K = _Kernels()


def _require_ext() -> None:
    """Kept for callers that predate per-group loading (no-op: `_K`
    loads the group an op needs)."""


# ---------------------------------------------------------------- public ops

def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _K.rms_norm(out, x, weight, eps)
        return out
    return torch_ref.rms_norm(x, weight, eps)


def fused_add_rms_norm(x: torch.Tensor, residual: torch.Tensor,
                       weight: torch.Tensor, eps: float):
    """Returns (normed, residual). On GPU, `residual` is updated IN PLACE
    (residual += x) and returned."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _K.fused_add_rms_norm(out, x, residual, weight, eps)
        return out, residual
    return torch_ref.fused_add_rms_norm(x, residual, weight, eps)


def rotary_embedding(positions: torch.Tensor, q: torch.Tensor, k: torch.Tensor,
                     head_dim: int, cos_sin_cache: torch.Tensor):
    """In-place on GPU; returns (q, k)."""
    if q.is_cuda:
        _K.rotary_embedding(positions, q, k, head_dim, cos_sin_cache)
        return q, k
    return torch_ref.rotary_embedding(positions, q, k, head_dim, cos_sin_cache)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda and x.dtype == torch.float32:
        # f32 verification mode: plain elementwise math, no bf16 kernel
        d = x.size(-1) // 2
        return torch.nn.functional.silu(x[..., :d]) * x[..., d:]
    if x.is_cuda:
        d = x.size(-1) // 2
        out = torch.empty(*x.shape[:-1], d, dtype=x.dtype, device=x.device)
        _K.silu_and_mul(out, x)
        return out
    return torch_ref.silu_and_mul(x)


def _transformed() -> bool:
    """Whether torch does more with a call than run it: forward-mode
    derivatives, vmap and the like, tracing, autocast. They know torch's
    operations and none of ours."""
    return _fwd_ad._current_level >= 0 \
        or torch._C._functorch.peek_interpreter_stack() is not None \
        or torch._C._len_torch_dispatch_stack() > 0 \
        or torch.is_autocast_enabled("cuda")


def _plain_rows(x: torch.Tensor, w: torch.Tensor, most: int) -> bool:
    """1 to `most` rows of bf16 on the GPU, 16-byte aligned rows, nothing to
    differentiate: what the kernels of small linear layers take."""
    return x.is_cuda and x.dim() == w.dim() == 2 and 1 <= x.size(0) <= most \
        and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 \
        and x.device == w.device and not _transformed() \
        and w.is_contiguous() and w.size(1) % 8 == 0 and w.numel() > 0 \
        and x.stride(1) == 1 \
        and (x.size(0) == 1 or x.stride(0) % 8 == 0) \
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 \
        and not (torch.is_grad_enabled()
                 and (x.requires_grad or w.requires_grad))


def _skinny(x: torch.Tensor, w: torch.Tensor, glu: bool = False) -> bool:
    """Whether x W^T runs on the weight-streaming kernels.

    The lines, with us on both sides (streamed, library; weights out of the
    caches): beyond 4 rows x comes through the caches once per 16 rows of W,
    and the library is ahead from where that costs more.
    Up to 4 rows always (28672 x 4096: 34.6, 56.3 for one row and 41.1, 55.9
    for four; 4096 x 4096: 7.2, 15.3 and 9.2, 15.5; a tie or 6 % behind at
    576 x 7168 and 2560 x 10240 for four).
    Up to 8: all but few rows of W with a long K (576 x 7168: 9.5, 8.2 at 8)
    and counts of rows that go unevenly on the CUs (5120 x 5120: 15.7, 14.5;
    as a SwiGLU pair 15.8, 16.9).
    Up to 16: to 4096 x 4096 (10.7, 15.5; 6144 x 4096: 16.3, 14.4) and K of
    7168 (2112 x 7168: 12.7, 12.6; 2048 x 8192: 14.6, 13.1); SwiGLU pairs,
    which save a launch, to 8192 (28672 x 4096: 50.3, 60.5), uneven ones
    excepted (5120 x 5120: 19.1, 17.9).
    K of 2048, where x fits the registers (7168 x 2048: 9.9, 12.7 at 16; 12288
    13.0, 14.8; 128256 91, 103; at 32 4096 x 2048: 8.4, 11.8; 5152 11.1, 11.8;
    8192 12.4, 12.8; 24576 23.3, 25.1; 128256 98, 105; as a pair 16384 17.3,
    19.5), but beyond 24 rows the library is ahead on both sides of 12288, three
    tiles per CU and a tie (10240 14.4, 13.6; 12288 15.2, 14.8; 16384 18.0,
    17.0); and K of 4096 with many rows of W up to 16 (12288 x 4096 22.0, 28.4;
    128256 167, 186).
    Up to 32: to 3072 x 2048 (7.4, 11.5; as a pair to 6144 x 2048 12.5, 15.0)
    and K of 4096 (1024 x 4096: 10.1, 11.3 at 24), where beyond 24
    rows the library has another kernel for few rows of W and K of 2560 and
    more (1024 x 2560: 8.0, 6.9; 2048 x 2816: 8.8, 9.5; 1024 x 2816 as a pair
    9.0, 9.5)."""
    M = x.size(0)
    if M > 32 or w.dim() != 2:
        return False
    return _skinny_shape(M, *w.shape, glu) and _plain_rows(x, w, 32)


def _skinny_shape(M: int, N: int, K: int, glu: bool) -> bool:
    if M <= 4:
        return True
    if K % 64 or N % 16:
        return False
    # x stays in registers while W streams
    if K == 2048 and N * K < 1 << 31:
        return glu or M <= 24 or not (8192 < N < 12288 or 12544 <= N < 24576)
    if K == 4096 and M <= 16 and N >= 12288 and N * K < 1 << 31:
        return True
    if M <= 16 and N < 1024 and K > 5120 and not glu:
        return False
    uneven = 4096 < N < 7168 and K > 4096
    if M <= 8:
        return (K <= 8192 or N >= 4096) and (glu or not uneven)
    if M <= 16:
        return K <= 8192 and not uneven if glu \
            else N * K <= 4096 * 4096 and K <= 7168
    return N * K <= (6144 if glu else 3072) * 2048 and K <= 4096 and (
        M <= 24 or K < 2560 or N >= 2048 or glu)


def _batched(x: torch.Tensor, w: torch.Tensor, glu: bool = False) -> bool:
    """Whether x W^T of up to 256 rows runs on the split kernel
    (csrc/batch_linear.hip) where the row streams do not take it.

    Both sides in us (split, library; weights out of the caches). The split
    of K is what the library does not always find: ahead from K of 10240 on
    (4096 x 14336: 24.3, 26.4 at 16 rows, 27.4, 34.9 at 48, 38.5, 49.4 at 128,
    47.3, 59.1 at 256; 7168 x 18432 at 256 88, 208), to 16384 rows of W
    (beyond, W is cut often enough without: 28672 x 14336 at 128 1 % behind).
    Fewer than 2048 rows of W with K below 13824 only to 64 rows (1024 x 10240
    15.1, 16.0 at 64, 17.2, 15.6 at 96, 26.3, 22.2 at 256, and 13.5, 11.5 at 16,
    where the norm behind it gives most of that back), of inner sizes in
    multiples of 512 (1024 x 11008 at 32 14.3, 18.0).
    K in no multiple of 256, which the library has few kernels for (4096 x
    2880: 1.1 to 1.25 times as fast from 17 to 128 rows, 28672 x 2880 1.24 to
    1.39; behind at 256). In odd multiples of 256: below 4096 only wide outputs
    and up to 64 rows (8192 x 2816 1.04 to 1.30, 16384 x 3840 1.05 to 1.18 but
    0.96 at 96, 4096 x 2816 0.80 to 0.95, 12288 x 3840 at 64 0.90); else to
    8192 rows of W (4096 x 5376 1.16 to 1.41; 3072 x 4352 0.86 to 0.98), beyond
    to 64 (16384 x 5376 1.07 to 1.18, at 96 to 128 0.99, 20480 x 5376 0.86 to
    0.92), to 16384 at K of 8192 and more (16384 x 8960 1.0 to 1.16; 20480 x
    8960 at 128 0.90). Beyond 32768 rows of W a workgroup has all of K and the
    library enough tiles: to 32 rows (40960 x 2880 1.20, 49152 x 5376 0.98 to
    1.02, 131072 x 8960 1.06; at 64 0.93 to 1.09, at 128 0.81 to 0.93), to 96 of
    a vocabulary of 200000 (201088 x 2880 207, 349 at 17 rows, 272, 357 at 96,
    287, 266 at 128; 262208 x 5376 455, 581, 612, 639 and 632, 574).
    K from 4096: to 6144 rows of W (3072 x 5120 at 64 1.19 times, 4096 x 7168
    at 128 1.67), fewer than 4096 only from K of 5120 on (3072 x 4096 0.86 to
    0.93 to 64 rows, 3072 x 4608 0.88 to 0.97); below 4608 only to 64 rows (4096
    x 4096 14.9, 14.2 there, ahead once the norm behind it sums the parts, and
    18.8, 16.9 at 128; 4096 x 4608 1.09 to 1.48 to 192 rows); at K of 8192 only
    beyond 32 rows (4096 x 8192 0.92 at 32, 1.19 at 33). To 8192 between K of
    4608 and 8192 (8192 x 7168: 1.02 to 1.47; 8192 x 4096 at 64 0.88, 8192 x
    8192 at 64 0.84); 16384 to 32768 to 64 rows (1.00 to 1.16), beyond to 32
    and from K of 5120 (49152 x 7168 at 32 1.08 and 0.96 at 64, 57344 x 5120
    1.08 and 0.95; 36864 x 4608 0.97, 49152 x 4096 0.82; 128256 x 4096 206,
    193). 193 to 256 rows: 6144 to 16384 with K from 7168 (1.06 to 1.67; 4096 x
    7168 0.91).
    SwiGLU pairs, which save a launch and a pass: from 12288 rows of W with
    more than 16 rows, 32 for K of 2048 (28672 x 4096: 48.9, 57.2 at 64, 73.6,
    79.8 at 256; 12288 x 2048 16.6, 20.2 at 64; 8192 x 4096 0.89), beyond 32768
    to 64 rows (57344 x 4096: 1.07 to 1.13, 0.90 at 256), at K of 8192 from
    20480 on (16384 x 8192 0.97). 20480 rows of W are 160 workgroups of 64 + 64
    columns, which leaves CUs idle: with K beyond 4096 not from 65 to 128 rows
    (20480 x 5120 1.14 at 32, 0.94 and 0.87 at 96 and 128, 0.99 at 192; x 7168
    0.97, 0.92; 22016 x 5120 0.93 at 128, 22528 x 5120 1.01)."""
    M = x.size(0)
    if not 9 <= M <= 256 or w.dim() != 2:
        return False
    return _batched_shape(M, *w.shape, glu) and _plain_rows(x, w, 256) \
        and M * x.stride(0) < 1 << 31


def _batched_shape(M: int, N: int, K: int, glu: bool) -> bool:
    if K % 64 or N % (32 if glu else 16) or (N + 128) * K >= 1 << 31:
        return False
    if glu:
        if 64 < M <= 128 and 16384 < N < 22528 and K > 4096:
            return False
        return M > (16 if K > 2048 else 32) and K >= 2048 and N >= (
            20480 if K >= 8192 else 12288) and (N <= 32768 or (N <= 65536 and M <= 64))
    if K >= 10240:
        return N <= 16384 and N >= (
            2048 if M > 64 and K < 13824 and K % 512 == 0 else 1024)
    if M < 17:
        return False
    if K % 512:
        if not (K >= 2560 and N >= 3072 and M <= 128):
            return False
        if N > 32768:
            return M <= 32 or (N >= 196608 and M <= 96)
        if K % 256:
            return True
        if K < 4096:
            return M <= 64 and N >= 8192 and (
                M <= 32 or not 12288 <= N < 16384)
        if N < 4096:
            return K >= 5120
        return M <= 64 or N <= (16384 if K >= 8192 else 8192)
    if K < 4096 or K > 8192 or N < 3072:
        return False
    if M > 192:
        return K >= 7168 and 6144 <= N <= 16384 and (K < 8192 or N <= 12288)
    if N <= 6144:
        return (N >= 4096 or K >= 5120) and (M <= 64 or K >= 4608) \
            and (M > 32 or K < 8192)
    if N <= 8192:
        return 4608 <= K < 8192
    if N <= 32768:
        return N >= 16384 and K < 8192 and M <= 64
    return N <= 65536 and 5120 <= K < 8192 and M <= 32


def _plain_bias(bias, w: torch.Tensor) -> bool:
    """None, or one that the kernels of small linear layers add."""
    return bias is None or (
        bias.dtype == torch.bfloat16 and bias.is_contiguous()
        and bias.shape == w.shape[:1] and bias.device == w.device
        and not (torch.is_grad_enabled() and bias.requires_grad))


def linear(x: torch.Tensor, w: torch.Tensor, bias=None) -> torch.Tensor:
    """x W^T (+ bias): the weight-streaming kernels for small decode steps, the
    split kernel for larger ones where it is ahead, the tiles for large batches'
    logits and for prompts whose large tiles fill no whole number of rounds,
    hipBLASLt otherwise."""
    if _plain_bias(bias, w):
        skinny = _skinny(x, w)
        if skinny or _batched(x, w):
            out = torch.empty(x.size(0), w.size(0), dtype=x.dtype,
                              device=x.device)
            if skinny:
                _K.skinny_linear(out, x, w, _none(bias, x))
            else:
                _K.batch_linear(out, x, w, _none(bias, x), 0, 0, False)
            return out
    if bias is None and w.dim() == 2 and x.dim() == 2 \
            and (_vocabulary_shape(x.size(0), *w.shape)
                 or _uneven_shape(x.size(0), *w.shape)) \
            and _tiles_fit(x, w, 64):
        out = torch.empty(x.size(0), w.size(0), dtype=x.dtype, device=x.device)
        _K.tile_linear(out, x, w)
        return out
    return torch.nn.functional.linear(x, w, bias)


class SplitRows:
    """A product whose K was split, before the sum of its parts [splits, M, N]
    f32: whoever normalises it next sums it in the same launch."""

    def __init__(self, part: torch.Tensor):
        self.part = part

    def add_rms_norm(self, residual, weight, eps: float):
        """fused_add_rms_norm of it, to the same bits; one launch for rows
        and weights in whole 16-byte chunks."""
        if not (self.part.is_cuda and residual.data_ptr() % 16 == 0
                and weight.data_ptr() % 16 == 0):
            rows = self.part[0]
            for p in self.part[1:]:
                rows = rows + p
            return fused_add_rms_norm(rows.to(residual.dtype), residual,
                                      weight, eps)
        out = torch.empty_like(residual)
        _K.add_rms_norm_parts(out, self.part, residual, weight, eps)
        return out, residual


def linear_parts(x: torch.Tensor, w: torch.Tensor):
    """linear(x, w) for the add and RMS norm behind it: SplitRows where the
    product is the split kernel's and in parts, of rows that the norm can sum
    (always ahead, by 0.4 us of 29 to 4 of 104)."""
    if w.size(0) <= 8192 and not _skinny(x, w) and _batched(x, w):
        part = _K.batch_parts(x, w)
        if part.numel():
            return SplitRows(part)
    return linear(x, w)


def linear_pair(x: torch.Tensor, w: torch.Tensor, x2: torch.Tensor,
                w2: torch.Tensor, bias=None, bias2=None):
    """(linear(x, w, bias), linear(x2, w2, bias2)): products that do not wait
    for one another, of the same K. One launch where both stream their weights
    (us, two launches and one, 32 rows, K of 2048: 3072 and 576 rows of W 14.8, 8.3,
    3072 and 4096 of one x 16.3, 12.2, 2048 and 2048 of two 14.5, 8.8; one row
    6.9, 4.9, 9.4, 6.7 and 7.2, 5.1)."""
    if x.size(0) == x2.size(0) <= 32 and x.dim() == x2.dim() == 2 \
            and w.size(1) == w2.size(1) and x.device == x2.device \
            and w.size(0) % 16 == w2.size(0) % 16 == 0 \
            and _skinny(x, w) and _skinny(x2, w2) \
            and _plain_bias(bias, w) and _plain_bias(bias2, w2) \
            and _pair_pays(x.size(0), w.size(0) + w2.size(0),
                           x.data_ptr() == x2.data_ptr()
                           and x.stride() == x2.stride()):
        out, out2 = (torch.empty(x.size(0), v.size(0), dtype=x.dtype,
                                 device=x.device) for v in (w, w2))
        _K.skinny_linear_pair(out, x, w, _none(bias, x), out2, x2, w2,
                              _none(bias2, x))
        return out, out2
    if _pair_tiled(x, w, x2, w2) and _plain_bias(bias, w) \
            and _plain_bias(bias2, w2):
        out, out2 = (torch.empty(x.size(0), v.size(0), dtype=x.dtype,
                                 device=x.device) for v in (w, w2))
        _K.tile_pair(out, x, w, _none(bias, x), out2, x2, w2, _none(bias2, x))
        return out, out2
    return linear(x, w, bias), linear(x2, w2, bias2)


def _pair_pays(M: int, N: int, one: bool) -> bool:
    """Workgroups that stay for several tiles keep one x in registers: of two,
    and more than 4 rows, the many tiles of wide products are better alone (K of
    2048, one launch as a share of two, 24576 and 576 rows of W at 16 and 32 rows
    1.02 and 1.20, with one x 0.84 and 0.81; 8192 and 1024 at 32 0.89)."""
    return one or M <= 4 or N < 16384


@functools.lru_cache(1024)
def _tile_plan(M: int, N: int):
    """The tiles that the kernels choose for M rows and N weight rows and the cost of
    their rounds (csrc/tile_gemm.h `run`): "whole" ones of 256 x 256, "quartered"
    in the last round, or "smaller" ones."""
    def share(rows, cols):          # tiles of an XCD
        return -(-(-(-M // rows) * -(-N // cols)) // 8)

    def rounds(n):
        return -(-n // 32)
    large = share(256, 256)
    rest = large % 32
    if rest > (16 if large < 32 else 8):
        rest = 0
    whole = 5 * rounds(large - rest) + 2 * rounds(4 * rest)
    small = min(3 * rounds(share(128, 256)), 3 * rounds(share(256, 128)),
                2 * rounds(share(128, 128)))
    if small < whole:
        return "smaller", small
    return "quartered" if rest else "whole", whole


def _tile_fill(M: int, N: int) -> float:
    """What share of its time a product of M rows and N weight rows keeps the
    chip's 256 workgroups busy for."""
    return M * N / (_tile_plan(M, N)[1] * 256 * 65536 / 5)


def _here(x: torch.Tensor) -> bool:
    """Whether a launch on the current device's stream is one on x's: torch's
    operations, which a kernel stands in for, find their way by themselves."""
    return x.device.index == torch.cuda.current_device()


def _tiles_fit(x: torch.Tensor, w: torch.Tensor, cols: int) -> bool:
    """Operands that the tiles' kernels take."""
    return _plain_rows(x, w, (1 << 24) - 1) and x.is_contiguous() and _here(x) \
        and w.size(1) % 64 == 0 and w.size(0) % cols == 0 \
        and max(w.shape) < 1 << 22 and w.numel() <= 0x7fff8000


def _tiled(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether a SwiGLU pair of a prompt's rows runs on the tiles, activation
    included (csrc/tile_linear.hip)."""
    return w.dim() == 2 and x.dim() == 2 \
        and _tiled_shape(x.size(0), *w.shape) and _tiles_fit(x, w, 128)


def _tiled_shape(M: int, N: int, K: int) -> bool:
    """The pass over the library's output that tiles spare is worth an unevenly
    filled last round where the chip is busy for 82 % of the time, or where K is
    short and the rows are many (us, library and activation, tiles: 28672 x 4096
    at 512 rows 120, 111, 1500 294, 294, 8192 1385, 1259; 22016 x 4096 at 1500 316,
    218, at 1000, 73 % busy, 175, 203; 35840 x 5120 at 3000 889, 766; 5760 x 2880 at
    8192 339, 189, at 1000, 57 %, 43, 54; 16384 x 3072 at 1500, 81 %, 144, 158;
    4096 x 2048 at 1000 26, 20, 8192 118, 107; 1024 x 2048 at 2048, 31 %, 20, 19 and
    1500 18, 19; 2816 x 2048 at 1500, 42 %, 28, 27; in one round of 256 x 256 3584 x 2048
    at 2378, 51 %, 39.6, 41.3, with weights from memory 44.2, 44.6, 2816 x 2048 at 3176,
    53 %, 40.3, 41.0 and 45.1, 43.8, 2048 x 2048 at 4379, 53 %, from memory 51.2, 43.3). Of
    410 sizes one is more than 1 % behind, 1.38 times as fast in the mean."""
    if M <= 256:
        return False
    fill = _tile_fill(M, N)
    return fill >= 0.82 or (K <= 2048 and M >= 1000 and fill >= (
        0.52 if K > 1536 and _tile_plan(M, N)[0] == "whole" else 0.42))


def _vocabulary_shape(M: int, N: int, K: int) -> bool:
    """Whether a large batch's logits run on the tiles, whose 256 rows are a
    step's (us, library and tiles: 128256 x 4096 290, 220 at 129 rows, 258, 225 at
    192, 299, 239 at 256; 151936 x 4096 303, 293 at 129, 356, 311 at 256; 256000 x
    4096 553, 477; 128256 x 8192 460, 427 at 160, 547, 469 at 256; 128256 x 6144
    361, 352 at 160, 446, 362 at 256; 131072 x 5120 279, 294 at 144, 338, 313 at
    256; 100352 x 4096 230, 201 at 129, 202, 203 at 160, 229, 205 at 256, but x 8192 358,
    390 at 160 and 385, 390 at 224. Fewer rows or a shorter
    K went either way: 262144 x 2304 0.94 to 0.98, 128256 x 2048 0.95 to 1.24, 151936 x
    4096 1.0 to 1.02 from 33 to 64 rows, 128256 x 8192 0.94 to 1.02. So do smaller
    vocabularies, by how full their last round is: 92416 x 4096 to 8192 0.73 to 0.91,
    81920 1.04 to 1.25, 65536 0.93 to 1.09, 49152 0.93 to 1.11, 32000 0.73 to
    0.95). Of a K of 6144 and more, up to 192 rows are ahead only where the last round
    is full (library over tiles at 144 and 160 rows, 128256 x 7168 1.08, 1.08, 102400
    0.96, 0.94, 120832 0.97, 0.94, 151936 0.93, 1.05, x 8192 0.90, 1.02, x 6144 0.95,
    1.03, 112640 x 6144 0.97, 0.96; at 208 and 256 102400 x 7168 1.09, 1.08, 151936 x
    8192 1.03, 1.14)."""
    if not (129 <= M <= 256 and K >= 4096
            and N >= (128000 if K >= 8192 else 100000)
            and (M > 224 or not 4096 < K < 6144)):
        return False
    tiles = -(-N // 256)
    return K < 6144 or M > 200 or tiles >= 0.95 * 256 * -(-tiles // 256)


def _uneven_shape(M: int, N: int, K: int) -> bool:
    """Whether a product of a prompt's rows whose tiles of 256 x 256 fill no whole
    number of rounds runs on the tiles, which cut the last round or take smaller
    ones. Whole rounds are the library's (0.94 to 0.99 times). us, library and
    tiles: 3072 x 2048 at 8192 rows 91, 84, 5901 86, 65; 5120 x 2048 at 3948 85,
    68; 2048 x 2048 at 2585 31, 27; 1024 x 1536 at 8192 28, 26; 4096 x 1024 at 4162
    56, 39; 3072 x 512 at 6541 51, 25; 4096 x 3072 at 4437 112, 93; 8192 x 3072 at
    6309 270, 228. K of 4096 with a quartered round 1.06, with smaller tiles 0.99 to
    1.02; up to 1024 rows 0.4 to 1.1. Smaller tiles that leave much of their rounds
    idle are behind (1024 x 3072 at 4192 rows, 43 % busy, 31, 38; 2048 x 2560 at 2315,
    47 %, 29, 34; 1024 x 1536 at 4807, 49 %, 21, 23; 2048 x 1536 at 2700, 55 %, 22, 23),
    from 56 % on not; 128 x 256 with a K of 1024 and more from 62 % on (1536 x 2048 at
    4000, 61 %, 27.0, 28.1, 1408 x 2560 at 4176, 58 %, 33, 35, 2560 x 1280 at 2233, 57 %,
    20, 21). One round of quarters is even or behind
    below 45 % (1024 rows of W at 2570, 39 %: x 256 6.8, 7.2, x 512 10.8, 8.2, x 1024 11.3,
    11.6, x 4096 27.9, 30.0; at 47 % x 4096 1.05). K below 256 went either way (0.81 to
    1.6). Of 480 sizes 2 are more than 1.5 % behind (2560 x 2560 at 8445 97.9, 100.3),
    1.20 times as fast in the mean."""
    if not (M > 2048 and 1024 <= N <= 8192 and 256 <= K <= 4096):
        return False
    kind, cost = _tile_plan(M, N)
    fill = _tile_fill(M, N)
    if cost == 2 and fill < 0.45 and not 256 < K <= 512:
        return False
    return kind == "quartered" or (kind == "smaller" and K <= 3072 and fill >= (
        0.555 if K < 1024 or cost == 2 else 0.62))


def _pair_tiled(x, w, x2, w2) -> bool:
    return x.dim() == x2.dim() == w.dim() == w2.dim() == 2 \
        and x.shape == x2.shape and w.size(0) % 256 == 0 \
        and _pair_tiled_shape(x.size(0), w.size(0) + w2.size(0), w.size(1)) \
        and x.device == x2.device \
        and _tiles_fit(x, w, 256) and _tiles_fit(x2, w2, 64)


def _pair_tiled_shape(M: int, N: int, K: int) -> bool:
    """Whether two products of a prompt's rows, N outputs together, run as one
    launch of tiles: no last round of their own (us, library twice and tiles, K of
    2048: 3072 + 576 at 128 rows 20, 16, 700 28, 19, 2048 42, 31, 8192 120, 99, at
    64 17, 16; 3072 + 4096 at 128 30, 23, 2048 67, 55, 6500 170, 149, but 87, 93 at
    3000, 100, 102 at 4096 and 187, 191 at 8192; 2048 + 576 at 8192 79, 82). K of
    5120 and 7168 gave 0.54 to 1.38 times. Few outputs of a long K gain little with
    weights from memory and lose with those that are in the caches (512 + 320 of 2048 at
    168 rows 16.3, 16.2 and 11.2, 16.0; 512 + 64 at 653 17.4, 16.5 and 14.3, 16.4; 2048 +
    64 of 1536 at 154 14.2, 13.5 and 12.1, 13.2), more of them with neither (3072 + 576 at
    241 17.5, 16.6 from the caches)."""
    return M >= 128 and K <= 2048 and N <= 7168 and (
        M * N >= 400000 or K <= 1024) and (
        M * N <= 20000000 or _tile_fill(M, N) >= 0.88)


def linear_swiglu(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x Wg^T) * (x Wu^T) for the stacked W = [Wg | Wu]."""
    skinny = _skinny(x, w, True)
    if skinny or _batched(x, w, True):
        out = torch.empty(x.size(0), w.size(0) // 2, dtype=x.dtype,
                          device=x.device)
        if skinny:
            _K.skinny_swiglu(out, x, w)
        else:
            _K.batch_linear(out, x, w, _none(None, x), 0, 0, True)
        return out
    if _tiled(x, w):
        out = torch.empty(x.size(0), w.size(0) // 2, dtype=x.dtype,
                          device=x.device)
        _K.tile_swiglu(out, x, w)
        return out
    return silu_and_mul(torch.nn.functional.linear(x, w))


def add_norm_linear(x: torch.Tensor, residual: torch.Tensor,
                    norm: torch.Tensor, eps: float, w: torch.Tensor,
                    bias=None, glu: bool = False):
    """fused_add_rms_norm of x and residual, then linear (glu: linear_swiglu
    of the stacked w); returns (product, residual). One launch for 1 and 2
    rows, always ahead there (us, two launches and one: 11.9, 10.5 at one row of
    6144 x 4096, 13.6, 11.4 at two); more rows cost every workgroup more than a
    launch is worth."""
    if norm_fits(x, residual, norm, w) and _plain_bias(bias, w):
        out = torch.empty(x.size(0), w.size(0) // (2 if glu else 1),
                          dtype=x.dtype, device=x.device)
        stream = torch.empty_like(x)
        _K.skinny_norm(out, stream, x, residual, norm, eps, w, _none(bias, x),
                       glu)
        return out, stream
    x, residual = fused_add_rms_norm(x, residual, norm, eps)
    return (linear_swiglu(x, w) if glu else linear(x, w, bias)), residual


def norm_fits(x, residual, norm, w) -> bool:
    """Whether add_norm_linear of these is one launch."""
    return x.dim() == 2 and x.size(0) <= 2 and _plain_rows(x, w, 2) \
        and _norm_rows(x, residual, norm)


def _norm_rows(x, residual, norm) -> bool:
    """Rows that a product can norm on the way."""
    return x.size(1) % 512 == 0 and x.size(1) <= 8192 and x.is_contiguous() \
        and residual.is_contiguous() and residual.shape == x.shape and norm.is_contiguous() \
        and all(t.dtype == torch.bfloat16 and t.device == x.device
                and t.data_ptr() % 16 == 0 for t in (residual, norm)) \
        and not (torch.is_grad_enabled() and (
            residual.requires_grad or norm.requires_grad))


def reshape_and_cache(k: torch.Tensor, v: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, slot_mapping: torch.Tensor) -> None:
    """k/v: [T, KH, D] (rows may be strided views into a fused qkv buffer)."""
    if k.is_cuda:
        _K.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
        return
    torch_ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def _whole_chunks(*rows: torch.Tensor) -> bool:
    """bf16 rows of whole 16-byte chunks"""
    return all(t.dim() == 2 and t.dtype == torch.bfloat16 and t.stride(1) == 1
               and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0
               for t in rows)


def rope_and_cache(positions: torch.Tensor, q: torch.Tensor, k: torch.Tensor,
                   v: torch.Tensor, head_dim: int, cos_sin: torch.Tensor,
                   k_cache: torch.Tensor, v_cache: torch.Tensor,
                   slot_mapping: torch.Tensor):
    """rotary_embedding of q and k [T, heads * head_dim], then
    reshape_and_cache of k and v. Returns (q, k). One launch for rows of
    whole 16-byte chunks."""
    if q.is_cuda and _whole_chunks(q, k, v) \
            and cos_sin.size(1) % 16 == 0 and cos_sin.size(1) <= head_dim \
            and cos_sin.is_contiguous() and positions.is_contiguous() \
            and head_dim % 8 == 0 and k_cache.size(3) == head_dim \
            and k.size(1) == v.size(1) == k_cache.size(1) * head_dim \
            and slot_mapping.is_contiguous() \
            and positions.numel() == slot_mapping.numel() == q.size(0):
        _K.rope_and_cache(positions, q, k, v, cos_sin, k_cache, v_cache,
                          slot_mapping)
        return q, k
    q, k = rotary_embedding(positions, q, k, head_dim, cos_sin)
    reshape_and_cache(k.unflatten(-1, (-1, head_dim)),
                      v.unflatten(-1, (-1, head_dim)), k_cache, v_cache,
                      slot_mapping)
    return q, k


# decode-attention implementation: "sp" = the matrix-core kernel
# (paged_attention_sp.hip), "fused" = the earlier single-pass one with 4
# waves per pair (paged_attention.hip). Overridable for A/B runs.
import os as _os
_PA_IMPL = _os.environ.get("KAITO_PA_IMPL", "sp")
# fused W4A16 GEMM for M>4: measured slower than dequant+hipBLASLt on
# MI355X (tools/bench_w4a16.py) — off unless explicitly enabled
W4A16_FUSED_GEMM = _os.environ.get("KAITO_W4A16_FUSED", "0") == "1"


def _sinks_arg(sinks, device):
    if sinks is None:
        return torch.empty(0, dtype=torch.float32, device=device)
    return sinks


def paged_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                    block_tables: torch.Tensor, seq_lens: torch.Tensor,
                    scale: float, window: int = 0,
                    sinks: torch.Tensor | None = None) -> torch.Tensor:
    if q.is_cuda:
        out = torch.empty_like(q)
        if _PA_IMPL == "sp" or window > 0 or sinks is not None \
                or k_cache.dtype == torch.uint8:
            # windows, sinks and fp8 pages: the matrix-core kernel only
            _K.paged_attention_sp(
                out, q, k_cache, v_cache, block_tables, seq_lens, scale,
                window, _sinks_arg(sinks, q.device))
        else:
            _K.paged_attention(out, q, k_cache, v_cache,
                                            block_tables, seq_lens, scale)
        return out
    return torch_ref.paged_attention(q, k_cache, v_cache, block_tables,
                                     seq_lens, scale, window, sinks)


def rope_paged_attention(positions: torch.Tensor, q: torch.Tensor,
                         k: torch.Tensor, v: torch.Tensor, head_dim: int,
                         cos_sin: torch.Tensor, k_cache: torch.Tensor,
                         v_cache: torch.Tensor, slot_mapping: torch.Tensor,
                         block_tables: torch.Tensor, seq_lens: torch.Tensor,
                         scale: float, window: int = 0,
                         sinks: torch.Tensor | None = None) -> torch.Tensor:
    """rope_and_cache of q, k and v [T, heads * head_dim], then
    paged_attention: decode rows, each of a sequence of its own with its own
    key as the last of seq_lens. Returns [T, QH, head_dim]; q and k may or may
    not be rotated afterwards. One launch for rotations of whole heads, up to
    8192 (row, kv head) pairs: every wave rotates its queries anew (one launch
    and two, us, 8 kv heads of 128: 1 row of 217 keys 7.6, 9.3; 16 of 3000 in
    fp8 27.0, 29.8; 250 of 300 55.3, 56.4; 512 of 300 105, 107; 2048 of 220
    296, 291). Two over one, 14 layouts of 1 to 32 kv heads of 64, 128 and 256
    dims, bf16 and fp8: 1.02 to 1.38 to 1024 pairs, with 220 and 1000 keys 0.97
    to 1.26 at 2048 to 6144 and 0.99 to 1.12 at 8192; with 30 keys, whose
    attention is hardly more than the rotations, 0.91 to 1.39 and 0.89 to 1.05
    there, which the step's lengths on the device do not tell."""
    QH, KH = q.size(1) // head_dim, k_cache.size(1)
    if q.is_cuda and _PA_IMPL == "sp" and q.size(0) * KH <= 8192 \
            and _whole_chunks(q, k, v) and cos_sin.size(1) == head_dim and head_dim in (64, 128, 256) \
            and k_cache.size(2) == 16 and k_cache.size(3) == head_dim \
            and k.size(1) == v.size(1) == KH * head_dim \
            and k_cache.is_contiguous() and v_cache.is_contiguous() \
            and cos_sin.is_contiguous() and cos_sin.data_ptr() % 16 == 0 \
            and positions.is_contiguous() and slot_mapping.is_contiguous() \
            and positions.numel() == slot_mapping.numel() == q.size(0) \
            == seq_lens.numel():
        out = torch.empty(q.size(0), QH, head_dim, dtype=q.dtype,
                          device=q.device)
        _K.rope_paged_attention(
            out, positions, q.unflatten(-1, (QH, head_dim)), k, v, cos_sin,
            k_cache, v_cache, slot_mapping, block_tables, seq_lens, scale,
            window, _sinks_arg(sinks, q.device))
        return out
    q, k = rope_and_cache(positions, q, k, v, head_dim, cos_sin, k_cache,
                          v_cache, slot_mapping)
    return paged_attention(q.unflatten(-1, (QH, head_dim)), k_cache, v_cache,
                           block_tables, seq_lens, scale, window, sinks)


def mla_decode(q: torch.Tensor, cache: torch.Tensor,
               block_tables: torch.Tensor, seq_lens: torch.Tensor,
               scale: float, r: int,
               q_rope: torch.Tensor | None = None) -> torch.Tensor:
    """Absorbed MLA decode over the compressed latent cache (DeepSeek).
    q: [T, H, r+rope], or [T, H, r] with q_rope [T, H, rope], of any token
    and head strides; cache: [NB, BS, r+rope] bf16. Returns [T, H, r]."""
    if q.is_cuda:
        if q_rope is None:
            assert q.is_contiguous()
            q, q_rope = q[..., :r], q[..., r:]
        out = torch.empty(q.size(0), q.size(1), r, dtype=q.dtype,
                          device=q.device)
        _K.mla_decode(out, q, q_rope, cache, block_tables, seq_lens, scale)
        return out
    if q_rope is not None:
        q = torch.cat([q, q_rope], -1)
    return torch_ref.mla_decode(q, cache, block_tables, seq_lens, scale, r)


def mla_prepare(q: torch.Tensor, kv_a: torch.Tensor, w: torch.Tensor,
                eps: float, positions: torch.Tensor, cos_sin: torch.Tensor,
                cache: torch.Tensor | None, slots: torch.Tensor | None):
    """GPU only: rotated q [T, H, 64] (any token and head strides), the
    normed latent and the rotated key part of kv_a [T, 512 + 64], both
    scattered into the cache, if one is given, as by mla_cache_write."""
    T, H, P = q.shape
    q_out = torch.empty(T, H, P, dtype=q.dtype, device=q.device)
    c = torch.empty(T, w.numel(), dtype=q.dtype, device=q.device)
    k = torch.empty(T, P, dtype=q.dtype, device=q.device)
    _K.mla_prepare(q_out, c, k, _none(cache, q), q, kv_a, w, eps, positions,
                   cos_sin, positions if slots is None else slots)
    return q_out, c, k


def _head_rows_fit(x: torch.Tensor, w: torch.Tensor) -> bool:
    """The library is ahead from 32 rows of 128 heads on (us, 512 x 128: 14.4,
    13.8; 24 rows 13.0, 13.6; 64 heads 8.9, 12.9; 16 heads 6.7, 12.8)."""
    T, H, K = x.shape
    return x.is_cuda and x.dtype == w.dtype == torch.bfloat16 and T <= 32 \
        and T * H <= 3072 and K % 64 == 0 and 0 < K <= 512 \
        and w.size(2) % 32 == 0 and w.is_contiguous() \
        and w.data_ptr() % 16 == 0 and x.stride(2) == 1 \
        and x.stride(0) % 4 == 0 and x.stride(1) % 4 == 0 \
        and x.data_ptr() % 8 == 0


def head_rows(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [T, H, K] (any token and head strides) times w [H, K, N] per head:
    [T, H, N]. One launch for up to 32 rows, a batched library product and
    its transposition beyond: W is read once per 32 rows."""
    if _head_rows_fit(x, w):
        y = torch.empty(*x.shape[:2], w.size(2), dtype=x.dtype,
                        device=x.device)
        _K.head_rows(y, x, w)
        return y
    return torch.bmm(x.transpose(0, 1), w).transpose(0, 1)


def mla_prepare_rows(x: torch.Tensor, wx: torch.Tensor, q: torch.Tensor,
                     kv_a: torch.Tensor, w: torch.Tensor, eps: float,
                     positions: torch.Tensor, cos_sin: torch.Tensor,
                     cache: torch.Tensor | None, slots: torch.Tensor | None):
    """(head_rows(x, wx), *mla_prepare(q, ...)); one launch where head_rows
    is one."""
    if not _head_rows_fit(x, wx) or x.size(0) != q.size(0):
        return head_rows(x, wx), *mla_prepare(q, kv_a, w, eps, positions,
                                              cos_sin, cache, slots)
    T, H, P = q.shape
    y, q_out, c, k = (torch.empty(*s, dtype=q.dtype, device=q.device)
                      for s in ((T, x.size(1), wx.size(2)), (T, H, P),
                                (T, w.numel()), (T, P)))
    _K.mla_prepare_rows(q_out, c, k, _none(cache, q), q, kv_a, w, eps,
                        positions, cos_sin,
                        positions if slots is None else slots, y, x, wx)
    return y, q_out, c, k


def mla_cache_write(cache: torch.Tensor, c_kv: torch.Tensor,
                    k_pe: torch.Tensor, slots: torch.Tensor) -> None:
    """Scatter latent rows (c_kv ‖ k_pe) into the paged MLA cache;
    negative slots (graph-bucket padding) are skipped."""
    _K.mla_cache_write(cache, c_kv, k_pe, slots)


def prefill_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                      cu_seqlens: torch.Tensor, scale: float,
                      max_seqlen: int | None = None, window: int = 0,
                      sinks: torch.Tensor | None = None,
                      tiles=None) -> torch.Tensor:
    """Causal attention of whole prompts. `tiles` = (tile_seq, tile_qbase)
    of build_query_tiles spares a read of cu_seqlens on the host."""
    if q.is_cuda:
        out = torch.empty_like(q)
        tile_seq, tile_qbase = tiles or _build_tiles(cu_seqlens)
        _K.prefill_attention(out, q, k, v, tile_seq, tile_qbase,
                                          cu_seqlens, scale, window,
                                          _sinks_arg(sinks, q.device),
                                          max_seqlen or 0)
        return out
    return torch_ref.prefill_attention(q, k, v, cu_seqlens, scale, window,
                                       sinks)


def latent_kv(c: torch.Tensor, w_kc: torch.Tensor, w_vc: torch.Tensor):
    """Keys [T, H, D] and values [T, H, V] of latent rows c [T, r]: c times
    w_kc [H, D, r] and w_vc [H, r, V]. One launch (and a transposition of
    w_vc) for prompts that fill the chip with 256 x 256 tiles, library products
    else (us, library and tiles, 128 + 128 dims of 512: 8192 rows of 16 heads
    59.2, 41.0, 4096 34.0, 27.0, 2048 21.5, 21.6; 4096 of 128 heads 208, 134,
    512 31.9, 32.7)."""
    T, (H, D, r), V = c.size(0), w_kc.shape, w_vc.size(2)
    if c.is_cuda and _latent_tiles(T, H * (D + V), r) and T < 1 << 22 \
            and c.dtype == w_kc.dtype == w_vc.dtype == torch.bfloat16 \
            and H * D % 256 == V % 64 == r % 64 == 0 \
            and w_vc.shape[:2] == (H, r) and not _transformed() and all(
                t.is_contiguous() and t.data_ptr() % 16 == 0
                and not (torch.is_grad_enabled() and t.requires_grad)
                for t in (c, w_kc, w_vc)):
        kv = torch.empty(T, H * (D + V), dtype=c.dtype, device=c.device)
        _K.latent_kv(kv, c, w_kc, w_vc)
        return kv[:, :H * D].unflatten(-1, (H, D)), \
            kv[:, H * D:].unflatten(-1, (H, V))
    k = linear(c.to(w_kc.dtype), w_kc.view(H * D, r)).view(T, H, D)
    v = torch.matmul(c.to(w_vc.dtype).unsqueeze(0), w_vc)
    return k, v.transpose(0, 1)


def _latent_tiles(T: int, N: int, r: int) -> bool:
    """From a product of 4096 x 4096 on (library over tiles; 16 to 128 heads of 256
    dims there: 1.19, 1.22, 1.14 with 256 latent columns, 1.19, 1.26, 1.12 with 512,
    1.20, 1.18, 1.07 with 1024, 1.19, 1.15, 1.10 with 1536; half as large 1.02, 0.99,
    0.90, 0.99, 0.79, 0.91, 0.95, 0.89; larger 1.1 to 2.0). Few tokens of many heads
    are about even to 512 columns (128 heads of 512 tokens 0.93, 0.98, 256 of 256
    0.99), beyond not before 640 (128 heads 0.96 at 512, 1.02 at 513, 1.20 at 640; 256
    heads 0.71 at 256, 0.80 at 512)."""
    return T * N >= 4096 * 4096 and (r <= 512 or T >= 640)


def mla_prefill_attention(q, q_pe, k, k_pe, v, cu_seqlens, scale: float,
                          tiles=None) -> torch.Tensor:
    """Causal latent attention of whole prompts (GPU, bf16): q [T, H, 128]
    beside q_pe [T, H, 64], k [T, H, 128] beside k_pe [T, 64] shared by the
    heads, v [T, H, 128]; token and head strides are free. -> [T, H, 128]."""
    out = torch.empty(v.shape, dtype=v.dtype, device=v.device)
    tile_seq, tile_qbase = tiles or _build_tiles(cu_seqlens)
    _K.mla_prefill_attention(out, q, q_pe, k, k_pe, v, tile_seq, tile_qbase,
                             cu_seqlens, scale)
    return out


def context_attention(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, cu_seqlens_q: torch.Tensor,
                      kv_lens: torch.Tensor, block_tables: torch.Tensor,
                      scale: float, window: int = 0,
                      sinks: torch.Tensor | None = None,
                      tiles=None) -> torch.Tensor:
    """Suffix-query causal attention over the paged cache (chunked
    prefill / prefix-cache continuation). `tiles` as in
    prefill_attention."""
    if q.is_cuda:
        out = torch.empty_like(q)
        tile_seq, tile_qbase = tiles or _build_tiles(cu_seqlens_q)
        _K.context_attention(out, q, k_cache, v_cache, tile_seq,
                                          tile_qbase, cu_seqlens_q, kv_lens,
                                          block_tables, scale, window,
                                          _sinks_arg(sinks, q.device))
        return out
    return torch_ref.context_attention(q, k_cache, v_cache, cu_seqlens_q,
                                       kv_lens, block_tables, scale, window,
                                       sinks)


def gelu_and_mul(x: torch.Tensor) -> torch.Tensor:
    """GeGLU: gelu_tanh(x[..., :d]) * x[..., d:] (gemma MLPs)."""
    if x.is_cuda:
        d = x.size(-1) // 2
        out = torch.empty(*x.shape[:-1], d, dtype=x.dtype, device=x.device)
        _K.gelu_and_mul(out, x)
        return out
    return torch_ref.gelu_and_mul(x)


def gelu(x: torch.Tensor) -> torch.Tensor:
    """Plain tanh-approx GELU (phi-2 ungated MLP)."""
    if x.is_cuda:
        out = torch.empty_like(x)
        _K.gelu(out, x.contiguous())
        return out
    return torch_ref.gelu_tanh(x)


def layer_norm(x: torch.Tensor, weight: torch.Tensor,
               bias: torch.Tensor | None, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        b = bias if bias is not None else \
            torch.empty(0, dtype=x.dtype, device=x.device)
        _K.layer_norm(out, x, weight, b, eps)
        return out
    return torch_ref.layer_norm(x, weight, bias, eps)


def fused_add_layer_norm(x: torch.Tensor, residual: torch.Tensor,
                         weight: torch.Tensor, bias: torch.Tensor | None,
                         eps: float):
    """Returns (normed, residual); residual += x in place on GPU."""
    if x.is_cuda:
        out = torch.empty_like(x)
        b = bias if bias is not None else \
            torch.empty(0, dtype=x.dtype, device=x.device)
        _K.fused_add_layer_norm(out, x, residual, weight, b, eps)
        return out, residual
    new_res = (x.float() + residual.float()).to(x.dtype)
    return torch_ref.layer_norm(new_res, weight, bias, eps), new_res


def mfma_tile_gemm(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return _K.mfma_tile_gemm(a, b)


QTILE = 64  # query tiles of a step's chunks: flash_prefill.h TILE


def _build_tiles(cu_seqlens: torch.Tensor):
    """build_query_tiles for callers that hold the offsets on the device."""
    cs = cu_seqlens.tolist()
    return build_query_tiles([b - a for a, b in zip(cs, cs[1:])],
                             cu_seqlens.device)


def moe_gate_silu(act: torch.Tensor, x: torch.Tensor,
                  w_gate_up: torch.Tensor, sorted_ids: torch.Tensor,
                  offsets: torch.Tensor, e_base: int,
                  n_local_experts: int, bias: torch.Tensor | None = None,
                  act_mode: int = 0, act_limit: float = 7.0) -> None:
    """Fused MoE stage 1 (GPU only): gather rows by sorted token ids,
    gate/up grouped GEMM per expert, activation epilogue into `act`
    (act_mode 0 = SwiGLU, 1 = clamped swiglu min(g, limit)·sigmoid(1.702
    g)·(clamp(u, ±limit) + 1); optional
    per-expert [E, 2*IE] bias; 2 = ungated squared relu with weights
    [E, IE, H])."""
    b = bias if bias is not None else         torch.empty(0, dtype=x.dtype, device=x.device)
    _K.moe_gate_silu(act, x, w_gate_up, sorted_ids, offsets, b, act_mode,
                     e_base, n_local_experts, act_limit)


def moe_down_rows(y, act, w_down, offsets, e_base: int, n_local_experts: int,
                  bias=None) -> None:
    """Stage 2 of decode-sized steps (GPU only): y [TK, H] f32, the down
    product (+ optional [E, H] bias) of every sorted row."""
    _K.moe_down_rows(y, act, w_down, offsets, _none(bias, act), e_base,
                     n_local_experts)


PAIRS_MAX = 256       # pairs of a step whose experts find their own rows


def moe_pairs_pay(pairs: int, n_local: int, up_rows: int, H: int) -> bool:
    """Whether a step's local experts, of up_rows x H, find their rows among
    the pairs. The sort's launch is saved, and every workgroup of 16 weight rows
    scans them, of experts that no token chose too. us a layer, sorted and by
    pairs: 8 experts of 2048 x 2048 (3072 workgroups), top 2, 19.9, 18.5 at 1
    token, 26.5, 22.6 at 2, 43.0, 39.9 at 16, 73.9, 71.6 at 128; 12 of 2048 x 1408
    (3648), top 3, 21.7, 19.2 at 1. More workgroups need more pairs: 8 of 4096 x
    4096 (6144) 43.7, 44.8 at 1, 61.0, 65.1 at 2, 112.4, 112.6 at 8, 127.2, 125.8
    at 12; with H of 2048, where they stay for several tiles, 16 of 2048 x 1024
    (4096), top 4, 19.9, 20.5 at 1, 28.6, 25.7 at 2, 16 of 2048 x 2048 (6144) 33.2,
    34.6 at 3, 36.8, 31.3 at 4. 8 of 4096 x 14336 (16384) 118, 122 and 179, 185 at
    1 and 2; 32 of 2048 x 2048 (12288) 21.2, 25.3 at 1; 24 of 2048 x 1024, top 4,
    19.9, 20.9 at 1; 128 of 2048 x 768, top 8, 32.5, 41.2 and 191, 221 at 1 and
    32."""
    workgroups = n_local * (up_rows + H) // 16
    if pairs > PAIRS_MAX or n_local > 16 or workgroups > 8704:
        return False
    return workgroups <= 3840 or \
        pairs >= (n_local // 2 if H == 2048 else 2 * n_local)


def moe_shared_pays(T: int, pairs: int, n_experts: int, H: int,
                    I: int) -> bool:
    """Whether an expert of every token, of the routed ones' sizes H x I, runs in
    their launches (us, products of its own and beside, up and down together; 8
    of 2048 x 2048, top 2: 44.9, 39.2 at 4 tokens, 54.7, 46.9 at 32; 16 of 1024 x
    512, top 4, 1.05 to 1.41 times as fast, 8 of 7168 x 2048, top 8, 1.03 to 1.07,
    8 of 4096 x 4096, top 2, 1.05 at 8 to 16). Its rows beyond 16 are a second pass
    over its weights unless the others have two tiles of rows too (more than 12
    pairs an expert), which wide or few experts do not win back: 8 of 4096 x 4096
    0.93 to 0.96 at 17 to 32, 4 of 4096 x 8192, top 1, 0.84 to 0.88, 16 of 5120 x
    1536, top 6, 0.95 at 32, 4 of 2048 x 2048 0.85 at 24 and 1.01 at 32; 6 of 2880
    x 2880 1.09 to 1.13. One token of very large ones: 4 of 2048 x 8192 61.8,
    65.4, 8 of 2048 x 4096 40.5, 37.6."""
    if T > 16:
        return T <= 32 and (pairs > 12 * n_experts
                            or (H < 3072 and n_experts > 4))
    return T > 1 or I <= 4096


def moe_up_pairs(act, x, w_gate_up, topi, n_experts: int, e_base: int,
                 n_local_experts: int, bias=None, act_mode: int = 0,
                 act_limit: float = 7.0, all_w=None, all_act=None) -> None:
    """moe_gate_silu with the rows of `act` in the order of the pairs of
    `topi` [T, top] int32, up to PAIRS_MAX of them: no sort (GPU only).
    all_w [2 IE, H]: an expert of every token beside them (SwiGLU, no
    biases), its rows go to all_act [T, IE]."""
    _K.moe_up_pairs(act, x, w_gate_up, topi, _none(bias, x), act_mode,
                    n_experts, e_base, n_local_experts, act_limit,
                    _none(all_w, x), _none(all_act, x))


def moe_down_pairs(y, act, w_down, topi, n_experts: int, e_base: int,
                   n_local_experts: int, bias=None, all_w=None, all_act=None,
                   all_y=None) -> None:
    """moe_down_rows with rows in the order of the pairs (GPU only). all_w
    [H, IE]: the expert of every token, all_y [T, H] bf16 its result."""
    _K.moe_down_pairs(y, act, w_down, topi, _none(bias, act), n_experts,
                      e_base, n_local_experts, _none(all_w, y),
                      _none(all_act, y), _none(all_y, y))


def moe_grouped_up(act, x, w, sorted_ids, offsets, e_base: int, bias=None,
                   act_mode: int = 0, act_limit: float = 7.0) -> None:
    """moe_gate_silu for prompt-sized steps (GPU, bf16): `act` [TK, IE]
    exactly, widths multiples of 64, every tile bound read on the device."""
    _K.moe_grouped_up(act, x, w, sorted_ids, offsets, _none(bias, x),
                      act_mode, e_base, act_limit)


def moe_grouped_down(y, act, w, offsets, e_base: int, bias=None) -> None:
    """y[s] = act[s] w[e]^T (+ bias) of the sorted rows (GPU, bf16; y bf16
    or f32)."""
    _K.moe_grouped_down(y, act, w, offsets, _none(bias, act), e_base)


def moe_combine(out, y, pos, topi, topw, e_base: int, e_local: int, x=None,
                w_id=None, shared=None) -> None:
    """out[t] = sum over t's choices of topw * y[pos] (experts e_base ..
    e_base + e_local) + w_id x + shared, summed in f32; out bf16 or f32. pos
    None: rows of y in the order of the pairs."""
    _K.moe_combine(out, y, _none(pos, y), topi, topw,
                   out if w_id is None else x, _none(w_id, y),
                   _none(shared, y), e_base, e_local)


def moe_combine_norm(residual, weight, eps: float, y, pos, topi, topw,
                     e_base: int, e_local: int, x=None, w_id=None,
                     shared=None):
    """moe_combine rounded to bf16, then (GPU, rows up to 8192) with a bf16
    residual fused_add_rms_norm, with an f32 one post_norm_residual, in
    place. Returns the bf16 rows of those."""
    out = torch.empty(residual.shape, dtype=torch.bfloat16,
                      device=residual.device)
    _K.moe_combine_norm(out, residual, y, _none(pos, y), topi, topw,
                        out if w_id is None else x, _none(w_id, y),
                        _none(shared, y), weight, eps, e_base, e_local)
    return out


ROUTE_MAX = 1024      # router outputs of the kernels; more run as torch ops
ROUTE_MODES = {"softmax": 0, "sigmoid": 1, "logits": 2}


def _route_out(T: int, top: int, device):
    f32 = dict(dtype=torch.float32, device=device)
    return (torch.empty(T, top, dtype=torch.int32, device=device),
            torch.empty(T, top, **f32), torch.empty(T, **f32))


def moe_route(logits, correction, top: int, n_real: int, groups: int = 1,
              keep: int = 1, renorm: bool = False, scale: float = 1.0,
              mode: str = "softmax"):
    """Expert choice from f32 router logits [T, N]: scores s = softmax (or,
    by `mode`, sigmoid); the choice adds `correction` [N] f32 (None:
    nothing); outputs form `groups` equal groups of neighbours scored by
    their largest choice (sigmoid: the sum of their two largest), of which
    the `keep` best stay eligible; the `top` largest eligible choices are
    taken. Weights are s (without the correction), over their sum + 1e-20
    with `renorm`, times scale. Mode "logits" chooses by the logits and
    weighs by a softmax over the taken ones. Returns (indices [T, top]
    int32, weights [T, top] f32, summed weight [T] f32 of the taken outputs
    with index >= n_real)."""
    if logits.is_cuda and logits.size(1) <= ROUTE_MAX and top <= 64 \
            and groups <= 64:
        topi, topw, w_id = _route_out(logits.size(0), top, logits.device)
        _K.moe_route(topi, topw, w_id, logits, _none(correction, logits),
                     n_real, groups, keep, renorm, scale, ROUTE_MODES[mode])
        return topi, topw, w_id
    return torch_ref.moe_route(logits, correction, top, n_real, groups, keep,
                               renorm, scale, mode)


def _router_logits(x: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """x gate^T in f32, whatever the operands and the number of rows: a
    token's experts do not hang on the length of the step it came in. (bf16
    logits, widened afterwards, take a launch more: 8192 rows of 2048 to 8
    outputs 11.1 us, f32 ones 9.0; 32 rows of 7168 to 256 outputs 12.6 and
    10.7.)"""
    if x.is_cuda and x.dtype == gate.dtype == torch.bfloat16:
        return torch.mm(x, gate.t(), out_dtype=torch.float32)
    return torch.nn.functional.linear(x.float(), gate.float())


def _gate_short(x, gate) -> bool:
    T = x.size(0)
    return T <= 512 and T * gate.size(0) <= 8192


def _gate_long(T: int, N: int, H: int, f32: bool) -> bool:
    """Whether tiles of 16 rows form the logits of a long step. us, library and
    choice, and tiles; T rows, N outputs, rows of H. An f32 router saves the cast
    of the rows: 8 outputs 15.7, 8.4 and 38.0, 14.4 (600 and 8192 rows of 2048),
    32 outputs 16.5, 13.0 and 37.7, 26.4; beyond 16 outputs and H of 3072 only from
    1024 rows on (32 x 7168: 27.7, 34.3 at 257, 33.8, 34.6 at 600, 38.2, 35.0 at
    1024). A bf16 one has to be small: 8 outputs 9.1, 7.0 and 14.7, 10.8, of 4096
    9.8, 9.7 and 19.1, 17.9; 16 outputs 9.2, 7.6 and 15.0, 12.1, of 2880 11.3, 9.0,
    of 3072 9.2, 9.3, of 4096 9.8, 11.0; 32 outputs of 2048 15.7, 16.0 at 8192."""
    if H % 32 or N > 32:
        return False
    if f32:
        return N <= 16 or H <= 3072 or T >= 1024
    return N <= 16 and H <= 2880 or N <= 8 and H <= 4096


def _gate_in_route(x, gate) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 and gate.size(0) <= 32
            and gate.is_contiguous()
            and gate.dtype in (torch.bfloat16, torch.float32)
            and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.size(1) % 8 == 0 and x.data_ptr() % 16 == 0
            and gate.data_ptr() % 16 == 0)


def moe_norm_gate_route(x, residual, norm_w, eps: float, gate, correction,
                        top: int, n_real: int, groups: int = 1, keep: int = 1,
                        renorm: bool = False, scale: float = 1.0,
                        mode: str = "softmax"):
    """fused_add_rms_norm, then moe_gate_route of its rows: (rows, residual,
    indices, weights, identity weight); one launch where the choice is."""
    def aligned(t):
        return t.dtype == torch.bfloat16 and t.is_contiguous() \
            and t.data_ptr() % 16 == 0
    if _gate_short(x, gate) and _gate_in_route(x, gate) \
            and aligned(x) and aligned(residual) \
            and aligned(norm_w) and residual.shape == x.shape \
            and x.size(1) <= 8192:
        topi, topw, w_id = _route_out(x.size(0), top, x.device)
        xn = torch.empty_like(x)
        _K.moe_norm_gate_route(topi, topw, w_id, xn, residual, x, norm_w, eps,
                               gate, _none(correction, x), n_real, groups,
                               keep, renorm, scale, ROUTE_MODES[mode])
        return xn, residual, topi, topw, w_id
    xn, residual = fused_add_rms_norm(x, residual, norm_w, eps)
    return (xn, residual) + moe_gate_route(
        xn, gate, correction, top, n_real, groups, keep, renorm, scale, mode)


def moe_gate_route(x, gate, correction, top: int, n_real: int,
                   groups: int = 1, keep: int = 1, renorm: bool = False,
                   scale: float = 1.0, mode: str = "softmax"):
    """moe_route of the logits x gate^T, formed in f32. One launch for short
    steps and narrow routers: a workgroup per row reads the whole router, 8
    outputs after one another, so that wider ones and longer steps take tiles
    of 16 rows (_gate_long) or leave the product to the library. us, one launch
    and two; rows of 2048 and 7168, bf16 router: 8 outputs 5.1, 9.4 and 6.1,
    13.2 at 32 rows, 5.7, 9.5 and 7.0, 11.4 at 512; 32 outputs 9.2, 9.6 and
    12.2, 13.7 at 32 rows, 9.6, 9.6 and 13.3, 13.7 at 256, 10.3, 9.7 and 16.0,
    13.9 at 512; 48 outputs 12.0, 9.5 and 16.5, 13.6 at 32."""
    T = x.size(0)
    long = _gate_long(T, gate.size(0), x.size(1),
                      gate.dtype == torch.float32)
    if (long or _gate_short(x, gate)) and _gate_in_route(x, gate):
        topi, topw, w_id = _route_out(T, top, x.device)
        _K.moe_gate_route(topi, topw, w_id, x, gate, _none(correction, x),
                          n_real, groups, keep, renorm, scale,
                          ROUTE_MODES[mode])
        return topi, topw, w_id
    return moe_route(_router_logits(x, gate), correction, top, n_real, groups, keep, renorm,
                     scale, mode)


def moe_plan(topi, topw, n: int):
    """moe_sort, and the sorted row of every pair ([TK] int32)."""
    if topi.is_cuda and n <= ROUTE_MAX:
        TK, dev = topi.numel(), topi.device
        tok = torch.empty(TK, dtype=torch.int32, device=dev)
        pos = torch.empty(TK, dtype=torch.int32, device=dev)
        gates = torch.empty(TK, dtype=torch.float32, device=dev)
        offsets = torch.empty(n + 1, dtype=torch.int32, device=dev)
        _K.moe_sort(tok, gates, offsets, pos, topi, topw)
        return tok, gates, offsets, pos
    return torch_ref.moe_plan(topi, topw, n)


def moe_sort(topi, topw, n: int):
    """(token, expert) pairs ordered by expert, stable: (token of each
    sorted row [TK] int32, its weight [TK] f32, exclusive offsets [n + 1]
    int32)."""
    return moe_plan(topi, topw, n)[:3]


def w4a16_gemv(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor,
               zeros: torch.Tensor, group: int) -> torch.Tensor:
    """Group-quantized W4A16 linear, small M (decode): out = x @ W^T with
    W dequantized on the fly inside the kernel."""
    if x.is_cuda:
        x = x.contiguous()
        out = torch.empty(x.size(0), qweight.size(0), dtype=x.dtype,
                          device=x.device)
        _K.w4a16_gemv(out, x, qweight, scales, zeros, group)
        return out
    return torch_ref.w4a16_gemv(x, qweight, scales, zeros, group)


def w4a16_swiglu(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor,
                 zeros: torch.Tensor, group: int):
    """silu(x Wg^T) * (x Wu^T) of the packed W = [Wg | Wu] in one launch, for
    a few rows x [M, K]; None for other sizes."""
    N, K = qweight.size(0) // 2, x.size(1)
    if not (x.is_cuda and x.dtype == torch.bfloat16 and x.size(0) <= 16
            and qweight.size(0) % 2 == 0 and x.data_ptr() % 16 == 0
            and qweight.data_ptr() % 16 == 0
            and _K.w4a16_in_tiles(x.size(0), 2 * N, K, group, True)):
        return None
    out = torch.empty(x.size(0), N, dtype=x.dtype, device=x.device)
    _K.w4a16_swiglu(out, x.contiguous(), qweight, scales, zeros, group)
    return out


def _packed_norm_rows(x, residual, norm, qweight) -> bool:
    """Rows that a product with packed weights can norm on the way."""
    return x.is_cuda and x.dim() == 2 and 1 <= x.size(0) <= 2 \
        and x.dtype == torch.bfloat16 and x.data_ptr() % 16 == 0 \
        and qweight.data_ptr() % 16 == 0 and _norm_rows(x, residual, norm) \
        and not (torch.is_grad_enabled() and x.requires_grad) \
        and not _transformed()


def w4a16_norm_linear(x, residual, norm, eps: float, qweight, scales, zeros,
                      group: int, glu: bool = False):
    """w4a16_gemv (glu: SwiGLU of the pair) of fused_add_rms_norm's rows and its
    residual, of 1 and 2 rows in one launch; None for other sizes."""
    if not (_packed_norm_rows(x, residual, norm, qweight)
            and qweight.is_contiguous() and scales.is_contiguous()
            and zeros.is_contiguous() and qweight.size(0) % (2 if glu else 1) == 0
            and _K.w4a16_norm_in_tiles(x.size(0), qweight.size(0), x.size(1),
                                       group, glu)):
        return None
    out = torch.empty(x.size(0), qweight.size(0) // (2 if glu else 1),
                      dtype=x.dtype, device=x.device)
    stream = torch.empty_like(x)
    _K.w4a16_norm_linear(out, stream, x, residual, norm, eps, qweight, scales,
                         zeros, group, glu)
    return out, stream


def w4a16_streams(x: torch.Tensor, group: int) -> bool:
    """Whether x [M, K] runs on the packed weights (w4a16_gemv) or on a
    dequantized copy through the library's GEMM: M <= 4 always; up to 32
    rows in the kernel's slices of 64 k (8 llama-3.1-8b layers' linears at M
    = 16: 96 us a layer, of which 75 more for the copy alone)."""
    return x.size(0) <= 4 or (
        x.is_cuda and x.size(0) <= 32 and x.dtype == torch.bfloat16
        and x.size(1) % 64 == 0 and group % 64 == 0)


def w4a16_dequant(qweight: torch.Tensor, scales: torch.Tensor,
                  zeros: torch.Tensor, group: int,
                  out: torch.Tensor = None) -> torch.Tensor:
    """Dequantize packed 4-bit weights to bf16 [N, K] (feeds hipBLASLt
    MFMA for large-M GEMMs)."""
    if qweight.is_cuda:
        if out is None:
            out = torch.empty(qweight.size(0), qweight.size(1) * 8,
                              dtype=torch.bfloat16, device=qweight.device)
        _K.w4a16_dequant(out, qweight, scales, zeros, group)
        return out
    ref = torch_ref.w4a16_unpack(qweight, scales, zeros, group)
    return ref.to(torch.bfloat16) if out is None else out.copy_(ref)


def w4a16_gemm(x: torch.Tensor, qweight: torch.Tensor, scales: torch.Tensor,
               zeros: torch.Tensor, group: int) -> torch.Tensor:
    """Fused inline-dequant MFMA GEMM (GPU): y = x @ dequant(W)^T.
    The 4-bit weights never round-trip through a full-precision scratch
    buffer. CPU falls back to the unpack reference."""
    if x.is_cuda:
        out = torch.empty(x.size(0), qweight.size(0), dtype=x.dtype,
                          device=x.device)
        _K.w4a16_gemm(out, x.contiguous(), qweight, scales,
                                   zeros, group)
        return out
    return torch_ref.w4a16_gemv(x, qweight, scales, zeros, group)


# ---- stateful sequence mixers (hybrid stacks; kernel group "mix") --------
#
# Batch layout shared by these ops: the rows of all chunks of a step are
# concatenated; chunk b owns rows cu_seqlens[b]..cu_seqlens[b+1], belongs
# to the sequence held in state slot state_slots[b] (<0: padding, skipped)
# and starts at sequence position seq_starts[b] (0: fresh sequence, the
# slot's old content is ignored). token_seq[t] is the chunk of row t.
# Activations may be bf16 or f32 (one dtype per call); states, small
# per-channel parameters and all recurrence math are f32.

def _none(t, like):
    return t if t is not None else \
        torch.empty(0, dtype=torch.float32, device=like.device)


def causal_conv_update(x, weight, bias, conv_state, cu_seqlens, state_slots,
                       seq_starts, token_seq, act: int = 0):
    """Depthwise causal short convolution with a carried tail.
    x [T, C] (row stride free); weight [C, taps] f32; conv_state
    [slots, taps-1, C] in x's dtype, advanced in place; act 0 none,
    1 silu. Returns [T, C]."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _K.causal_conv_update(out, x, weight, _none(bias, x), conv_state,
                              cu_seqlens, state_slots, seq_starts, token_seq,
                              act)
        return out
    return torch_ref.causal_conv_update(x, weight, bias, conv_state,
                                        cu_seqlens, state_slots, seq_starts,
                                        act)


def gated_delta_rule(q, k, v, gate, a, b, a_log, dt_bias, norm_w, state,
                     cu_seqlens, state_slots, seq_starts, qk_eps: float,
                     norm_eps: float):
    """Gated delta rule with fused unit-norm of q/k, decay/beta
    activations, output RMS norm and silu gate. q/k [T, G, D], v/gate
    [T, H, V], a/b [T, H] (row strides free); state [slots, H, D, V] f32
    in place. Returns [T, H*V]."""
    if v.is_cuda:
        T, H, V = v.shape
        out = torch.empty(T, H * V, dtype=v.dtype, device=v.device)
        _K.gated_delta_rule(out, q, k, v, gate, a, b, a_log, dt_bias, norm_w,
                            state, cu_seqlens, state_slots, seq_starts,
                            qk_eps, norm_eps)
        return out
    return torch_ref.gated_delta_rule(
        q, k, v, gate, a, b, a_log, dt_bias, norm_w, state, cu_seqlens,
        state_slots, seq_starts, qk_eps, norm_eps).reshape(v.size(0), -1)


def _rglru_aligned(u, w, bias):
    return u.is_cuda and u.dtype == torch.bfloat16 and w.size(1) in (64, 128) \
        and u.size(0) > 0 and u.stride(1) == 1 and u.stride(0) % 8 == 0 \
        and u.data_ptr() % 16 == 0 and w.is_contiguous() \
        and bias.is_contiguous()


def rglru_gates(u, w, bias):
    """Gate pre-activations of rglru_scan: u [T, B*bw] by blocks of channels
    times w [B, bw, 2*bw] f32, + bias [B, 1, 2*bw] f32, summed in f32.
    Returns [B, T, 2*bw] f32."""
    T, (B, bw, n) = u.size(0), w.shape
    if _rglru_aligned(u, w, bias):
        gates = torch.empty(B, T, n, dtype=torch.float32, device=u.device)
        _K.rglru_gates(gates, u, w, bias)
        return gates
    return torch.baddbmm(bias, u.float().view(T, B, bw).transpose(0, 1), w)


def rglru(u, w, bias, y, decay_rate, state, cu_seqlens, state_slots,
          seq_starts, token_seq=None):
    """rglru_scan of the rows' own rglru_gates."""
    T, B = u.size(0), state_slots.size(0)
    # prompt-sized steps (the rule of the segment-parallel scan): the gates
    # stay in registers. 65 -> 32 us from 128 tokens on, 173 -> 132 at 8192
    if token_seq is not None and _rglru_aligned(u, w, bias) \
            and T >= 4 * B and T >= 128 \
            and y.dtype == u.dtype and y.stride(1) == 1 and state.is_contiguous():
        out = torch.empty(u.shape, dtype=u.dtype, device=u.device)
        _K.rglru_rows(out, u, w, bias, y, decay_rate, state, cu_seqlens,
                      state_slots, seq_starts, token_seq)
        return out
    return rglru_scan(u, rglru_gates(u, w, bias), y, decay_rate, state,
                      cu_seqlens, state_slots, seq_starts, token_seq)


def rglru_scan(u, gates, y, decay_rate, state, cu_seqlens, state_slots,
               seq_starts, token_seq=None):
    """Real-gated linear recurrence + GELU gate branch. u/y [T, W] (row
    strides free); gates [B, T, 2*W/B] f32; decay_rate [W] f32; state
    [slots, W] f32 in place. Returns [T, W]."""
    if u.is_cuda:
        out = torch.empty(u.shape, dtype=u.dtype, device=u.device)
        # with token_seq, prompt-sized steps take the segment-parallel scan
        _K.rglru_scan(out, u, gates, y, decay_rate, state, cu_seqlens,
                      state_slots, seq_starts,
                      token_seq if token_seq is not None else
                      torch.empty(0, dtype=torch.int32, device=u.device))
        return out
    return torch_ref.rglru_scan(u, gates, y, decay_rate, state, cu_seqlens,
                                state_slots, seq_starts)


def qk_norm_cache_write(q, k, v, q_w, k_w, eps: float, k_cache, v_cache,
                        slot_mapping, positions=None, inv_freq=None,
                        rot_mag: float = 1.0, v_first=None,
                        v_lambda: float = 0.0, unit_norm: bool = False,
                        interleaved: bool = False):
    """Per-head RMS norm of q [T, H, D] / k [T, G, D] (f32 weights [D] or
    None), optional rotation (inv_freq [R] f32: dim i of every head is
    paired with dim i + R, or with `interleaved` dim 2i with 2i + 1,
    angle = position * inv_freq[i] in f32, cos and
    sin times rot_mag), optional value blend v <- (1 - v_lambda) v +
    v_lambda v_first, fused with the scatter of k and v [T, G, V] into
    the paged caches [blocks, G, block_size, D|V]. With `unit_norm` (and
    no weights) q and k are divided by their RMS per head after the
    rotation. Returns q normed and rotated, [T, H, D]."""
    if q.is_cuda:
        qn = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        rot = inv_freq is not None and inv_freq.numel() > 0
        _K.qk_norm_cache_write(
            qn, q, k, v, _none(q_w, q), _none(k_w, q), eps, k_cache, v_cache,
            slot_mapping,
            positions if rot else torch.empty(0, dtype=torch.long,
                                              device=q.device),
            inv_freq if rot else _none(None, q), rot_mag,
            v_first if v_first is not None else
            torch.empty(0, dtype=q.dtype, device=q.device), v_lambda,
            unit_norm, interleaved)
        return qn
    return torch_ref.qk_norm_cache_write(q, k, v, q_w, k_w, eps, k_cache,
                                         v_cache, slot_mapping, positions,
                                         inv_freq, rot_mag, v_first, v_lambda,
                                         unit_norm, interleaved)


WINDOW_MFMA_SIZES = (64, 128, 256)          # key sizes of the MFMA kernel
WINDOW_MFMA_VSIZES = (32, 64, 128, 256)     # value sizes


def window_attention(q, k_cache, v_cache, block_tables, token_seq, positions,
                     scale: float, softcap: float = 0.0, r1=None, r2=None,
                     window: int = 0, tiles=None, keep_first: int = 0,
                     sinks=None, chunk: int = 0, sigmoid_bias=None,
                     gate=None, dist_bias=None, temp_coef: float = 0.0,
                     temp_every: int = 1):
    """Causal attention of query rows [T, H, D] over the paged cache (key
    size D, value size V may differ). A query at position i sees keys
    j <= i with i - j < window or j < keep_first (window <= 0: all), or,
    with `chunk` > 0, keys j <= i of i's own block of `chunk` absolute
    positions (block b = positions [b*chunk, (b+1)*chunk)). Options: tanh score capping, the distance penalty
    r1*ln(1 + r2*distance), and per-head `sinks` [H] f32 whose exp joins
    the softmax denominator. With
    `sigmoid_bias` [H] f32 there is no softmax: a visible key's weight is
    sigmoid(score + bias), not normalised over the keys. `gate` [T, H]
    (row stride free) multiplies every head's output by its sigmoid.
    `dist_bias` [H, N] f32: entry min(i - j, N - 1) of the head's row is
    added to the score. `temp_coef` scales the products of the query at
    position i by 1 + temp_coef*ln((i + 1) // temp_every + 1).
    Returns [T, H, V].

    `tiles` = (tile_seq, tile_qbase, cu_seqlens, seq_starts) describes the
    step's chunks as 64-row query tiles (build_query_tiles); with it, bf16
    inputs of supported head sizes take the MFMA prompt kernel. Without
    it (decode steps) or for f32 / other sizes, the one-row-per-workgroup
    f32 kernel runs."""
    if q.is_cuda:
        T, H, D = q.shape
        out = torch.empty(T, H, v_cache.size(3), dtype=q.dtype,
                          device=q.device)
        if (tiles is not None and q.dtype == torch.bfloat16
                and D in WINDOW_MFMA_SIZES
                and v_cache.size(3) in WINDOW_MFMA_VSIZES):
            tile_seq, tile_qbase, cu, starts = tiles
            _K.window_attention_tiles(
                out, q, k_cache, v_cache, block_tables, tile_seq, tile_qbase,
                cu, starts, scale, softcap, _none(r1, q), _none(r2, q),
                window, keep_first, _none(sinks, q), chunk,
                _none(sigmoid_bias, q), _none(gate, q), _none(dist_bias, q),
                temp_coef, temp_every)
            return out
        _K.window_attention(out, q, k_cache, v_cache, block_tables, token_seq,
                            positions, scale, softcap, _none(r1, q),
                            _none(r2, q), window, keep_first,
                            _none(sinks, q), chunk, _none(sigmoid_bias, q),
                            _none(gate, q), _none(dist_bias, q), temp_coef,
                            temp_every)
        return out
    return torch_ref.window_attention(q, k_cache, v_cache, block_tables,
                                      token_seq, positions, scale, softcap,
                                      r1, r2, window, keep_first, sinks,
                                      chunk, sigmoid_bias, gate, dist_bias,
                                      temp_coef, temp_every)


def query_tiles(chunk_lens, starts=None):
    """64-row query tiles of a step's chunks, as numpy arrays (chunk of a
    tile, its first row). Tiles with the most keys ahead of them (`starts`:
    the chunks' first positions) come first, so that a causal launch does
    not end on its longest workgroups."""
    lens = np.asarray(chunk_lens, dtype=np.int64)
    n = -(-lens // QTILE)
    seq = np.repeat(np.arange(len(lens)), n)
    base = (np.arange(int(n.sum())) - np.repeat(np.cumsum(n) - n, n)) * QTILE
    ahead = base if starts is None else base + np.asarray(starts)[seq]
    order = np.argsort(-ahead, kind="stable")
    return seq[order].astype(np.int32), base[order].astype(np.int32)


def build_query_tiles(chunk_lens, device, starts=None):
    """query_tiles as int32 tensors (tile_seq, tile_qbase)."""
    return tuple(torch.from_numpy(t).to(device)
                 for t in query_tiles(chunk_lens, starts))


def embed_positions(ids, positions, table, where, scale: float):
    """table[ids] * scale + where[positions] in f32, and its rounding to bf16, in
    one launch; None for other tables or rows than plain ones of bf16."""
    if not (table.is_cuda and table.dim() == where.dim() == 2
            and ids.dim() == positions.dim() == 1
            and table.size(1) == where.size(1) and table.size(1) % 8 == 0
            and ids.numel() == positions.numel() and not _transformed()
            and _here(table)
            and all(t.is_contiguous() and t.device == table.device
                    for t in (ids, positions, table, where))
            and ids.dtype == positions.dtype == torch.int64
            and all(t.dtype == torch.bfloat16 and t.data_ptr() % 16 == 0
                    and not (torch.is_grad_enabled() and t.requires_grad)
                    for t in (table, where))):
        return None
    x32 = torch.empty(ids.numel(), table.size(1), dtype=torch.float32,
                      device=table.device)
    out = torch.empty_like(x32, dtype=torch.bfloat16)
    _K.embed_positions(x32, out, ids, positions, table, where, scale)
    return x32, out


def post_norm_residual(x32, y, w, eps: float, out_dtype, y2=None, w_y=None,
                       w_y2=None):
    """x32 [T, H] f32 += rms(m) * w in place, m = y or, with y2,
    (rms(y)*w_y + rms(y2)*w_y2)/2. Returns x32 rounded to out_dtype."""
    if x32.is_cuda:
        if out_dtype == torch.float32:
            xo = x32
        else:
            xo = torch.empty(x32.shape, dtype=out_dtype, device=x32.device)
        _K.post_norm_residual(x32, xo, y, w, eps, _none(y2, y),
                              _none(w_y, y), _none(w_y2, y))
        return xo
    return torch_ref.post_norm_residual(x32, y, w, eps, out_dtype, y2, w_y,
                                        w_y2)


def rms_norm_cast(x, weight, eps: float, out_dtype):
    """RMS norm of f32 or bf16 rows (row stride free) with an f32 weight
    → out_dtype."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _K.rms_norm_cast(out, x, weight, eps)
        return out
    return torch_ref.rms_norm_cast(x, weight, eps, out_dtype)


def mlstm_scan(q, k, v, ogate, ipre, fpre, norm_w, state_c, state_n, state_m,
               cu_seqlens, state_slots, seq_starts, cap: float,
               q_scale: float, norm_eps: float, denom_floor: float = 1e-6):
    """Matrix-memory (mLSTM) recurrence with fused gate activations,
    normaliser, per-head RMS norm and sigmoid output gate. q/k [T, H, D],
    v/ogate [T, H, V] (row strides free), ipre/fpre [T, H] f32; states
    C [slots, H, D, V], n [slots, H, D], m [slots, H] f32 in place.
    Returns [T, H*V]."""
    if v.is_cuda:
        T, H, V = v.shape
        out = torch.empty(T, H * V, dtype=v.dtype, device=v.device)
        _K.mlstm_scan(out, q, k, v, ogate, ipre, fpre, norm_w, state_c,
                      state_n, state_m, cu_seqlens, state_slots, seq_starts,
                      cap, q_scale, norm_eps, denom_floor)
        return out
    return torch_ref.mlstm_scan(q, k, v, ogate, ipre, fpre, norm_w, state_c,
                                state_n, state_m, cu_seqlens, state_slots,
                                seq_starts, cap, q_scale, norm_eps,
                                denom_floor)


def ssd_scan(x, B, C, dt, z, a_log, dt_bias, d_skip, norm_w, state,
             cu_seqlens, state_slots, seq_starts, norm_groups: int,
             norm_eps: float):
    """Scalar-decay selective state space with fused step-size
    activation, skip term, silu(z) gate and grouped RMS norm. x
    [T, H, P], B/C [T, G, N], z [T, H*P] (row strides free), dt [T, H]
    f32; state [slots, H, N, P] f32 in place. Returns [T, H*P]."""
    if x.is_cuda:
        T, H, P = x.shape
        out = torch.empty(T, H * P, dtype=x.dtype, device=x.device)
        _K.ssd_scan(out, x, B, C, dt, z, a_log, dt_bias, d_skip, norm_w,
                    state, cu_seqlens, state_slots, seq_starts, norm_groups,
                    norm_eps)
        return out
    return torch_ref.ssd_scan(x, B, C, dt, z, a_log, dt_bias, d_skip, norm_w,
                              state, cu_seqlens, state_slots, seq_starts,
                              norm_groups, norm_eps)


def residual_add_norm(x32, y, w, eps: float, out_dtype, y2=None,
                      s1: float = 1.0, s2: float = 1.0):
    """Pre-norm residual step on an f32 stream [T, H]: x32 += s1*y
    (+ s2*y2) in place; returns rms(x32)*w rounded to out_dtype, the next
    sub-layer's input (None when w is None)."""
    if x32.is_cuda:
        h = torch.empty(x32.shape, dtype=out_dtype, device=x32.device) \
            if w is not None else x32
        _K.residual_add_norm(x32, h, y, _none(y2, y), _none(w, y), s1, s2,
                             eps)
        return h if w is not None else None
    return torch_ref.residual_add_norm(x32, y, w, eps, out_dtype, y2, s1, s2)


def clamped_glu(gu, limit: float, alpha: float = 1.702):
    """[gate | up] rows [T, 2F] -> g*sigmoid(alpha*g)*(u + 1) [T, F] with
    g = min(gate, limit), u = clamp(up, -limit, limit)."""
    if gu.is_cuda:
        out = torch.empty(gu.size(0), gu.size(1) // 2, dtype=gu.dtype,
                          device=gu.device)
        _K.clamped_glu(out, gu, limit, alpha)
        return out
    return torch_ref.clamped_glu(gu, limit, alpha)


def sigmoid_mul(x, gate):
    """x [T, N] * sigmoid(gate [T, Ng]) (gate's row stride free); with
    Ng < N each gate column serves N/Ng consecutive columns of x (one
    gate per head)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _K.sigmoid_mul(out, x, gate)
        return out
    return torch_ref.sigmoid_mul(x, gate)


def gelu_glu(gu):
    """[gate | up] rows [T, 2F] -> gelu_tanh(gate) * up [T, F]."""
    if gu.is_cuda:
        out = torch.empty(gu.size(0), gu.size(1) // 2, dtype=gu.dtype,
                          device=gu.device)
        _K.gelu_glu(out, gu)
        return out
    return torch_ref.gelu_glu(gu)


def relu_glu(gu):
    """[gate | up] rows [T, 2F] -> relu(gate) * up [T, F]."""
    if gu.is_cuda:
        out = torch.empty(gu.size(0), gu.size(1) // 2, dtype=gu.dtype,
                          device=gu.device)
        _K.relu_glu(out, gu)
        return out
    return torch_ref.relu_glu(gu)


def relu2(x):
    """relu(x)^2, element-wise, rows [T, N] (row stride free)."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _K.relu2(out, x)
        return out
    return torch_ref.relu2(x)


# ---- latent attention (kernel group "latent") -----------------------------

def bigram_embed(ids, embed, scale: float, table, buckets: int,
                 mul_prev: int, mul_cur: int, prev_state, cu_seqlens,
                 state_slots, seq_starts, token_seq):
    """f32 rows embed[ids]*scale (+ the hashed bigram row: (previous *
    mul_prev + token * mul_cur) mod buckets, row `buckets` for a
    sequence's first token). The token before a chunk's first row comes
    from prev_state [slots] int64, which is advanced to the chunk's last
    token. table None: token embedding only."""
    if ids.is_cuda:
        out = torch.empty(ids.size(0), embed.size(1), dtype=torch.float32,
                          device=ids.device)
        none = torch.empty(0, dtype=embed.dtype, device=ids.device)
        _K.bigram_embed(out, ids, embed, scale,
                        table if table is not None else none, buckets,
                        mul_prev, mul_cur,
                        prev_state if table is not None else
                        torch.empty(0, dtype=torch.long, device=ids.device),
                        cu_seqlens, state_slots, seq_starts, token_seq)
        return out
    return torch_ref.bigram_embed(ids, embed, scale, table, buckets,
                                  mul_prev, mul_cur, prev_state, cu_seqlens,
                                  state_slots, seq_starts)


def latent_rope_cache_write(q, dkv, norm_w, eps: float, cache, slot_mapping,
                            positions, inv_freq, dim: int, pad_to: int = 0,
                            interleaved: bool = False, rot_mag: float = 1.0):
    """Rotation of the last 2R dims of every head of q [T, H, dim + 2R]
    (R = len(inv_freq); i paired with i + R, or with `interleaved` 2i
    with 2i + 1; angle = position * inv_freq[i] in f32; cos and sin times
    rot_mag) and, with dkv [T, rank + 2R] given (row stride
    free), the latent row: RMS norm of the first rank dims with the f32
    weight norm_w, rotation of the last 2R, scatter into the paged latent
    cache [blocks, block_size, rank + 2R] at slot_mapping (negative slots
    skipped). Returns q rotated, contiguous; with pad_to, every head is
    zero-padded to that many dims."""
    if q.is_cuda:
        out = torch.empty(q.size(0), q.size(1), max(pad_to, q.size(2)),
                          dtype=q.dtype, device=q.device)
        own = dkv is not None
        _K.latent_rope_cache_write(
            out, q, dkv if own else torch.empty(0, 0, dtype=q.dtype,
                                                device=q.device),
            norm_w if own else _none(None, q), eps,
            cache if own else torch.empty(0, dtype=q.dtype, device=q.device),
            slot_mapping, positions, inv_freq, dim, interleaved, rot_mag)
        return out
    out = torch_ref.latent_rope_cache_write(q, dkv, norm_w, eps, cache,
                                            slot_mapping, positions,
                                            inv_freq, dim, interleaved,
                                            rot_mag)
    if pad_to > out.size(2):
        out = torch.nn.functional.pad(out, (0, pad_to - out.size(2)))
    return out


def latent_attention(q, cache, block_tables, token_seq, positions,
                     scale: float, rank: int, sinks=None, window: int = 0):
    """Causal attention of latent-space queries [T, H, rank + P] over the
    paged latent cache [blocks, block_size, rank + P]: score = q . row *
    scale over rows 0..position of the row's sequence (with window > 0 the
    last `window` of them), optional per-head
    sinks in the denominator, output = weighted sum of the rows' first
    `rank` dims, [T, H, rank]. One pass over the cache serves all heads."""
    if q.is_cuda:
        out = torch.empty(q.size(0), q.size(1), rank, dtype=q.dtype,
                          device=q.device)
        _K.latent_attention(out, q, cache, block_tables, token_seq,
                            positions, scale, _none(sinks, q), window)
        return out
    return torch_ref.latent_attention(q, cache, block_tables, token_seq,
                                      positions, scale, rank, sinks, window)


def latent_gather(cache, block_tables, ctx_lens, first_keys=None):
    """Whole pages of the step's sequences out of the paged latent cache:
    chunk b's first ceil(ctx_lens[b] / block_size) pages, in block-table
    order, without those that end before position first_keys[b] (a host
    list; their table entries name some gathered page, whose rows the mask
    must hide). Returns (rows [pages * block_size, row], scratch block tables
    [B, max pages] int32 numbering the gathered pages consecutively).
    ctx_lens is a host list, so the shapes are known without a device
    read; rows past a sequence's length are whatever the page holds and
    stay behind the causal mask."""
    bs, mb = cache.size(1), block_tables.size(1)
    counts = [-(-int(n) // bs) for n in ctx_lens]
    idx, tables, base = [], [], 0
    width = max(max(counts), 1)
    for b, n in enumerate(counts):
        skip = min(int(first_keys[b]) // bs, n) if first_keys else 0
        idx.extend(range(b * mb + skip, b * mb + n))
        tables.append([0] * skip + list(range(base, base + n - skip))
                      + [0] * (width - n))
        base += n - skip
    dev = cache.device
    pages = block_tables.reshape(-1)[
        torch.tensor(idx, dtype=torch.long, device=dev)].long()
    rows = cache[pages].reshape(-1, cache.size(2))
    return rows, torch.tensor(tables, dtype=torch.int32, device=dev)


def latent_expand(kn, vv, lat, H: int, D: int, V: int, rank: int, Dp: int,
                  Vp: int, block_size: int):
    """Step-local paged K/V scratch from gathered latent rows (GPU): kn
    [N, H*D] and vv [N, H*V] are the up-projected unrotated keys and
    values of rows lat [N, rank + P]; head h's key is [kn_h | lat's last P
    dims | zeros] of width Dp, its value [vv_h | zeros] of width Vp.
    Returns k [N / block_size, H, block_size, Dp], v [..., Vp]."""
    pages = lat.size(0) // block_size
    k_s = torch.empty(pages, H, block_size, Dp, dtype=lat.dtype,
                      device=lat.device)
    v_s = torch.empty(pages, H, block_size, Vp, dtype=lat.dtype,
                      device=lat.device)
    _K.latent_expand(k_s, v_s, kn, vv, lat, H, D, V, rank)
    return k_s, v_s


# ---- looped parallel-layer stacks (groups "mix" and "diag") -----------------

def linear_f32(x, weight, bias=None):
    """x [T, K] @ weight [N, K]^T (+ bias) with the result kept in f32.
    Inputs in the activation dtype are multiplied exactly and summed in
    f32, and the result is not rounded back to the activation dtype: what
    feeds a recurrence's gates. On the GPU this is the vendor bf16 GEMM
    with an f32 output; where the build lacks that, an f32 GEMM."""
    global _MM_F32_OUT
    if x.dtype != torch.float32 and x.is_cuda and _MM_F32_OUT:
        try:
            out = torch.mm(x, weight.t(), out_dtype=torch.float32)
            return out if bias is None else out + bias
        except (RuntimeError, TypeError):
            _MM_F32_OUT = False
    return torch.nn.functional.linear(x.float(), weight.float(), bias)


_MM_F32_OUT = True


def scaled_residual_add_norm(x32, terms, w, eps: float, out_dtype,
                             x_add=None):
    """Residual step with per-channel sub-layer scales on an f32 stream
    [T, H]: x32 += sum of v*y over `terms`, one to three pairs (y [T, H]
    in the activation dtype, v [H] f32), (+ x_add [T, H] f32), in place;
    returns rms(x32)*w rounded to out_dtype, the next layer's input (None
    when w is None)."""
    assert 1 <= len(terms) <= 3
    if x32.is_cuda:
        h = torch.empty(x32.shape, dtype=out_dtype, device=x32.device) \
            if w is not None else x32
        y0 = terms[0][0]
        ys = [t[0] for t in terms] + [_none(None, y0)] * (3 - len(terms))
        vs = [t[1] for t in terms] + [_none(None, y0)] * (3 - len(terms))
        _K.scaled_residual_add_norm(x32, h, ys[0], ys[1], ys[2], vs[0],
                                    vs[1], vs[2], _none(x_add, y0),
                                    _none(w, y0), eps)
        return h if w is not None else None
    return torch_ref.scaled_residual_add_norm(x32, terms, w, eps, out_dtype,
                                              x_add)


def token_shift(h, mu, state, cu_seqlens, state_slots, seq_starts,
                token_seq):
    """Blend of every row with the row before it: h_t + (h_{t-1} - h_t)*mu
    (mu [H] f32). A chunk's first row takes its predecessor from state
    [slots, H] (h's dtype; zeros at position 0), which is advanced to the
    chunk's last row. Returns [T, H]."""
    if h.is_cuda:
        out = torch.empty(h.shape, dtype=h.dtype, device=h.device)
        _K.token_shift(out, h, mu, state, cu_seqlens, state_slots,
                       seq_starts, token_seq)
        return out
    return torch_ref.token_shift(h, mu, state, cu_seqlens, state_slots,
                                 seq_starts)


def diag_delta_rule(r, k, v, w_pre, a_pre, gate, norm_w, state, cu_seqlens,
                    state_slots, seq_starts, decay_rate: float, k_eps: float,
                    norm_eps: float, a_bias=None):
    """Generalized delta rule with a decay per key channel: r/k/v/gate
    [T, H, D] (row strides free), w_pre/a_pre [T, H*D] f32 (decay and
    removal-rate pre-activations), norm_w [H*D] f32, state [slots, H, D, D]
    f32 in place. S <- diag(w) S - (a*u)(u^T S) + k v^T with u the unit
    key, w = exp(-decay_rate*sigmoid(w_pre)), a = sigmoid(a_pre + a_bias)
    (a_bias [H*D] f32, optional); read-out S^T r divided by its RMS per
    head, times norm_w, times sigmoid(gate). Returns [T, H*D]."""
    if r.is_cuda:
        T, H, D = r.shape
        out = torch.empty(T, H * D, dtype=r.dtype, device=r.device)
        _K.diag_delta_rule(out, r, k, v, w_pre, a_pre, _none(a_bias, r), gate,
                           norm_w, state, cu_seqlens, state_slots, seq_starts,
                           decay_rate, k_eps, norm_eps)
        return out
    if a_bias is not None:
        a_pre = a_pre + a_bias
    return torch_ref.diag_delta_rule(r, k, v, w_pre, a_pre, gate, norm_w,
                                     state, cu_seqlens, state_slots,
                                     seq_starts, decay_rate, k_eps, norm_eps)


def hgrn2_scan(q, v, f_pre, lower, norm_w, state, cu_seqlens, state_slots,
               seq_starts, norm_eps: float, f_bias=None):
    """Linear attention with a lower-bounded forget gate that also sets
    the write: q [T, H, D] (silu applied inside), v [T, H, V] (row strides
    free), f_pre [T, H*D] f32, lower [H*D] f32, norm_w [V] f32, state
    [slots, H, D, V] f32 in place. f = lower + (1 - lower) sigmoid(f_pre +
    f_bias) (f_bias [H*D] f32, optional), S <- diag(f) S + (1 - f) v^T, o = S^T silu(q), RMS-normed over V with
    norm_w. Returns [T, H*V]."""
    if q.is_cuda:
        T, H, V = v.shape
        out = torch.empty(T, H * V, dtype=q.dtype, device=q.device)
        _K.hgrn2_scan(out, q, v, f_pre, _none(f_bias, q), lower, norm_w,
                      state, cu_seqlens, state_slots, seq_starts, norm_eps)
        return out
    if f_bias is not None:
        f_pre = f_pre + f_bias
    return torch_ref.hgrn2_scan(q, v, f_pre, lower, norm_w, state,
                                cu_seqlens, state_slots, seq_starts,
                                norm_eps)


# ---- hyper-connected residual streams (kernel group "streams") -------------

def stream_embed(ids, table, g, w_in, w, eps: float):
    """Opens a stack of S residual streams (S = len(w_in)): RMS-normed table
    rows times g as S equal f32 copies [T, S, H], and the first sub-layer's
    input rms(sum_s w_in[s] x_s)*w in the table's dtype. g and w are f32,
    one number or one per coordinate. Returns (x, h)."""
    if ids.is_cuda:
        T, H = ids.numel(), table.size(1)
        x = torch.empty(T, w_in.numel(), H, dtype=torch.float32,
                        device=ids.device)
        h = torch.empty(T, H, dtype=table.dtype, device=ids.device)
        _K.stream_embed(x, h, ids, table, g, w_in, w, eps)
        return x, h
    return torch_ref.stream_embed(ids, table, g, w_in, w, eps)


def stream_mix_norm(x, y, mix, w_out, w_in, w, eps: float, out_dtype,
                    write_x: bool = True):
    """A sub-layer's write and the next one's read on residual streams x
    [T, S, H] f32: x_t <- sum_s mix[s, t] x_s + w_out[t]*y for all t from
    the old streams, in place; u = sum_s w_in[s] x_s of the new ones.
    Returns rms(u)*w in out_dtype, or u itself with w None (then
    write_x=False leaves the streams unstored). y [T, H] may be the
    activation dtype or f32; w is one number or one per coordinate."""
    if x.is_cuda:
        h = torch.empty(x.size(0), x.size(2), dtype=out_dtype,
                        device=x.device)
        _K.stream_mix_norm(x, h, y, mix, w_out, w_in, _none(w, x), eps,
                           write_x)
        return h
    return torch_ref.stream_mix_norm(x, y, mix, w_out, w_in, w, eps,
                                     out_dtype, write_x)


# ---- sandwich-normed stacks (kernel groups "lnorm", "diag" and "mix") --------

def layer_norm_cast(x, w, b, eps: float, out_dtype):
    """Layer norm of f32 or bf16 rows [T, H] with f32 weight and bias →
    out_dtype."""
    if x.is_cuda:
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _K.layer_norm_cast(out, x, w, b, eps)
        return out
    return torch_ref.layer_norm_cast(x, w, b, eps, out_dtype)


def embed_layer_norm(ids, table, scale: float, w, b, eps: float):
    """Opens a residual stream: x = table[ids]*scale in f32 and its layer
    norm in the table's dtype. Returns (x [T, H] f32, h [T, H])."""
    if ids.is_cuda:
        shape = (ids.numel(), table.size(1))
        x = torch.empty(shape, dtype=torch.float32, device=ids.device)
        h = torch.empty(shape, dtype=table.dtype, device=ids.device)
        _K.embed_layer_norm(x, h, ids, table, scale, w, b, eps)
        return x, h
    return torch_ref.embed_layer_norm(ids, table, scale, w, b, eps)


def sandwich_norm_residual(x32, y, w, b, w_next, b_next, eps: float,
                           out_dtype, y2=None):
    """Residual step with a layer norm on both sides of a sub-layer, on an
    f32 stream [T, H]: x32 += ln(y + y2)*w + b in place; returns the next
    sub-layer's input ln(x32)*w_next + b_next in out_dtype (None when
    w_next is None). y and y2 (optional) are f32 or bf16, each its own;
    weights and biases f32."""
    if x32.is_cuda:
        h = torch.empty(x32.shape, dtype=out_dtype, device=x32.device) \
            if w_next is not None else x32
        _K.sandwich_norm_residual(x32, h, y, _none(y2, y), w, b,
                                  _none(w_next, y), _none(b_next, y), eps)
        return h if w_next is not None else None
    return torch_ref.sandwich_norm_residual(x32, y, w, b, w_next, b_next,
                                            eps, out_dtype, y2)


def gla_scan(q, k, v, gate, low, a2, a_bias, tau: float, q_scale: float,
             norm_w, state, cu_seqlens, state_slots, seq_starts,
             norm_eps: float):
    """Gated linear attention with a decay per key channel: q/k [T, H, D],
    v/gate [T, H, V] (row strides free), low [T, R] f32 (row stride free),
    a2 [R, H*D] and a_bias [H*D] f32, norm_w [V] f32, state [slots, H, D, V]
    f32 in place. alpha = sigmoid(low @ a2 + a_bias)^(1/tau), S <-
    diag(alpha) S + k v^T, o = S^T q * q_scale, RMS-normed over V with
    norm_w, times silu(gate). Returns [T, H*V]."""
    if q.is_cuda:
        T, H, V = v.shape
        out = torch.empty(T, H * V, dtype=q.dtype, device=q.device)
        _K.gla_scan(out, q, k, v, gate, low, a2, a_bias, tau, q_scale, norm_w,
                    state, cu_seqlens, state_slots, seq_starts, norm_eps)
        return out
    return torch_ref.gla_scan(q, k, v, gate, low, a2, a_bias, tau, q_scale,
                              norm_w, state, cu_seqlens, state_slots,
                              seq_starts, norm_eps)


def scaled_softcap(x, scale: float, cap: float):
    """x f32, in place: cap*tanh(x*scale/cap) (cap <= 0: x*scale)."""
    if x.is_cuda:
        _K.scaled_softcap(x, scale, cap)
        return x
    return torch_ref.scaled_softcap(x, scale, cap)
