"""Decoder layers of the llama kind at sizes where a step's norms go into the products
beside them (1 and 2 rows ahead of the product, split products ahead of the norm),
against the same layers with a launch for each: the same bits of the hidden rows and
of the residual stream, whatever of a layer has a bias, packed weights, an adapter or
a hook. And a layer of experts with one of every token."""
import dataclasses

import pytest
import torch

from kaito_amd import ops
from kaito_amd.engine import lora
from kaito_amd.models import get_model_config
from kaito_amd.models.llama import AttnMetadata, LlamaForCausalLM
from kaito_amd.models.moe import MoEMLP
from kaito_amd.parallel.state import init_parallel

DEV = "cuda"
H, INTER, KEYS = 4096, 10240, 40


def _model(bias=False, packed=False):
    init_parallel(1)
    cfg = dataclasses.replace(
        get_model_config("tiny-llama-test"), hidden_size=H, num_layers=3,
        num_heads=32, num_kv_heads=8, head_dim=128, intermediate_size=INTER,
        attention_bias=bias)
    with torch.device(DEV):
        m = LlamaForCausalLM(cfg).eval()
    g = torch.Generator(device=DEV).manual_seed(5)
    for name, p in m.named_parameters():
        v = torch.randn(p.shape, device=DEV, generator=g)
        if name.endswith("norm") or name.endswith("layernorm"):
            v = 1 + 0.3 * v
        elif p.dim() == 2 and "embed" not in name:
            v = v * p.size(1) ** -0.5
        p.data.copy_(v)
    m.init_rope(torch.device(DEV))
    if packed:
        for layer in m.layers:
            for p in (layer.self_attn.qkv_proj, layer.self_attn.o_proj,
                      layer.mlp.gate_up_proj, layer.mlp.down_proj):
                p.quantize_(128)
    return m


def _step(m, T):
    """Hidden rows of a step of T sequences with KEYS keys each, and the rows
    and residual stream that go into the last norm."""
    cfg = m.cfg
    g = torch.Generator(device=DEV).manual_seed(T)
    pages = (KEYS + 15) // 16
    bt = torch.arange(T * pages, dtype=torch.int32, device=DEV).view(T, pages)
    caches = [tuple(torch.randn(T * pages, cfg.num_kv_heads, 16, cfg.head_dim,
                                device=DEV, generator=g).bfloat16()
                    for _ in "kv") for _ in m.layers]
    last = torch.full((T,), KEYS - 1, device=DEV)
    meta = AttnMetadata(
        is_prefill=False, block_tables=bt,
        slot_mapping=bt[:, -1].long() * 16 + (KEYS - 1) % 16,
        seq_lens=torch.full((T,), KEYS, dtype=torch.int32, device=DEV))
    ids = torch.randint(0, cfg.vocab_size, (T,), device=DEV, generator=g)
    with torch.inference_mode():
        return m(ids, last, caches, meta), caches


def _alone(mp):
    """A launch for each norm, product and sum."""
    mp.setattr(ops, "norm_fits", lambda *a: False)
    mp.setattr(ops, "w4a16_norm_linear", lambda *a: None)
    mp.setattr(ops, "linear_parts", ops.linear)


def _compare(m, T, fused, rel=0.0):
    """fused: norms in products and split products ahead of norms. rel: how far
    the two may be apart, the same bits else."""
    def close(a, b):
        if not rel:
            return torch.equal(a, b)
        return (a.double() - b.double()).norm() <= rel * b.double().norm()
    with pytest.MonkeyPatch.context() as mp:
        _alone(mp)
        want, theirs = _step(m, T)
    took = []

    def count(name, yes):
        f = getattr(ops, name)

        def call(*args, **kw):
            out = f(*args, **kw)
            if yes(out):
                took.append(name)
            return out
        mp.setattr(ops, name, call)
    with pytest.MonkeyPatch.context() as mp:
        count("add_norm_linear", lambda o: True)
        count("w4a16_norm_linear", lambda o: o is not None)
        count("linear_parts", lambda o: isinstance(o, ops.SplitRows))
        got, ours = _step(m, T)
    assert len(took) == fused, took
    assert torch.isfinite(got).all() and got.float().std() > 0.1
    assert close(got, want), (got.double() - want.double()).norm() / want.norm()
    # keys of every layer: of the hidden rows that went into it
    for a, b in zip(ours, theirs):
        assert close(a[0], b[0]) and close(a[1], b[1])


# norms in products: an MLP's in each of three layers, the input's in two; split
# products: down of each layer (10240 inputs), o of each from 17 rows on
STEPS = [(1, 5), (2, 5), (3, 0), (9, 3), (16, 3), (17, 6), (64, 6), (250, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize("T,fused", STEPS)
@pytest.mark.parametrize("bias", [False, True])
def test_steps(T, fused, bias):
    m = _model(bias)
    if bias:
        assert m.layers[0].self_attn.qkv_proj.bias is not None
    _compare(m, T, fused)


@pytest.mark.gpu
@pytest.mark.parametrize("T,fused", [(1, 3), (2, 5), (3, 0), (17, 0)])
@pytest.mark.parametrize("bias", [False, True])
def test_packed_weights(T, fused, bias):
    """1 and 2 rows: the MLPs' norms, of 2 the input's of two layers too. Alone, one
    row's gate and up are streamed and rounded to 8 bits before their product, two
    rows' qkv summed in another order: up to four roundings of 2^-9 of a layer's
    rows that the other side has not, 2^-7, of three layers that do not depend on
    one another 2^-6 at most as a norm. A norm, sum or bias left out is some 1."""
    _compare(_model(bias, packed=True), T, fused, 2.0 ** -6 if T <= 2 else 0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 17])
def test_adapters(T, monkeypatch):
    monkeypatch.setattr(lora, "is_active", lambda: True)
    monkeypatch.setattr(lora, "maybe_apply", lambda m, x, out: out * 1.25)
    _compare(_model(), T, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("T,where,fused", [
    (1, "self_attn", 4), (2, "mlp", 4), (1, "self_attn.qkv_proj", 4),
    (2, "mlp.gate_up_proj", 4), (17, "self_attn", 5), (17, "mlp", 5),
    (17, "self_attn.o_proj", 5), (17, "mlp.down_proj", 5), (17, "", 2),
    (1, "", 5)])
def test_hooks(T, where, fused):
    """A hook on the second layer or a part of it, which doubles its rows."""
    m = _model()
    layer = m.layers[1]

    def double(mod, args, out):
        if isinstance(out, tuple):
            return (out[0] * 2,) + out[1:]
        return out * 2
    (layer.get_submodule(where) if where else layer).register_forward_hook(
        double)
    _compare(m, T, fused)


@pytest.mark.gpu
@pytest.mark.parametrize("T,beside", [(1, True), (4, True), (17, True),
                                      (32, True), (33, False), (64, False)])
def test_shared_expert_of_a_layer(T, beside, monkeypatch):
    """The routed experts' weighted sum and the shared expert, as rows and behind
    the norm, against 64 bits. The shared result and the sum round to bf16, by
    2^-9 of their values at most. So do gates, ups and their products: an error
    of up to 2^-9 of each term of the 512, three times, is 2^-9 of the row's root
    mean square as a standard deviation at most, and below 2^-6 in eight."""
    init_parallel(1)
    cfg = dataclasses.replace(
        get_model_config("tiny-moe-test"), hidden_size=1024, num_experts=8,
        num_experts_per_tok=2, moe_intermediate_size=512, n_shared_experts=1)
    with torch.device(DEV):
        m = MoEMLP(cfg)
    g = torch.Generator(device=DEV).manual_seed(T)
    for p in m.parameters():
        p.data.copy_(torch.randn(p.shape, device=DEV, generator=g)
                     * p.size(-1) ** -0.5)
    x, r = (torch.randn(T, 1024, device=DEV, generator=g).bfloat16()
            for _ in "xr")
    w = 1 + torch.randn(1024, device=DEV, generator=g).bfloat16() * 0.2
    joined = []
    up = ops.moe_up_pairs
    monkeypatch.setattr(ops, "moe_up_pairs", lambda *a, **kw: (
        joined.append("all_w" in kw), up(*a, **kw))[1])
    with torch.inference_mode():
        out = m(x)
        topi, topw, _ = m._choose(x)
        normed, _ = ops.fused_add_rms_norm(x, r.clone(), w, 1e-6)
        # the layer behind a norm, whose sum a second norm takes
        rows, stream = m.forward_add_norm(x, r.clone(), w, 1e-6, defer=True)
        last, _ = rows.add_rms_norm(stream.clone(), w, 1e-6)
        again = m(normed)
    assert joined == ([beside] * 3 if joined else [])
    assert bool(joined) or not beside

    def expert(x, gu, down):
        a, b = (x.double() @ gu.double().T).chunk(2, -1)
        return (a * torch.sigmoid(a) * b) @ down.double().T
    shared = expert(x, m.w_shared_gate_up, m.w_shared_down)
    routed = torch.zeros_like(shared)
    for e in range(8):
        share = (topw.double() * (topi == e)).sum(1, keepdim=True)
        routed += share * expert(x, m.w_gate_up[e], m.w_down[e])
    ref = shared + routed
    bound = 2.0 ** -9 * (ref.abs() + shared.abs()) + 2.0 ** -6 * sum(
        v.square().mean(1, keepdim=True).sqrt() for v in (shared, routed))
    err = (out.double() - ref).abs()
    assert (err <= bound).all(), (err / bound).max()
    want, _ = ops.fused_add_rms_norm(again, stream.clone(), w, 1e-6)
    assert torch.equal(last, want)
