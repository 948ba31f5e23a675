"""Modules that a caller watches or replaces are called as modules: hooks run, get
tensors and may change them, whatever the layer would otherwise do in fewer
launches."""
import dataclasses

import pytest
import torch

from kaito_amd import ops
from kaito_amd.engine import EngineConfig, LLMEngine, SamplingParams
from kaito_amd.models import get_model_config
from kaito_amd.parallel.state import init_parallel

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _engine(device, name, **changes):
    init_parallel(1)
    mc = dataclasses.replace(get_model_config(name), **changes)
    if device == "cpu":
        mc = dataclasses.replace(mc, dtype=torch.float32)
    torch.manual_seed(7)
    return LLMEngine(EngineConfig(
        model=mc, device=device, max_num_seqs=4, max_model_len=256,
        num_gpu_blocks=64, enforce_eager=True))


def _generate(eng):
    out = eng.generate([list(range(3, 25))],
                       SamplingParams(max_tokens=4, temperature=0.0,
                                      ignore_eos=True))
    return out[0].output_token_ids


def _watch(modules):
    """Forward hooks on modules; the calls of each, of its tensors' types."""
    calls = {m: [] for m in modules}

    def seen(m, args, out):
        first = out[0] if isinstance(out, tuple) else out
        calls[m].append((type(args[0]), type(first)))
    handles = [m.register_forward_hook(seen) for m in modules]
    return calls, handles


def _check_watched(eng, modules):
    calls, handles = _watch(modules)
    _generate(eng)
    for h in handles:
        h.remove()
    for m, c in calls.items():
        # a prompt step, then one for each of the other three tokens
        assert len(c) == 4, (type(m).__name__, c)
        assert all(issubclass(t, torch.Tensor) for pair in c for t in pair), c


@pytest.mark.parametrize("device", DEVICES)
def test_mixers_of_a_hybrid_layer(device):
    eng = _engine(device, "tiny-gurapel-test")
    layers = [l for l in eng.runner.model.layers if l.spec.kind == "parallel"]
    assert layers
    _check_watched(eng, [m for l in layers for m in (l.attn, l.rglru)])


@pytest.mark.parametrize("of", ["module", "class"])
@pytest.mark.parametrize("device", DEVICES)
def test_replaced_forward_of_a_mixer(device, of, monkeypatch):
    """What wraps a module by giving it, or all of its class, a forward of its own
    is not passed by."""
    eng = _engine(device, "tiny-gurapel-test")
    layer = next(l for l in eng.runner.model.layers
                 if l.spec.kind == "parallel")
    where = layer.rglru if of == "module" else type(layer.rglru)
    plain, calls = where.forward, []

    def forward(*args):
        if of == "module" or args[0] is layer.rglru:
            calls.append(args[-4].size(0))
        return plain(*args)
    monkeypatch.setattr(where, "forward", forward)
    _generate(eng)
    assert calls == [22, 1, 1, 1]


@pytest.mark.parametrize("name,part", [
    ("LlamaAttention", "self_attn"), ("LlamaMLP", "mlp"),
    ("RowParallelLinear", "mlp.down_proj")])
def test_replaced_forward_of_a_class(name, part, monkeypatch):
    """Nor in a decoder layer, and it is called as it was: without `defer`."""
    eng = _engine("cpu", "tiny-llama-test")
    want = _generate(eng)
    monkeypatch.setattr(ops, "linear_parts", _in_parts)
    mine = [l.get_submodule(part) for l in eng.runner.model.layers]
    cls, calls = type(mine[0]), []
    assert cls.__name__ == name
    plain = cls.forward

    def forward(self, *args):
        if self in mine:
            calls.append(self)
        out = plain(self, *args)
        assert isinstance(out, torch.Tensor)
        return out
    monkeypatch.setattr(cls, "forward", forward)
    assert _generate(eng) == want
    assert len(calls) == 4 * len(mine)


@pytest.mark.parametrize("device", DEVICES)
def test_query_projection_of_latent_attention(device):
    eng = _engine(device, "tiny-deepseek-test", q_lora_rank=0)
    _check_watched(eng, [l.self_attn.q_proj for l in eng.runner.model.layers])


@pytest.mark.parametrize("device", DEVICES)
def test_gate_projection(device):
    eng = _engine(device, "tiny-llama-test")
    _check_watched(eng, [l.mlp.gate_up_proj for l in eng.runner.model.layers])


@pytest.mark.gpu
def test_packed_gate_projection():
    eng = _engine("cuda", "tiny-llama-test", hidden_size=1024,
                  intermediate_size=1024)
    for l in eng.runner.model.layers:
        l.mlp.gate_up_proj.quantize_(128)
    _check_watched(eng, [l.mlp.gate_up_proj for l in eng.runner.model.layers])


def _in_parts(x, w):
    """Every product as if the split kernel had made it."""
    y = x.float() @ w.float().t()
    return ops.SplitRows(torch.stack([y * 0.75, y * 0.25]))


@pytest.mark.parametrize("which", [
    lambda ls: [ls[0]], lambda ls: [ls[1]], lambda ls: [ls[0].self_attn],
    lambda ls: [ls[0].mlp], lambda ls: [m for l in ls for m in (
        l, l.self_attn, l.mlp, l.self_attn.o_proj, l.mlp.down_proj)]],
    ids=["first", "second", "attention", "mlp", "all"])
def test_decoder_layers_with_products_in_parts(monkeypatch, which):
    eng = _engine("cpu", "tiny-llama-test")
    want = _generate(eng)
    monkeypatch.setattr(ops, "linear_parts", _in_parts)
    assert _generate(eng) == want
    _check_watched(eng, which(eng.runner.model.layers))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["tiny-moe-test", "tiny-gurapel-test",
                                  "tiny-deepseek-test", "tiny-llama-test"])
@pytest.mark.parametrize("which", ["first", "last", "mlp", "all"])
def test_layers_on_the_gpu(name, which):
    eng = _engine("cuda", name)
    ls = eng.runner.model.layers
    _check_watched(eng, {
        "first": [ls[0]], "last": [ls[-1]], "mlp": [l.mlp for l in ls],
        "all": [m for l in ls for m in (l, l.mlp)]}[which])
