"""The MFMA prompt attention (ops/csrc/flash_prefill.h) at the edges of its
tiles: 32-row waves, workgroups of 128 flattened rows, 64- (wide heads 32-)
key tiles, head groups that are flattened and groups that are not. Outputs
are bf16 of values whose weights entered the second product as bf16: two
roundings of 2^-9 each relative to the largest terms."""
import math

import pytest
import torch

from kaito_amd import ops
from kaito_amd.ops import torch_ref as R

DEV = "cuda"
TOL = 2 * 2.0 ** -8          # of the values' magnitude (up to about 3)


def _bf16(*shape):
    return torch.randn(*shape, device=DEV).to(torch.bfloat16)


def _cu(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                        dtype=torch.int32, device=DEV)


def _check(out, ref):
    assert torch.isfinite(out).all()
    assert (out.cpu().float() - ref).abs().max().item() < 3 * TOL


@pytest.mark.gpu
@pytest.mark.parametrize("QH,KH,D,lens,window,sink", [
    (4, 1, 128, [1, 31, 32, 33], 0, False),
    (8, 2, 128, [63, 64, 65, 129], 0, True),
    (3, 3, 128, [127, 128, 129, 193], 0, False),     # one head per group
    (6, 2, 64, [1, 200, 70], 0, False),              # group of 3
    (16, 1, 64, [9, 40, 100], 33, False),
    (8, 1, 96, [64, 65, 130], 0, False),
    (2, 1, 256, [31, 33, 150], 64, True),
    (4, 4, 256, [64, 96, 129], 0, False),
    (8, 2, 128, [300], 1, False),
    (5, 1, 128, [260, 3], 100, True),
])
@pytest.mark.parametrize("scale_sign", [1.0, -1.0])
def test_whole_prompts(QH, KH, D, lens, window, sink, scale_sign):
    torch.manual_seed(len(lens) + D)
    T = sum(lens)
    qkv = _bf16(T, (QH + 2 * KH) * D)        # rows of a fused projection
    q, k, v = qkv.split([QH * D, KH * D, KH * D], -1)
    q, k, v = (t.unflatten(-1, (-1, D)) for t in (q, k, v))
    sinks = torch.randn(QH, device=DEV) if sink else None
    scale = scale_sign / math.sqrt(D)
    out = ops.prefill_attention(q, k, v, _cu(lens), scale, window=window,
                                sinks=sinks)
    ref = R.prefill_attention(
        q.cpu().float(), k.cpu().float(), v.cpu().float(), _cu(lens).cpu(),
        scale, window, sinks.cpu() if sink else None)
    _check(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("QH,KH,D", [(4, 1, 128), (3, 1, 128), (4, 2, 96),
                                     (4, 4, 96), (8, 1, 64), (4, 4, 64),
                                     (4, 2, 256)])
@pytest.mark.parametrize("lens", [[1], [31, 1, 32, 7], [32] * 40, [33, 5],
                                  [64, 40, 63] * 60, [65, 3]])
@pytest.mark.parametrize("window,sink,scale", [(0, False, 1.0), (0, True, 0.1),
                                               (9, False, -0.2)])
def test_short_prompts(QH, KH, D, lens, window, sink, scale):
    """Up to 32 rows, one wave per head, up to 64, two, and one row more; with
    the longest prompt given and without."""
    torch.manual_seed(D + len(lens))
    T, cu = sum(lens), _cu(lens)
    q, k, v = _bf16(T, QH, D), _bf16(T, KH, D), _bf16(T, KH, D)
    sinks = torch.randn(QH, device=DEV) if sink else None
    ref = R.prefill_attention(q.cpu().float(), k.cpu().float(),
                              v.cpu().float(), cu.cpu(), scale, window,
                              sinks.cpu() if sink else None)
    for longest in (max(lens), None):
        _check(ops.prefill_attention(q, k, v, cu, scale, longest, window,
                                     sinks), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("shift,pad", [(1, 0), (0, 4), (3, 5)])
def test_rows_off_16_bytes(shift, pad):
    """Rows and strides that 16 bytes do not divide: those of a copy."""
    torch.manual_seed(shift)
    KH, D, T = 2, 64, 150
    wide = _bf16(T, 2 * KH * D + pad + 8).view(-1)

    def rows(at):
        return wide.as_strided((T, KH, D), (2 * KH * D + pad + 8, D, 1), at)

    q = _bf16(T, 4, D)
    k, v = rows(shift), rows(shift + KH * D)
    out = ops.prefill_attention(q, k, v, _cu([T]), D ** -0.5)
    ref = ops.prefill_attention(q, k.clone(), v.clone(), _cu([T]), D ** -0.5)
    assert torch.equal(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("QH,KH,D,pairs,window", [
    (4, 1, 128, [(64, 64), (65, 1), (191, 33)], 0),
    (8, 8, 128, [(300, 129), (128, 128)], 0),
    (8, 1, 64, [(90, 17), (257, 64)], 50),
    (2, 2, 256, [(97, 33), (32, 32)], 0),
])
@pytest.mark.parametrize("fp8", [False, True])
def test_suffixes_over_pages(QH, KH, D, pairs, window, fp8):
    torch.manual_seed(D + QH)
    kv, ql = [p[0] for p in pairs], [p[1] for p in pairs]
    mb = -(-max(kv) // 16)
    bt = torch.randperm(len(kv) * mb, device=DEV).int().view(len(kv), mb)
    kc, vc = (_bf16(len(kv) * mb, KH, 16, D) for _ in range(2))
    if fp8:
        k8, v8 = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
        kc, vc = k8.to(torch.bfloat16), v8.to(torch.bfloat16)
        args = (k8.view(torch.uint8), v8.view(torch.uint8))
    else:
        args = (kc, vc)
    q = _bf16(sum(ql), QH, D)
    kl = torch.tensor(kv, dtype=torch.int32, device=DEV)
    scale = D ** -0.5
    out = ops.context_attention(q, *args, _cu(ql), kl, bt, scale, window)
    ref = R.context_attention(q.cpu().float(), kc.cpu().float(),
                              vc.cpu().float(), _cu(ql).cpu(), kl.cpu(),
                              bt.cpu(), scale, window)
    _check(out, ref)


SCALES = [None, 0.1, 0.22, 1 / 16, 1 / 12]


@pytest.mark.gpu
@pytest.mark.parametrize("D,window", [(64, 32), (64, 100), (96, 40),
                                      (128, 100), (128, 1024), (256, 32),
                                      (256, 1024)])
@pytest.mark.parametrize("G", [1, 2, 4])
@pytest.mark.parametrize("scale", SCALES)
def test_rows_past_a_window(D, window, G, scale):
    """Rows that see nothing of the first key tile which their workgroup
    reads: 128 / G positions from multiples of that number, behind a window
    that starts inside a tile, with no sink to bound the maximum."""
    torch.manual_seed(D + window + G)
    lens = [window + 201, 1]
    T = sum(lens)
    q, k, v = _bf16(T, 2 * G, D), _bf16(T, 2, D), _bf16(T, 2, D)
    s = scale or D ** -0.5
    k = (k.float() * D ** -0.5 / s).to(torch.bfloat16)   # scores of order 1
    out = ops.prefill_attention(q, k, v, _cu(lens), s, window=window)
    ref = R.prefill_attention(q.float(), k.float(), v.float(), _cu(lens), s,
                              window)
    _check(out, ref.cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("D,G", [(64, 1), (64, 2), (128, 4), (256, 1),
                                 (256, 2)])
@pytest.mark.parametrize("window", [32, 100, 1024])
@pytest.mark.parametrize("fp8", [False, True])
def test_suffix_rows_past_a_window(D, G, window, fp8):
    """The same over pages, the suffix starting anywhere in a tile."""
    torch.manual_seed(D + window)
    kv, ql = [window + 333, window + 140], [201, 129]
    mb = -(-max(kv) // 16)
    bt = torch.randperm(2 * mb, device=DEV).int().view(2, mb)
    kc, vc = (_bf16(2 * mb, 2, 16, D) for _ in range(2))
    args = kc, vc
    if fp8:
        args = tuple(t.to(torch.float8_e4m3fn) for t in args)
        kc, vc = (t.to(torch.bfloat16) for t in args)
        args = tuple(t.view(torch.uint8) for t in args)
    q = _bf16(sum(ql), 2 * G, D)
    kl = torch.tensor(kv, dtype=torch.int32, device=DEV)
    out = ops.context_attention(q, *args, _cu(ql), kl, bt, D ** -0.5, window)
    ref = R.context_attention(q.float(), kc.float(), vc.float(), _cu(ql), kl,
                              bt, D ** -0.5, window)
    _check(out, ref.cpu())


@pytest.mark.gpu
def test_sinks_without_weight():
    """A sink of -inf absorbs nothing, also behind a masked first tile."""
    torch.manual_seed(5)
    T, QH, D = 300, 4, 64
    q, k, v = _bf16(T, QH, D), _bf16(T, QH, D), _bf16(T, QH, D)
    sinks = torch.tensor([float("-inf"), 0.5, -2e30, 3.0], device=DEV)
    out = ops.prefill_attention(q, k, v, _cu([T]), D ** -0.5, window=40,
                                sinks=sinks)
    ref = R.prefill_attention(q.float(), k.float(), v.float(), _cu([T]),
                              D ** -0.5, 40, sinks)
    _check(out, ref.cpu())


@pytest.mark.gpu
def test_long_prompt_of_a_windowed_model():
    """Windowed layers of 64-dim heads (window 32), prompts past the first
    masked tile: logits of the engine on the GPU and on the CPU."""
    from kaito_amd.engine import EngineConfig, LLMEngine
    from kaito_amd.models import get_model_config
    from kaito_amd.parallel.state import init_parallel
    init_parallel(1)
    n, state, logits = 300, None, []
    for dev in ("cpu", DEV):
        torch.manual_seed(11)
        eng = LLMEngine(EngineConfig(
            model=get_model_config("tiny-gemma3-test"), device=dev,
            max_num_seqs=2, max_model_len=512, num_gpu_blocks=64,
            enforce_eager=True))
        model = eng.runner.model
        if state is None:
            state = {k: t.clone() for k, t in model.state_dict().items()}
        model.load_state_dict(state)
        eng.extend_request(0, [(7 * i + 3) % 500 for i in range(n)])
        # whole, and as a suffix behind cached tokens
        logits.append(eng.step_explicit([(0, 200)],
                                        [(0, i) for i in range(200)]).cpu())
        logits.append(eng.step_explicit([(0, n - 200)],
                                        [(0, i) for i in range(n - 200)]).cpu())
    for ref, out in zip(logits[:2], logits[2:]):
        assert torch.isfinite(out).all()
        # bf16 activations through 4 layers, as in the CPU engine's
        assert (out - ref).norm() < 0.05 * ref.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("H,lens", [(1, [1, 64, 65]), (16, [200, 33]),
                                    (5, [129, 128, 127])])
def test_latent_prompts(H, lens):
    """Split heads: 128 + 64 key dims, the 64 shared by the heads."""
    torch.manual_seed(H)
    T = sum(lens)
    q = _bf16(T, H, 192)
    q_pe, k_pe = _bf16(T, H, 64), _bf16(T, 64)
    k = _bf16(T, H, 128)
    v = _bf16(H, T, 128).transpose(0, 1)
    scale = 192 ** -0.5
    out = ops.mla_prefill_attention(q[..., :128], q_pe, k, k_pe, v,
                                    _cu(lens), scale)
    qf = torch.cat([q[..., :128], q_pe], -1)
    kf = torch.cat([k, k_pe[:, None].expand(T, H, 64)], -1)
    vf = torch.cat([v, torch.zeros_like(q_pe)], -1)
    ref = R.prefill_attention(qf.cpu().float(), kf.cpu().float(),
                              vf.cpu().float(), _cu(lens).cpu(), scale)
    _check(out, ref[..., :128])


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,mode", [
    (4, 1, 128, 128, "cap"), (6, 2, 64, 32, "keep"), (4, 4, 256, 128, "sig"),
    (4, 2, 128, 64, "bias"), (2, 1, 256, 256, "chunk"),
    (8, 1, 64, 256, "gate"), (16, 1, 128, 256, "cap"),
])
def test_window_options(H, G, D, V, mode):
    """Portions behind earlier tokens, every option of the paged window
    attention, against its plain reference."""
    torch.manual_seed(H + V)
    kv, ql = [200, 64, 131], [130, 64, 33]
    mb = -(-max(kv) // 16)
    bt = torch.randperm(len(kv) * mb, device=DEV).int().view(len(kv), mb)
    kc, vc = _bf16(len(kv) * mb, G, 16, D), _bf16(len(kv) * mb, G, 16, V)
    T = sum(ql)
    q = _bf16(T, H, D)
    starts = [a - b for a, b in zip(kv, ql)]
    seq = torch.repeat_interleave(torch.arange(3), torch.tensor(ql)).int()
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, ql)])
    opt = dict(window=50)
    vec = torch.rand(H, device=DEV)
    if mode == "cap":
        opt.update(softcap=4.0, r1=vec, r2=vec * 2)
    elif mode == "keep":
        opt.update(keep_first=35, sinks=vec)
    elif mode == "sig":
        opt.update(sigmoid_bias=vec - 4.0)
    elif mode == "bias":
        opt.update(dist_bias=torch.randn(H, 40, device=DEV), temp_coef=0.1,
                   temp_every=16, window=0)
    elif mode == "chunk":
        opt.update(chunk=48)
    else:
        opt.update(gate=_bf16(T, H))
    tiles = ops.build_query_tiles(ql, DEV, starts) + (
        _cu(ql), torch.tensor(starts, dtype=torch.int32, device=DEV))
    out = ops.window_attention(q, kc, vc, bt, seq.to(DEV), pos.to(DEV),
                               D ** -0.5, tiles=tiles, **opt)
    opt = {k: t.cpu().float() if torch.is_tensor(t) else t
           for k, t in opt.items()}
    ref = ops.window_attention(q.cpu().float(), kc.cpu().float(),
                               vc.cpu().float(), bt.cpu(), seq, pos,
                               D ** -0.5, **opt)
    _check(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("fp8", [False, True])
def test_page_rows_behind_the_last_key(D, fp8):
    """What the last page holds behind a sequence has no say, in tiles read
    whole (64 and 128 keys) and in those read in part."""
    torch.manual_seed(D)
    kv, ql = [64, 79, 128, 17, 129, 1], [64, 40, 3, 17, 65, 1]
    mb = 9
    bt = torch.randperm(len(kv) * mb, device=DEV).int().view(len(kv), mb)
    kc, vc = (_bf16(len(kv) * mb, 2, 16, D) for _ in range(2))
    for b, n in enumerate(kv):          # everything behind the keys is NaN
        for i in range(mb):
            kc[bt[b, i].long(), :, max(0, min(16, n - 16 * i)):] = math.nan
            vc[bt[b, i].long(), :, max(0, min(16, n - 16 * i)):] = math.nan
    args = kc, vc
    if fp8:
        args = tuple(t.to(torch.float8_e4m3fn) for t in args)
        kc, vc = (t.to(torch.bfloat16) for t in args)
        args = tuple(t.view(torch.uint8) for t in args)
    q = _bf16(sum(ql), 4, D)
    kl = torch.tensor(kv, dtype=torch.int32, device=DEV)
    out = ops.context_attention(q, *args, _cu(ql), kl, bt, D ** -0.5)
    ref = R.context_attention(q.float(), kc.float(), vc.float(), _cu(ql), kl,
                              bt, D ** -0.5)
    _check(out, ref.cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("D,V", [(64, 64), (64, 256), (128, 32), (128, 128),
                                 (256, 64), (256, 256)])
@pytest.mark.parametrize("window,keep", [(0, 0), (100, 0), (70, 5)])
def test_pages_of_16_keys_and_others(D, V, window, keep):
    """Pages of 16 keys have copies of their own: the same keys in pages of 8
    and 32 give the same bits."""
    torch.manual_seed(D + V)
    starts, ql, mb = [130, 0, 33], [129, 70, 31], 20
    q, n = _bf16(sum(ql), 4, D), len(ql)
    k, v = _bf16(n, mb * 16, 2, D), _bf16(n, mb * 16, 2, V)
    st = torch.tensor(starts, dtype=torch.int32, device=DEV)
    tiles = ops.build_query_tiles(ql, DEV) + (_cu(ql), st)
    outs = []
    for bs in (16, 8, 32):
        pages = mb * 16 // bs
        bt = torch.randperm(n * pages, device=DEV).int().view(n, pages)
        caches = []
        for rows in (k, v):
            c = torch.empty(n * pages, 2, bs, rows.size(3), device=DEV,
                            dtype=torch.bfloat16)
            c[bt.view(-1).long()] = rows.view(n * pages, bs, 2, -1) \
                .transpose(1, 2)
            caches.append(c)
        outs.append(ops.window_attention(
            q, *caches, bt, None, None, D ** -0.5, window=window, tiles=tiles,
            keep_first=keep))
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
