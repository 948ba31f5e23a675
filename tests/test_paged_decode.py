"""The MFMA decode attention (ops/csrc/paged_attention_sp.hip) at the edges
of its 32-key tiles and of the rules that choose 2, 4 or 8 waves per
workgroup and several workgroups per (sequence, kv head). Weights are f32, so
the outputs are off by their rounding to bf16 (2^-9) and f32 sums; the bound
is four times that at the values' largest magnitude."""
import pytest
import torch

from kaito_amd import ops
from kaito_amd.ops import torch_ref as R

DEV = "cuda"


def _run(G, KH, D, lens, max_blocks=None, window=0, sink=False, fp8=False):
    torch.manual_seed(G * D + len(lens))
    mb = max(max_blocks or 0, -(-max(lens) // 16), 1)
    used = [-(-n // 16) for n in lens]
    perm = torch.randperm(sum(used) + 1)
    bt = torch.zeros(len(lens), mb, dtype=torch.int32)
    at = 0
    for i, n in enumerate(used):
        bt[i, :n] = perm[at:at + n]
        at += n
    kc, vc = (torch.randn(sum(used) + 1, KH, 16, D).to(torch.bfloat16)
              for _ in range(2))
    args = (kc, vc)
    if fp8:
        args = tuple(t.to(torch.float8_e4m3fn) for t in args)
        kc, vc = (t.to(torch.bfloat16) for t in args)
        args = tuple(t.view(torch.uint8) for t in args)
    # a strided query, as cut from a fused projection
    q = torch.randn(len(lens), G * KH * D + 64).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    sinks = torch.randn(G * KH) if sink else None
    q3 = q.to(DEV)[:, :G * KH * D].unflatten(-1, (-1, D))
    out = ops.paged_attention(
        q3, *(t.to(DEV) for t in args), bt.to(DEV), sl.to(DEV), D ** -0.5,
        window, sinks.to(DEV) if sink else None).cpu().float()
    live = [i for i, n in enumerate(lens) if n > 0]
    ref = R.paged_attention(q3.cpu().float()[live], kc.float(), vc.float(),
                            bt[live], sl[live], D ** -0.5, window, sinks)
    assert torch.isfinite(out).all()
    err = (out[live] - ref).abs()
    assert (err <= 2.0 ** -7 * (ref.abs() + 0.1)).all(), err.max()
    dead = [i for i, n in enumerate(lens) if n == 0]
    assert (out[dead] == 0).all()


EDGES = [1, 15, 16, 17, 31, 32, 33, 0, 64, 65, 127, 128, 129, 300]


@pytest.mark.gpu
@pytest.mark.parametrize("G,KH,D", [(1, 2, 64), (8, 1, 64), (1, 1, 128),
                                    (3, 2, 128), (4, 2, 128), (7, 1, 128),
                                    (8, 1, 128), (1, 2, 256), (4, 1, 256)])
@pytest.mark.parametrize("fp8", [False, True])
def test_edges(G, KH, D, fp8):
    _run(G, KH, D, EDGES, fp8=fp8)
    _run(G, KH, D, EDGES, max_blocks=17, window=40, sink=not fp8, fp8=fp8)


@pytest.mark.gpu
@pytest.mark.parametrize("KH,lens,max_blocks", [
    (8, [40, 200, 7] * 11, 13),           # 264 pairs
    (8, [64, 70, 90, 3] * 17, 6),         # 544 pairs
    (2, [1900, 33, 0, 2047], 128),        # few pairs, long table: splits
    (1, [5000], 700),
    (8, [17], 4096),                      # splits that are all but one empty
])
@pytest.mark.parametrize("D,fp8", [(128, False), (128, True), (256, False)])
def test_launch_rules(KH, lens, max_blocks, D, fp8):
    _run(4, KH, D, lens, max_blocks, fp8=fp8)
    _run(2, KH, D, lens, max_blocks, window=530, sink=True, fp8=fp8)


@pytest.mark.gpu
@pytest.mark.parametrize("D,pairs,max_blocks", [
    (128, 128, 64), (128, 129, 64),           # splits or none
    (64, 512, 8), (64, 513, 8), (128, 256, 8), (128, 257, 8),   # 8 | 4 waves
    (64, 1024, 8), (64, 1025, 8), (64, 2048, 8), (64, 2049, 8),  # 4 | 2 | 4
    (128, 768, 8), (128, 769, 8), (128, 1536, 8), (128, 1537, 8),
    (256, 512, 8), (256, 513, 8), (256, 1024, 8), (256, 1025, 8),
    (64, 4095, 8), (64, 4096, 8), (256, 4096, 8), (128, 4096, 16),  # 4 | 2 | 4
])
@pytest.mark.parametrize("fp8", [False, True])
def test_pair_lines(D, pairs, max_blocks, fp8):
    """Both sides of the lines between numbers of waves."""
    lens = [(i * 37) % 97 for i in range(pairs)]
    _run(2, 1, D, lens, max_blocks, sink=fp8, fp8=fp8)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("window,sink", [(0, False), (0, True), (700, True)])
def test_split_edges(D, window, sink):
    """Under a table that asks for splits: sequences whose keys the first
    workgroup has alone (8 tiles) and one key more, and twice to four times
    as many."""
    _run(4, 2, D, [0, 1, 256, 257, 512, 513, 1024, 1025, 2048, 6000], 4096,
         window, sink)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("window", [0, 20])
def test_slots_outside_the_sequence(D, fp8, window):
    """What a page's last user left behind the sequence's end, or before its
    window, has no say, not even a NaN."""
    lens = [1, 4, 8, 15, 16, 17, 28, 32, 36, 52]
    bt = torch.arange(4 * len(lens), dtype=torch.int32).view(-1, 4)
    kc, vc = (torch.randn(bt.numel(), 2, 16, D).to(torch.bfloat16)
              for _ in range(2))
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn).to(torch.bfloat16)
                  for t in (kc, vc))
    dead_k, dead_v = kc.clone(), vc.clone()
    for i, n in enumerate(lens):
        key = torch.arange(64).view(4, 16)
        out = (key >= n) | (key < n - window if window else key < 0)
        for t in (dead_k, dead_v):
            t[bt[i].long()] = torch.where(
                out[:, None, :, None], float("nan"), t[bt[i].long()].float()
            ).to(torch.bfloat16)
    q = torch.randn(len(lens), 4, D).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    got = []
    for c in ((dead_k, dead_v), (kc, vc)):
        if fp8:
            c = tuple(t.to(torch.float8_e4m3fn).view(torch.uint8) for t in c)
        got.append(ops.paged_attention(
            q.to(DEV), *(t.to(DEV) for t in c), bt.to(DEV), sl.to(DEV),
            D ** -0.5, window).cpu())
    assert torch.equal(*got)


@pytest.mark.gpu
@pytest.mark.parametrize("D,KH,gap,max_blocks", [
    (128, 8, 2, 1), (128, 1, 40, 4), (64, 8, 20, 2), (256, 2, 700, 60),
    (128, 2, 5000, 400),              # other tiles, waves and splits
])
def test_weights_keep_f32(D, KH, gap, max_blocks):
    """One key of weight w = exp(-s) and value -1 against keys of weight 1
    whose values sum to w up to 2^-14: what is left shows w's error 2^14
    times larger. f32 weights and sums are off by a few 2^-24, so what is
    left by 2^-8 and its rounding, 2^-9; 16-bit weights by up to 2^-3."""
    torch.manual_seed(D + gap)
    T, nb = 64, max_blocks * 64 + 1
    bt = torch.arange(1, nb, dtype=torch.int32).view(T, -1)
    n = gap + 3                       # keys: two of weight 1, filler, w
    kc, vc = (torch.zeros(nb, KH, 16, D).to(torch.bfloat16)
              for _ in range(2))
    kc[..., 0] = -4096.0              # filler weighs nothing
    x = (torch.rand(T, KH) * 0.9 + 0.05) * D ** 0.5
    x = x.to(torch.bfloat16).double()
    w = torch.exp(-x * torch.tensor(D ** -0.5, dtype=torch.float32).double())
    target = w * (1 + 2.0 ** -14)
    v1 = target.to(torch.bfloat16).double()
    v2 = (target - v1).to(torch.bfloat16).double()

    def row(t, key):
        return int(bt[t, key // 16]), key % 16
    for t in range(T):
        b, o = row(t, n - 1)
        kc[b, :, o, 0] = -x[t].to(torch.bfloat16)
        vc[b, :, o] = -1.0
        for key, v in ((0, v1), (1, v2)):
            b, o = row(t, key)
            kc[b, :, o, 0] = 0.0
            vc[b, :, o] = v[t].to(torch.bfloat16)[:, None]
    q = torch.zeros(T, KH, D).to(torch.bfloat16)
    q[..., 0] = 1.0
    sl = torch.full((T,), n, dtype=torch.int32)
    out = ops.paged_attention(*(t.to(DEV) for t in (q, kc, vc, bt, sl)),
                              D ** -0.5).cpu().double()
    ref = (v1 + v2 - w) / (2 + w)
    err = ((out - ref[..., None]) / ref[..., None]).abs()
    assert err.max() < 2.0 ** -6, err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("G,KH,D", [(1, 2, 64), (8, 1, 64), (3, 2, 128),
                                    (4, 8, 128), (4, 1, 256)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens,max_blocks,window", [
    (EDGES, 20, 0), (EDGES, 20, 40), ([1900, 33, 1, 2047], 128, 0),
    ([1, 16, 17, 300] * 70, 19, 0)])
def test_rotated_on_the_way(G, KH, D, fp8, lens, max_blocks, window):
    """One launch or rope_and_cache and attention behind it: the same pages and
    results, rows without a slot and slots of no sequence's page among them."""
    torch.manual_seed(G * D + len(lens))
    T, pages = len(lens), sum(-(-n // 16) for n in lens) + 2
    perm = torch.randperm(pages)
    bt = torch.zeros(T, max_blocks, dtype=torch.int32)
    slots = torch.full((T,), -1)
    at = 0
    for i, n in enumerate(lens):
        u = -(-n // 16)
        bt[i, :u] = perm[at:at + u]
        if n and i % 5 != 3:
            slots[i] = int(bt[i, (n - 1) // 16]) * 16 + (n - 1) % 16
        at += u
    slots[0] = int(perm[-1]) * 16 + 5        # a page that nobody reads
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [torch.randn(pages, KH, 16, D, device=DEV).to(dt) for _ in "kv"]
    if fp8:
        caches = [c.view(torch.uint8) for c in caches]
    qkv = torch.randn(T, (G + 2) * KH * D + 8, device=DEV).to(torch.bfloat16)
    q, k, v = qkv[:, 8:].split([G * KH * D, KH * D, KH * D], -1)
    pos = torch.randint(0, 500, (T,), device=DEV)
    cs = torch.randn(500, D, device=DEV)
    bt, slots = bt.to(DEV), slots.to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    sinks = torch.randn(G * KH, device=DEV) if window else None
    a, b = ([c.clone() for c in caches] for _ in "ab")
    before = qkv.clone()
    out = ops.rope_paged_attention(pos, q, k, v, D, cs, *a, slots, bt, sl,
                                   D ** -0.5, window, sinks)
    assert torch.equal(qkv, before)
    q, k = ops.rope_and_cache(pos, q, k, v, D, cs, *b, slots)
    ref = ops.paged_attention(q.unflatten(-1, (-1, D)), *b, bt, sl, D ** -0.5,
                              window, sinks)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    assert torch.isfinite(out).all() and torch.equal(out, ref)


@pytest.mark.gpu
def test_rotations_at_any_address():
    """A table that does not start on 16 bytes takes the two launches."""
    D, KH, G = 64, 2, 2
    table = torch.randn(32 * D + 1, device=DEV)
    caches = [torch.randn(3, KH, 16, D, device=DEV).bfloat16() for _ in "kv"]
    qkv = torch.randn(2, (G + 2) * KH * D, device=DEV).bfloat16()
    pos = torch.tensor([3, 17], device=DEV)
    slots = torch.tensor([16 + 3, 32 + 1], device=DEV)
    bt = torch.tensor([[1, 0], [0, 2]], dtype=torch.int32, device=DEV)
    sl = torch.tensor([4, 18], dtype=torch.int32, device=DEV)
    outs = []
    for odd in (False, True):
        cs = table[1:].view(32, D)
        assert cs.data_ptr() % 16
        cs = cs if odd else cs.clone()
        q, k, v = qkv.clone().split([G * KH * D, KH * D, KH * D], -1)
        outs.append(ops.rope_paged_attention(
            pos, q, k, v, D, cs, *(c.clone() for c in caches), slots, bt, sl,
            D ** -0.5))
    assert torch.equal(*outs)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
def test_codes_are_widened_exactly(D):
    """One key per row weighs 1: the output is its value, whatever its code."""
    T = 256 // D
    codes = torch.arange(256, dtype=torch.uint8).view(T, 1, 1, D)
    kc = torch.full((T, 1, 16, D), 0x38, dtype=torch.uint8)     # 1.0
    vc = torch.zeros(T, 1, 16, D, dtype=torch.uint8)
    vc[:, :, :1] = codes
    bt, sl = torch.arange(T, dtype=torch.int32).view(T, 1), torch.ones(T)
    out = ops.paged_attention(
        torch.randn(T, 1, D, dtype=torch.bfloat16, device=DEV), kc.to(DEV),
        vc.to(DEV), bt.to(DEV), sl.int().to(DEV), D ** -0.5)
    want = codes.view(torch.float8_e4m3fn).float().view(T, 1, D)
    assert torch.equal(out.cpu().float().nan_to_num(1e9), want.nan_to_num(1e9))
