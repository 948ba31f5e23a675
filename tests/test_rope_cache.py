"""Rotation and cache scatter in one launch (ops/csrc/rope.hip) against the
two single kernels, bit for bit."""
import pytest
import torch

from kaito_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,QH,KH,D,R", [(1, 32, 8, 128, 128), (7, 4, 4, 64, 64),
                                         (300, 8, 1, 256, 256),
                                         (33, 6, 2, 80, 32), (5, 3, 3, 96, 16)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("pad", [0, 8, 4])
def test_matches_single_kernels(T, QH, KH, D, R, fp8, pad):
    torch.manual_seed(T + D)
    qkv = torch.randn(T, (QH + 2 * KH) * D + pad, device=DEV).to(torch.bfloat16)
    pos = torch.randint(0, 500, (T,), device=DEV)
    cs = torch.randn(500, R, device=DEV)
    nb = (T + 15) // 16 + 2
    slots = torch.randperm(nb * 16, device=DEV)[:T]
    slots[T // 2] = -1
    dt = torch.uint8 if fp8 else torch.bfloat16
    caches = [[torch.zeros(nb, KH, 16, D, device=DEV, dtype=dt)
               for _ in range(2)] for _ in range(2)]
    results = []
    for fused, (kc, vc) in zip((False, True), caches):
        buf = qkv.clone()
        q, k, v = buf[:, :(QH + 2 * KH) * D].split(
            [QH * D, KH * D, KH * D], -1)
        if fused:
            q, k = ops.rope_and_cache(pos, q, k, v, D, cs, kc, vc, slots)
        else:
            q, k = ops.rotary_embedding(pos, q, k, D, cs)
            ops.reshape_and_cache(k.unflatten(-1, (KH, D)),
                                  v.unflatten(-1, (KH, D)), kc, vc, slots)
        results.append((q, k, v, kc, vc))
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_plain_tensors_on_the_host():
    q, k, v = torch.randn(3, 64), torch.randn(3, 32), torch.randn(3, 32)
    kc, vc = torch.zeros(2, 2, 16, 16), torch.zeros(2, 2, 16, 16)
    pos, slots = torch.arange(3), torch.tensor([4, 0, 17])
    cs = torch.randn(8, 16)
    a, b = ops.rope_and_cache(pos, q.clone(), k.clone(), v, 16, cs, kc, vc,
                              slots)
    qr, kr = ops.rotary_embedding(pos, q, k, 16, cs)
    assert torch.equal(a, qr) and torch.equal(b, kr)
    assert torch.equal(kc[1, :, 1], kr[2].view(2, 16))
