"""Kernels around absorbed MLA attention (ops/csrc/mla_attention.hip)."""
import pytest
import torch

from kaito_amd import ops
from kaito_amd.ops import torch_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf16(*shape, scale=1.0):
    return (torch.randn(*shape, device=DEV) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("H,lens,room", [
    (16, [1], 1), (16, [33, 16, 0, 15, 31, 32, 129, 1], 16),
    (20, [3000, 17, 2049], 190), (1, [700] * 9, 44), (128, [513, 64], 300),
    (16, [257 + 3 * i for i in range(270)], 68),
    (128, [1 + 3 * i for i in range(70)], 14),
    (120, [1 + 2 * i for i in range(131)], 17)])
def test_decode(H, lens, room):
    """Spans of a wave, splits (more table room than keys too), head tiles
    with unused columns, sequences that do not fill the last group of 8;
    whole rows of q and the two parts of it."""
    torch.manual_seed(H)
    T, BS = len(lens), 16
    nb = [(n + BS - 1) // BS for n in lens]
    cache = _bf16(sum(nb) + 1, BS, 576)
    bt = torch.zeros(T, max(room, max(nb)), dtype=torch.int32, device=DEV)
    perm = (torch.randperm(sum(nb)) + 1).int().to(DEV)
    at = 0
    for i, n in enumerate(nb):
        bt[i, :n] = perm[at:at + n]
        at += n
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = _bf16(T, H, 576, scale=0.5)
    scale = 192 ** -0.5
    out = ops.mla_decode(q, cache, bt, sl, scale, 512)
    parts = _bf16(H, T, 512), _bf16(T, H, 72)
    parts[0].copy_(q[..., :512].transpose(0, 1))
    parts[1][..., 8:].copy_(q[..., 512:])
    again = ops.mla_decode(parts[0].transpose(0, 1), cache, bt, sl, scale, 512,
                           parts[1][..., 8:])
    assert torch.equal(out, again)
    for i, n in enumerate(lens):
        if n == 0:
            assert not out[i].any()
            continue
        rows = cache[bt[i, :nb[i]].long()].reshape(-1, 576)[:n].double()
        p = torch.softmax(q[i].double() @ rows.T * scale, -1)
        ref = p @ rows[:, :512]
        # weights to 2^-9 each, independent; the result to 2^-9
        spread = (p.square() @ rows[:, :512].square()).sqrt()
        bound = 2.0 ** -9 * (ref.abs() + 6 * spread) + 1e-5
        assert ((out[i].double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("T,H,cached", [(1, 16, True), (5, 1, True),
                                        (33, 128, True), (7, 20, False)])
def test_prepare(T, H, cached):
    torch.manual_seed(T)
    q = _bf16(T, H, 192)
    kv_a, w = _bf16(T, 576), _bf16(512)
    pos = torch.randint(0, 100, (T,), device=DEV)
    cs = torch.randn(100, 64, device=DEV)
    cache = _bf16(6, 16, 576)
    slots = torch.randperm(96, device=DEV)[:T]
    slots[T // 2] = -1
    want = cache.clone()
    qp, c, k = ops.mla_prepare(q[..., 128:], kv_a, w, 1e-6, pos, cs,
                               cache if cached else None,
                               slots if cached else None)
    c0 = ops.rms_norm(kv_a[:, :512].contiguous(), w, 1e-6)
    q0, k0 = ops.rotary_embedding(
        pos, q[..., 128:].contiguous().view(T, -1),
        kv_a[:, 512:].contiguous(), 64, cs)
    assert torch.equal(qp.view(T, -1), q0) and torch.equal(k, k0)
    # the norm's sum in another order: one rounding
    assert ((c.float() - c0.float()).abs() <= 2.0 ** -7 * c0.abs()).all()
    if cached:
        ops.mla_cache_write(want, c, k, slots)
    assert torch.equal(cache, want)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33])
@pytest.mark.parametrize("H,K,N", [(1, 64, 32), (16, 128, 512),
                                   (3, 512, 128), (2, 192, 96)])
def test_head_rows(T, H, K, N):
    """One and two row tiles, halves of K, and the library beyond."""
    torch.manual_seed(T + K)
    x = _bf16(T, H, K + 64)[..., 32:32 + K]
    w = _bf16(H, K, N, scale=K ** -0.5)
    y = ops.head_rows(x, w)
    ref = torch.einsum("thk,hkn->thn", x.double(), w.double())
    mag = torch.einsum("thk,hkn->thn", x.double().abs(), w.double().abs())
    err = (y.double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -18 * mag).all()


def test_single_operations_agree():
    """mla_decode of the plain reference, CPU side of both argument forms."""
    q = torch.randn(2, 3, 576)
    cache, bt = torch.randn(4, 16, 576), torch.tensor([[1, 2], [3, 0]]).int()
    sl = torch.tensor([20, 9]).int()
    a = ops.mla_decode(q, cache, bt, sl, 0.1, 512)
    b = ops.mla_decode(q[..., :512], cache, bt, sl, 0.1, 512, q[..., 512:])
    assert torch.equal(a, b)
    assert torch.equal(a, R.mla_decode(q, cache, bt, sl, 0.1, 512))


@pytest.mark.parametrize("T,H,K,N,cached", [(1, 16, 128, 512, True),
                                            (16, 3, 64, 96, True),
                                            (17, 16, 128, 512, False),
                                            (32, 20, 128, 512, True)])
def test_prepare_beside_head_rows(T, H, K, N, cached):
    """One launch or two: the same bits."""
    torch.manual_seed(T + H)
    q, w, wx = _bf16(T, H, K + 64), _bf16(512), _bf16(H, K, N)
    kv_a = _bf16(T, 576)
    pos = torch.randint(0, 100, (T,), device=DEV)
    cs = torch.randn(100, 64, device=DEV)
    slots = torch.randperm(96, device=DEV)[:T]
    slots[T // 2] = -1
    a = _bf16(6, 16, 576)
    b = a.clone()
    args = (q[..., K:], kv_a, w, 1e-6, pos, cs)
    got = ops.mla_prepare_rows(q[..., :K], wx, *args, a if cached else None,
                               slots if cached else None)
    want = (ops.head_rows(q[..., :K], wx),
            *ops.mla_prepare(*args, b if cached else None,
                             slots if cached else None))
    for x, y in zip(got, want):
        assert torch.equal(x, y)
    assert torch.equal(a, b)


@pytest.mark.parametrize("T,H,D,V,K", [(4096, 16, 128, 128, 512),
                                       (4101, 16, 128, 128, 512),
                                       (16390, 8, 64, 64, 192),
                                       (5471, 12, 64, 192, 64)])
def test_latent_kv(T, H, D, V, K):
    """Rows and columns that end inside a tile; below the tiles' size the
    library. Sums of up to 512 f32 products, rounded to bf16 once."""
    torch.manual_seed(T + K)
    c = _bf16(T, K)
    wk, wv = _bf16(H, D, K, scale=K ** -0.5), _bf16(H, K, V, scale=K ** -0.5)
    for rows in (T, 33):
        k, v = ops.latent_kv(c[:rows], wk, wv)
        for out, w in ((k, wk.transpose(1, 2)), (v, wv)):
            w = w.contiguous()
            for h in (0, H // 2, H - 1):
                ref = c[:rows].double() @ w[h].double()
                rms = ref.square().mean().sqrt()
                err = (out[:, h].double() - ref).abs()
                assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * rms).all()


@pytest.mark.parametrize("T,N,r,tiles", [
    (4096, 4096, 512, True), (4095, 4096, 512, False), (512, 32768, 512, True),
    (3000, 32768, 1536, True), (512, 32768, 1536, False),
    (640, 32768, 1536, True), (2048, 4096, 1024, False),
    (4096, 4096, 1536, True), (6000, 32768, 1536, True),
    (8192, 2048, 256, True)])
def test_which_prompts_take_tiles(T, N, r, tiles):
    """The sides of the line on which either was measured to be faster."""
    assert ops._latent_tiles(T, N, r) == tiles
