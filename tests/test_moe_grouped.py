"""Grouped GEMMs of prompt-sized MoE steps (ops/csrc/moe_gemm.hip): expert
row counts around the 128- and 256-row tiles, empty experts, widths that end
inside a 256-column tile, ranks that hold part of the experts, activations,
biases, identity and shared experts. Activations and rows are bf16 between
the products (2^-8 each, f32 sums)."""
import pytest
import torch

from kaito_amd import ops

DEV = "cuda"


def _rand(*shape, std=1.0):
    return (std * torch.randn(*shape, device=DEV)).to(torch.bfloat16)


def _act(mode, h, n):
    if mode == 2:
        return h.relu().square()
    g, u = h[:, :n], h[:, n:]
    if mode == 1:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        return (u + 1) * g * torch.sigmoid(1.702 * g)
    return g * torch.sigmoid(g) * u


@pytest.mark.gpu
@pytest.mark.parametrize("counts,H,IE,mode,bias,part", [
    ([1], 64, 64, 0, False, None),
    ([127, 0, 129, 1], 128, 192, 0, True, None),
    ([0, 128, 300, 0, 77], 192, 64, 2, False, None),
    ([255, 257, 256], 128, 320, 1, True, None),
    ([900, 12], 320, 128, 0, False, None),
    ([64, 200, 3, 131], 128, 128, 0, False, (1, 2)),
    ([5] * 70, 64, 128, 1, False, None),           # more experts than lanes
])
@pytest.mark.parametrize("f32", [False, True])
def test_grouped_step(counts, H, IE, mode, bias, part, f32):
    torch.manual_seed(sum(counts))
    E, top = len(counts), 1
    T = sum(counts)
    lo, n = part or (0, E)
    topi = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    topi = topi[torch.randperm(T)].to(DEV).int()[:, None]
    topw = torch.rand(T, top, device=DEV) + 0.5
    x, shared = _rand(T, H), _rand(T, H)
    rows = 1 if mode == 2 else 2
    wu = _rand(E, rows * IE, H, std=H ** -0.5)
    wd = _rand(E, H, IE, std=IE ** -0.5)
    bu = _rand(E, 2 * IE) if bias else None
    bd = _rand(E, H) if bias else None
    w_id = torch.rand(T, device=DEV)
    tok, gates, off, pos = ops.moe_plan(topi, topw, E)
    act = torch.full((T, IE), float("nan"), device=DEV).to(torch.bfloat16)
    y = torch.full((T, H), float("nan"), device=DEV)
    y = y if f32 else y.to(torch.bfloat16)
    cut = slice(lo, lo + n)
    ops.moe_grouped_up(act, x, wu[cut].contiguous(), tok, off, lo,
                       bu[cut].contiguous() if bias else None, mode, 7.0)
    ops.moe_grouped_down(y, act, wd[cut].contiguous(), off, lo,
                         bd[cut].contiguous() if bias else None)
    out = torch.empty(T, H, device=DEV, dtype=torch.float32 if f32
                      else torch.bfloat16)
    ops.moe_combine(out, y, pos, topi, topw, lo, n, x, w_id, shared)
    ref = x.double() * w_id[:, None].double() + shared.double()
    for e in range(lo, lo + n):
        t = torch.nonzero(topi[:, 0] == e)[:, 0]
        h = x[t].double() @ wu[e].double().T
        if bias:
            h = h + bu[e].double()
        v = _act(mode, h, IE) @ wd[e].double().T
        if bias:
            v = v + bd[e].double()
        ref[t] += v * topw[t].double()
    assert torch.isfinite(out).all()
    err = (out.double() - ref).abs()
    rms = ref.square().mean().sqrt()
    # act and y rounded once each, out once: a few 2^-9 of the row's size
    assert err.max() <= 2.0 ** -5 * rms, err.max() / rms
    assert err.square().mean().sqrt() <= 2.0 ** -7.5 * rms


@pytest.mark.gpu
@pytest.mark.parametrize("counts,H,IE,mode,bias", [
    ([5000, 0, 130, 500], 1600, 1600, 0, True),    # 38 and 21 tiles per XCD
    ([700, 3201], 64, 1088, 2, False),             # 10 and 2; a K of 64
    ([4097, 1100], 192, 2176, 1, False),
])
def test_grouped_rounds(counts, H, IE, mode, bias):
    """Whole rounds of tiles, last ones in quarters or not, few steps of K."""
    test_grouped_step(counts, H, IE, mode, bias, None, False)


@pytest.mark.gpu
@pytest.mark.parametrize("counts,H,IE,mode,bias", [
    ([1800, 1400, 1100, 700, 500, 300, 120, 81], 2880, 1024, 0, False),
    ([200] * 15, 320, 1088, 0, True),          # up: 256 rows x 128 weight rows
    ([250, 130] * 4, 384, 1600, 1, True),
    ([120] * 8, 320, 2048, 0, False),          # 128 x 128, one round
    ([20] * 64, 1024, 512, 0, False),          # two of them
    ([130, 1] * 9, 576, 2112, 2, False),       # 128 x 256
    ([90, 0, 128] * 23, 64, 512, 0, True),     # more experts than lanes
])
@pytest.mark.parametrize("f32", [False, True])
def test_grouped_shapes(counts, H, IE, mode, bias, f32):
    """Each shape of tiles, several rounds of one, the same one on all XCDs."""
    test_grouped_step(counts, H, IE, mode, bias, None, f32)


@pytest.mark.gpu
@pytest.mark.parametrize("counts,H,IE,mode,bias,part", [
    ([1], 64, 64, 0, False, None),
    ([3, 0, 16, 17, 1], 256, 192, 0, True, None),
    ([0, 15, 33], 192, 512, 2, False, None),
    ([70, 2], 512, 64, 1, True, None),
    ([9, 20, 3, 12], 128, 128, 0, True, (1, 2)),
    ([2] * 70, 64, 256, 1, False, None),
])
def test_streamed_step(counts, H, IE, mode, bias, part):
    """The decode-sized kernels (ops/csrc/moe.hip): passes of 16 and 32 rows
    per expert, K in stages of 256 and 64."""
    torch.manual_seed(sum(counts))
    E, T = len(counts), sum(counts)
    lo, n = part or (0, E)
    topi = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    topi = topi[torch.randperm(T)].to(DEV).int()[:, None]
    topw = torch.rand(T, 1, device=DEV) + 0.5
    x = _rand(T, H)
    wu = _rand(E, (1 if mode == 2 else 2) * IE, H, std=H ** -0.5)
    wd = _rand(E, H, IE, std=IE ** -0.5)
    bu = _rand(E, 2 * IE) if bias and mode != 2 else None
    bd = _rand(E, H) if bias else None
    tok, _, off, pos = ops.moe_plan(topi, topw, E)
    cut = slice(lo, lo + n)
    act = torch.full((T, IE), float("nan"), device=DEV).to(torch.bfloat16)
    y = torch.full((T, H), float("nan"), device=DEV)
    out = torch.empty(T, H, device=DEV)
    ops.moe_gate_silu(act, x, wu[cut].contiguous(), tok, off, lo, n,
                      bu[cut].contiguous() if bu is not None else None, mode,
                      7.0)
    ops.moe_down_rows(y, act, wd[cut].contiguous(), off, lo, n,
                      bd[cut].contiguous() if bias else None)
    ops.moe_combine(out, y, pos, topi, topw, lo, n)
    ref = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in range(lo, lo + n):
        t = torch.nonzero(topi[:, 0] == e)[:, 0]
        h = x[t].double() @ wu[e].double().T
        if bu is not None:
            h = h + bu[e].double()
        v = _act(mode, h, IE) @ wd[e].double().T
        if bias:
            v = v + bd[e].double()
        ref[t] = v * topw[t].double()
    rms = ref.square().mean().sqrt()
    err = (out.double() - ref).abs()    # act rounded to bf16 once
    assert err.max() <= 2.0 ** -5.5 * rms, err.max() / rms
    assert err.square().mean().sqrt() <= 2.0 ** -8 * rms


@pytest.mark.gpu
@pytest.mark.parametrize("counts,IE,mode,bias,part", [
    ([5, 0, 16, 17, 1, 40, 3, 33], 2048, 0, True, None),
    ([2, 1, 3, 0, 1, 1, 2, 2], 2048, 2, False, None),
    ([16, 9, 1, 30, 2, 8, 7], 1600, 1, True, (1, 5)),
])
def test_streamed_step_staying(counts, IE, mode, bias, part):
    """K = 2048 and enough tiles: workgroups that go from tile to tile."""
    test_streamed_step(counts, 2048, IE, mode, bias, part)


@pytest.mark.gpu
def test_several_choices_sum():
    torch.manual_seed(3)
    T, H, K = 50, 2056, 6
    y = _rand(T * K, H)
    topi = torch.randint(0, 9, (T, K), device=DEV).int()
    topw = torch.rand(T, K, device=DEV)
    pos = torch.randperm(T * K, device=DEV).int()
    out = torch.empty(T, H, device=DEV)
    ops.moe_combine(out, y, pos, topi, topw, 2, 5)
    live = ((topi >= 2) & (topi < 7)).double() * topw.double()
    ref = (y[pos.long()].view(T, K, H).double() * live[..., None]).sum(1)
    assert torch.allclose(out.double(), ref, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,H,IE,mode,ident,part", [
    (1, 4, 1, 64, 64, 0, 0, None),
    (33, 5, 3, 256, 128, 1, 0, (1, 3)),
    (64, 9, 4, 128, 192, 2, 2, None),           # 256 pairs, identity experts
    (32, 8, 2, 2048, 2048, 0, 0, None),         # workgroups that stay
    (100, 8, 2, 2048, 1536, 0, 1, (2, 6)),
])
def test_rows_of_pairs(T, E, top, H, IE, mode, ident, part):
    """Experts that find their own rows write what sorted ones hold."""
    torch.manual_seed(T + E)
    lo, n = part or (0, E)
    topi = torch.stack([torch.randperm(E + ident, device=DEV)[:top]
                        for _ in range(T)]).int()
    topw = torch.rand(T, top, device=DEV)
    x = _rand(T, H)
    wu = _rand(n, (1 if mode == 2 else 2) * IE, H, std=H ** -0.5)
    wd = _rand(n, H, IE, std=IE ** -0.5)
    bd = _rand(n, H)
    tok, _, off, pos = ops.moe_plan(topi, topw, E + ident)
    act = torch.zeros(T * top, IE, device=DEV, dtype=torch.bfloat16)
    y = torch.zeros(T * top, H, device=DEV)
    act2, y2 = act.clone(), y.clone()
    ops.moe_gate_silu(act, x, wu, tok, off, lo, n, None, mode)
    ops.moe_down_rows(y, act, wd, off, lo, n, bd)
    ops.moe_up_pairs(act2, x, wu, topi, E + ident, lo, n, None, mode)
    ops.moe_down_pairs(y2, act2, wd, topi, E + ident, lo, n, bd)
    assert torch.equal(act2, act[pos.long()])
    assert torch.equal(y2, y[pos.long()])
    a, b = (torch.empty(T, H, device=DEV) for _ in range(2))
    w_id = torch.rand(T, device=DEV)
    ops.moe_combine(a, y, pos, topi, topw, lo, n, x, w_id, x)
    ops.moe_combine(b, y2, None, topi, topw, lo, n, x, w_id, x)
    assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("T,H", [(1, 8), (3, 2048), (5, 2056), (2, 4104),
                                 (2, 8192)])
@pytest.mark.parametrize("wide", [True, False])
@pytest.mark.parametrize("post", [True, False])
def test_sum_and_norm(T, H, wide, post):
    """The sum over the experts inside the residual norm behind it."""
    torch.manual_seed(H)
    topi = torch.randint(0, 4, (T, 2), device=DEV).int()
    topw = torch.rand(T, 2, device=DEV)
    y = torch.randn(2 * T, H, device=DEV)
    y = y if wide else y.to(torch.bfloat16)
    shared = _rand(T, H)
    args = (y, None, topi, topw, 1, 3, None, None, shared)
    s = torch.empty(T, H, device=DEV, dtype=torch.bfloat16)
    ops.moe_combine(s, *args)
    if post:
        res, w = torch.randn(T, H, device=DEV), torch.rand(H, device=DEV)
        r2 = res.clone()
        ref = ops.post_norm_residual(res, s, w, 1e-5, torch.bfloat16)
    else:
        res, w = _rand(T, H), _rand(H)
        r2 = res.clone()
        ref, res = ops.fused_add_rms_norm(s, res, w, 1e-5)
    out = ops.moe_combine_norm(r2, w, 1e-5, *args)
    # sums of squares in another order: 2^-20 of the factor, then one rounding
    assert ((r2 - res).abs() <= 2.0 ** -20 * (1 + res.abs())).all() if post \
        else torch.equal(r2, res)
    assert ((out.float() - ref.float()).abs()
            <= 2.0 ** -7 * ref.float().abs()).all()
    assert (out != ref).float().mean() < 0.02


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,N,f32", [(1, 8, 2, False), (32, 2048, 8, False),
                                       (3, 2056, 32, True),
                                       (300, 8192, 20, False)])
def test_norm_and_choice(T, H, N, f32):
    """The residual norm inside the router's launch."""
    torch.manual_seed(H + N)
    x, res, w = _rand(T, H), _rand(T, H), _rand(H)
    gate = torch.randn(N, H, device=DEV).to(torch.float32 if f32
                                            else torch.bfloat16)
    ref, r1 = ops.fused_add_rms_norm(x, res.clone(), w, 1e-5)
    xn, r2, *chosen = ops.moe_norm_gate_route(x, res, w, 1e-5, gate, None, 2, N)
    assert torch.equal(r1, r2)
    assert ((xn.float() - ref.float()).abs()
            <= 2.0 ** -7 * ref.float().abs()).all()
    assert (xn != ref).float().mean() < 0.02
    for a, b in zip(chosen, ops.moe_gate_route(xn, gate, None, 2, N)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("pairs,n_local,ff,H,pay", [
    (2, 8, 2048, 2048, True), (256, 8, 2048, 2048, True),
    (257, 8, 2048, 2048, False), (32, 16, 2880, 2880, True),
    (2, 8, 4096, 4096, False), (24, 8, 4096, 4096, True),
    (4, 16, 1024, 2048, False), (8, 16, 1024, 2048, True),
    (2, 8, 14336, 4096, False), (4, 24, 1024, 2048, False),
    (2, 32, 2048, 2048, False), (256, 128, 768, 2048, False)])
def test_which_steps_go_by_pairs(pairs, n_local, ff, H, pay):
    """The sides of the line on which either was measured to be faster."""
    assert ops.moe_pairs_pay(pairs, n_local, 2 * ff, H) == pay
