"""Expert choice and expert sort (ops/csrc/moe_route.hip) against their plain
references: modes, groups, router sizes around a wave's 64 lanes, and the
logits formed in the same launch. Scores are f32 on both sides; choices are
compared where the reference decides by more than the logits' rounding."""
import pytest
import torch

from kaito_amd import ops
from kaito_amd.ops import torch_ref as R

DEV = "cuda"


def _check(got, want, N):
    (gi, gw, gd), (wi, ww, wd) = got, want
    full = [torch.zeros(wi.size(0), N, device=DEV).scatter_(
        1, i.long().to(DEV), w.to(DEV)) for i, w in ((gi, gw), (wi, ww))]
    assert torch.allclose(full[0], full[1], atol=2e-5), \
        (full[0] - full[1]).abs().max()
    assert torch.allclose(gd, wd.to(DEV), atol=2e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "logits"])
@pytest.mark.parametrize("T,N,top,groups,keep", [
    (1, 1, 1, 1, 1), (5, 8, 2, 4, 2), (33, 64, 6, 8, 3), (7, 65, 4, 1, 1),
    (130, 160, 6, 8, 3), (9, 256, 8, 8, 4), (4, 1000, 3, 1, 1),
    (6, 12, 3, 12, 5)])
def test_choice(mode, T, N, top, groups, keep):
    torch.manual_seed(T + N)
    z = 2 * torch.randn(T, N, device=DEV)
    corr = None if mode == "logits" else 0.1 * torch.randn(N, device=DEV)
    if mode == "logits":
        groups, keep = 1, 1
    for renorm in (False, True):
        a = (top, max(1, N - 2), groups, keep, renorm, 1.5, mode)
        _check(ops.moe_route(z, corr, *a), R.moe_route(z, corr, *a), N)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,N,H,mode", [
    (1, 8, 2048, "logits"), (32, 8, 64, "sigmoid"), (17, 64, 2056, "softmax"),
    (512, 3, 4104, "logits"), (3, 9, 8, "softmax")])
def test_choice_with_logits(dtype, T, N, H, mode):
    torch.manual_seed(T + N)
    x = torch.randn(T, H + 8, device=DEV).to(torch.bfloat16)[:, :H]
    gate = torch.randn(N, H, device=DEV).to(dtype) * 3 / H ** 0.5
    top = min(2, N)
    z = (x.double() @ gate.double().T).float()
    a = (top, N, 1, 1, True, 1.0, mode)
    # rows whose choice or weights hang on less than the logits' rounding
    # would have to be left out: there are none at these seeds
    _check(ops.moe_gate_route(x, gate, None, *a),
           R.moe_route(z, None, *a), N)


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,n", [(1, 1, 1), (32, 2, 8), (63, 1, 3),
                                     (43, 6, 64), (129, 2, 200), (5, 8, 1024),
                                     (2731, 3, 8), (8192, 2, 8)])
def test_sort_is_stable(T, top, n):
    torch.manual_seed(T + n)
    topi = torch.randint(0, max(1, n - n // 4), (T, top), device=DEV).int()
    topw = torch.rand(T, top, device=DEV)
    for a, b in zip(ops.moe_plan(topi, topw, n), R.moe_plan(topi, topw, n)):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "logits"])
@pytest.mark.parametrize("N,groups,keep,top,why", [
    (16, 8, 1, 4, "groups"), (130, 10, 1, 20, "groups"), (8, 1, 1, 3, "-inf"),
    (100, 4, 2, 6, "-inf"), (6, 3, 3, 6, "-inf")])
def test_more_choices_than_eligible_outputs(mode, N, groups, keep, top, why):
    """Outputs are taken once each: eligible ones first, then others at
    their own score, as a sort leaves them."""
    torch.manual_seed(N)
    z, corr = torch.randn(5, N, device=DEV), None
    if mode == "logits":
        if why == "groups":
            return                    # this mode has none
        z[:, 1:] = float("-inf")
        groups = keep = 1
    elif why == "-inf":
        corr = torch.full((N,), float("-inf"), device=DEV)
        corr[N // 2:N // 2 + 2] = 0.5
    a = (top, N, groups, keep, False, 1.0, mode)
    gi, gw, _ = ops.moe_route(z, corr, *a)
    wi, ww, _ = R.moe_route(z, corr, *a)
    gi, wi = gi.long(), wi.long()
    assert all(len(set(r)) == top for r in gi.tolist())
    s = {"softmax": torch.softmax(z, -1), "sigmoid": torch.sigmoid(z),
         "logits": torch.softmax(z, -1)}[mode]
    assert torch.allclose(gw, s.gather(1, gi), atol=2e-6)
    sure = 2 if why == "-inf" and mode != "logits" else \
        1 if why == "-inf" else N // groups
    assert torch.equal(gi[:, :sure], wi[:, :sure])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "logits"])
@pytest.mark.parametrize("N,groups,keep", [(8, 1, 1), (70, 1, 1), (64, 8, 2)])
def test_a_nan_is_not_passed_over(mode, N, groups, keep):
    """A router that forms a NaN for one output shows it in the weights."""
    torch.manual_seed(N)
    z = torch.randn(6, N, device=DEV)
    z[torch.arange(6), torch.arange(6) * (N // 6)] = float("nan")
    if mode == "logits":
        groups = keep = 1
    a = (2, N, groups, keep, True, 1.0, mode)
    got, want = ops.moe_route(z, None, *a), R.moe_route(z, None, *a)
    assert torch.isnan(want[1]).any(1).all()
    assert torch.isnan(got[1]).any(1).all()
    assert all(len(set(r)) == 2 for r in got[0].tolist())


@pytest.mark.parametrize("device", [
    "cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("N", [8, 40, 130])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_choice_does_not_hang_on_the_step(device, N, dtype):
    """Two outputs 2^-10 apart: the same experts and weights for a token
    alone, in a short step and in a long one. Logits rounded to bf16 (2^-9)
    would tie."""
    torch.manual_seed(N)
    H = 256
    x = torch.ones(600, H).to(torch.bfloat16)
    x[:, 1] = 2.0 ** -10
    gate = torch.zeros(N, H)
    gate[2, 0], gate[2, 1] = 1.0, -1.0    # 1 - 2^-10
    gate[5, 0] = 1.0                      # 1
    gate[7, 0], gate[7, 1] = 1.0, 1.0     # 1 + 2^-10
    x, gate = x.to(device), gate.to(dtype).to(device)
    w = None
    for T in (1, 32, 512, 600):
        i, topw, _ = ops.moe_gate_route(x[:T], gate, None, 3, N, renorm=True,
                                        mode="logits")
        assert (i.cpu() == torch.tensor([7, 5, 2])).all()
        w = topw[:1].cpu() if w is None else w
        assert torch.allclose(topw.cpu(), w, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("T,N", [(1, 32), (256, 32), (257, 32), (341, 24),
                                 (342, 24), (512, 16), (513, 16), (1, 33)])
def test_choice_on_both_sides_of_the_rule(T, N):
    torch.manual_seed(T)
    x = torch.randn(T, 64, device=DEV).to(torch.bfloat16)
    gate = torch.randn(N, 64, device=DEV).to(torch.bfloat16) / 4
    z = (x.double() @ gate.double().T).float()
    a = (2, N, 1, 1, True, 1.0, "softmax")
    _check(ops.moe_gate_route(x, gate, None, *a),
           R.moe_route(z, None, *a), N)


@pytest.mark.parametrize("device", [
    "cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("n_group,topk_group", [(1, 1), (1, 4), (0, 0),
                                                (1, 0), (4, 4)])
@pytest.mark.parametrize("routing", ["noaux_tc", "sigmoid_groups"])
def test_layers_without_a_group_limit(device, n_group, topk_group, routing):
    """Counts of kept groups mean nothing where there is one group or none."""
    from kaito_amd.engine.config import ModelConfig
    from kaito_amd.models.moe import MoEMLP
    from kaito_amd.parallel.state import init_parallel
    init_parallel(1)
    torch.manual_seed(2)
    m = MoEMLP(ModelConfig(
        name="t", hidden_size=64, num_experts=8, num_experts_per_tok=3,
        moe_intermediate_size=64, moe_routing=routing, n_group=n_group,
        topk_group=topk_group)).requires_grad_(False)
    for p in m.parameters():
        p.normal_(0, 0.2)
    x = torch.randn(9, 64).to(torch.bfloat16)
    s = torch.sigmoid(x.float() @ m.gate.float().T)
    sel = s + m.e_score_correction_bias if routing == "noaux_tc" else s
    want = sel.topk(3, -1)[1]
    got = m.to(device)._choose(x.to(device))[0].cpu()
    assert torch.equal(got.long().sort(-1)[0], want.sort(-1)[0])
    assert torch.isfinite(m(x.to(device)).float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,n", [(300, 8, 256), (2048, 1, 961),
                                     (2049, 1, 961), (700, 3, 960),
                                     (3000, 1, 1024), (513, 4, 1000),
                                     (4096, 8, 65), (257, 1, 2)])
@pytest.mark.parametrize("spread", ["all", "one", "last"])
def test_sort_of_many_experts(T, top, n, spread):
    torch.manual_seed(T)
    topi = {"all": torch.randint(0, n, (T, top)),
            "one": torch.full((T, top), n // 2),
            "last": (n - 1 - torch.arange(T * top) // 64 % n).view(T, top)}
    topi = topi[spread].to(DEV).int()
    topw = torch.rand(T, top, device=DEV)
    for a, b in zip(ops.moe_plan(topi, topw, n), R.moe_plan(topi, topw, n)):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,N,H,mode", [
    (513, 16, 64, "softmax"), (600, 1, 32, "softmax"), (529, 9, 2080, "logits"),
    (257, 32, 2176, "sigmoid"), (4099, 17, 96, "sigmoid")])
def test_choice_of_16_rows(dtype, T, N, H, mode):
    torch.manual_seed(T + N)
    x = torch.randn(T, H + 8, device=DEV).to(torch.bfloat16)[:, :H]
    gate = torch.randn(N, H, device=DEV).to(dtype) * 3 / H ** 0.5
    z = (x.double() @ gate.double().T).float()
    a = (min(2, N), N, 1, 1, True, 1.0, mode)
    _check(ops.moe_gate_route(x, gate, None, *a),
           R.moe_route(z, None, *a), N)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_choice_of_16_rows_not_finite(dtype):
    """Infinities and NaN of rows and router reach the choice as in the
    product of short steps."""
    torch.manual_seed(3)
    x = torch.randn(600, 256, device=DEV).to(torch.bfloat16)
    gate = (torch.randn(8, 256, device=DEV) / 16).to(dtype)
    gate[5, 7] = float("inf")
    x[3, 9], x[4, 9], x[40, 11] = float("inf"), -float("inf"), float("nan")
    a = (3, 8, 1, 1, False, 1.0, "logits")
    long = ops.moe_gate_route(x, gate, None, *a)
    short = ops.moe_gate_route(x[:512], gate, None, *a)
    assert torch.equal(long[0][:512], short[0])
    # weights: logits of unit size, sums of 256 products in another order
    torch.testing.assert_close(long[1][:512], short[1], rtol=1e-5, atol=1e-6,
                               equal_nan=True)


@pytest.mark.gpu
def test_choice_of_16_rows_large_router():
    """f32 weights beyond the largest bf16 whose logits are finite."""
    torch.manual_seed(4)
    x = torch.randn(600, 256, device=DEV).to(torch.bfloat16)
    gate = torch.randn(8, 256, device=DEV) / 16
    x[:, 9] = x[:, 9].clamp(-0.5, 0.5)
    gate[5, 9], gate[2, 9] = torch.finfo(torch.float32).max, -3.4e38
    a = (3, 8, 1, 1, False, 1.0, "logits")
    topi, topw, _ = ops.moe_gate_route(x, gate, None, *a)
    want = R.moe_route((x.double() @ gate.double().T).float(), None, *a)
    assert topw.isfinite().all()
    assert torch.equal(topi, want[0])
    # the products of 256 terms, every rounding at its worst
    size = (x.double().abs() @ gate.double().abs().T).float().gather(
        1, topi.long())
    assert ((topw - want[1]).abs() <= 768 * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("T,N,H,f32,tiles", [
    (600, 8, 2048, False, True), (8192, 16, 2880, False, True),
    (600, 8, 4096, False, True), (600, 16, 4096, False, False),
    (2048, 16, 3072, False, False), (8192, 32, 2048, False, False),
    (257, 32, 2048, True, True), (600, 16, 8192, True, True),
    (512, 32, 4096, True, False), (600, 24, 8192, True, False),
    (1024, 32, 8192, True, True), (8192, 8, 2040, True, False)])
def test_which_steps_choose_by_16_rows(T, N, H, f32, tiles):
    """The sides of the line on which either was measured to be faster."""
    assert ops._gate_long(T, N, H, f32) == tiles


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 5, 16, 17, 32])
@pytest.mark.parametrize("E,H,I,top", [(8, 2048, 2048, 2), (16, 2048, 256, 4),
                                       (4, 512, 192, 1), (6, 2048, 768, 6)])
def test_expert_of_every_token(T, E, H, I, top):
    """An expert of every token in the launches of the chosen ones, some of which
    nobody chose: every row is a linear layer each way (f32 sums of up to 2048
    terms, one rounding to bf16 on the way up). The routed rows keep their bits
    where the launches run on the kernel of before: workgroups that stay, whose
    sums have another order, are for K of 2048."""
    g = torch.Generator(device="cuda").manual_seed(T * E + I)

    def normal(*s):
        return torch.randn(*s, device="cuda", generator=g)
    x = normal(T, H).bfloat16()
    wu, wd = (normal(E, 2 * I, H) * H ** -.5).bfloat16(), \
        (normal(E, H, I) * I ** -.5).bfloat16()
    su, sd = (normal(2 * I, H) * H ** -.5).bfloat16(), \
        (normal(H, I) * I ** -.5).bfloat16()
    topi = torch.stack([torch.randperm(max(1, E - 1), device="cuda")[:top]
                        for _ in range(T)]).int() if top < E else \
        torch.arange(E, device="cuda").int().repeat(T, 1)

    def run(**kw):
        up = {k: kw[k] for k in ("all_w", "all_act") if k in kw}
        act = torch.empty(T * top, I, dtype=torch.bfloat16, device="cuda")
        ops.moe_up_pairs(act, x, wu, topi, E, 0, E, **up)
        y = torch.empty(T * top, H, device="cuda")
        down = dict(all_w=kw["all_d"], all_act=kw["all_act"],
                    all_y=kw["all_y"]) if kw else {}
        ops.moe_down_pairs(y, act, wd, topi, E, 0, E, **down)
        return act, y
    aa = torch.full((T, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    ay = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device="cuda")
    plain = run()
    beside = run(all_w=su, all_d=sd, all_act=aa, all_y=ay)

    def check(got, ref, unit):
        """unit: the result's own rounding; f32 sums that cancel beside it"""
        rms = ref.square().mean().sqrt()
        assert ((got.double() - ref).abs()
                <= unit * ref.abs() + 2.0 ** -12 * rms).all()

    def up(rows, w):
        gu = rows.double() @ w.double().T
        return gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]
    act, y = beside
    for e in range(E):
        mine = (topi == e).flatten().nonzero().flatten()
        if mine.numel():
            check(act[mine], up(x[mine // top], wu[e]), 2.0 ** -8)
            check(y[mine], act[mine].double() @ wd[e].double().T, 2.0 ** -20)
    if H != 2048:
        assert torch.equal(act, plain[0])
        if I != 2048:
            assert torch.equal(y, plain[1])
    check(aa, up(x, su), 2.0 ** -8)
    check(ay, aa.double() @ sd.double().T, 2.0 ** -8)


@pytest.mark.parametrize("E,H,I,top,beside,alone", [
    (8, 2048, 2048, 2, (1, 4, 16, 17, 32), (33,)),
    (4, 2048, 2048, 2, (1, 16, 25, 32), (17, 24)),
    (8, 4096, 4096, 2, (8, 16), (17, 24, 32)),
    (4, 4096, 8192, 1, (2, 16), (17, 32)),
    (16, 5120, 1536, 6, (6, 16), (17, 24, 32)),
    (8, 3584, 2560, 2, (8, 16), (17, 32)), (8, 7168, 2048, 8, (2, 17, 32), ()),
    (6, 2880, 2880, 2, (1, 17, 32), ()), (1, 2048, 2048, 1, (1, 17, 32), ()),
    (4, 2048, 8192, 2, (2, 16), (1,)), (8, 2048, 4096, 2, (1, 32), ())])
def test_which_shared_experts_join(E, H, I, top, beside, alone):
    """The sides of the line on which either was measured to be faster."""
    for T in beside:
        assert ops.moe_shared_pays(T, T * top, E, H, I), T
    for T in alone:
        assert not ops.moe_shared_pays(T, T * top, E, H, I), T


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["softmax", "sigmoid", "logits"])
@pytest.mark.parametrize("N,groups,keep,top", [
    (2, 2, 1, 1), (3, 1, 1, 3), (16, 1, 1, 2), (17, 1, 1, 5), (32, 4, 2, 3),
    (33, 1, 1, 33), (24, 3, 2, 4), (20, 4, 3, 5), (64, 2, 1, 8), (64, 64, 9, 4),
    (40, 5, 2, 8), (48, 3, 1, 16)])
def test_choice_at_the_widths_of_lanes(mode, N, groups, keep, top, monkeypatch):
    """Outputs around the 2 to 64 lanes that a choice looks at, groups of powers of
    two, all at once, and others, ties among them: as in a stable sort."""
    if mode == "logits":
        groups, keep = 1, 1
    torch.manual_seed(N + groups)
    z = torch.randn(19, N, device=DEV)
    z[7] = z[7].round()                       # ties
    z[8] = 0.5
    z[9, N // 2:] = z[9, :N - N // 2].clone()
    a = (top, N, groups, keep, True, 1.0, mode)
    got = ops.moe_route(z, None, *a)
    # the lower index first, which topk does not promise
    monkeypatch.setattr(torch.Tensor, "topk", lambda t, k, d: tuple(
        v[..., :k] for v in t.sort(dim=d, descending=True, stable=True)))
    _check(got, R.moe_route(z, None, *a), N)
