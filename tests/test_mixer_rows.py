"""Row kernels of the stateful mixers at the edges of their tiles: convolution
(16 rows of 16-byte channels), linear recurrent unit (segments of 64 rows, 8
at a time), delta rule (4 tokens at once), post-norm (rows in registers)."""
import pytest
import torch

from kaito_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
I32 = dict(dtype=torch.int32, device=DEV)


def _layout(lens, starts, slots, pad=0):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    ts = [b for b, n in enumerate(lens) for _ in range(n)] + [-1] * pad
    t = lambda v: torch.tensor(v, **I32)
    return t(cu), t(slots), t(starts), t(ts)



@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("C", [8, 1544, 44])
@pytest.mark.parametrize("lens", [[1, 1, 1], [2, 37, 1, 16], [64]])
def test_causal_conv(lens, C, taps, dt):
    torch.manual_seed(C + taps)
    T = sum(lens)
    starts = [5 * (i % 2) for i in range(len(lens))]
    slots = [2 * i + 1 for i in range(len(lens))]
    if len(lens) > 3:
        slots[1] = -1
    x = torch.randn(T, 2 * C, device=DEV).to(dt)[:, C:]
    w, b = torch.randn(C, taps, device=DEV), torch.randn(C, device=DEV)
    state = torch.randn(2 * len(lens), max(taps - 1, 1), C, device=DEV).to(dt)
    want = state.double().clone()
    lay = _layout(lens, starts, slots)
    out = ops.causal_conv_update(x, w, b, state, *lay, act=1)
    at = 0
    for n, st, slot in zip(lens, starts, slots):
        rows = x[at:at + n].double()
        if slot >= 0:
            old = want[slot] if st else torch.zeros_like(want[slot])
            seq = torch.cat([old[:taps - 1], rows])
            acc = b.double() + sum(seq[j:j + n] * w[:, j].double()
                                   for j in range(taps))
            mag = b.double().abs() + sum(
                (seq[j:j + n] * w[:, j].double()).abs() for j in range(taps))
            ref = acc * torch.sigmoid(acc)
            eps = 2.0 ** -8 if dt == torch.bfloat16 else 0.0
            err = (out[at:at + n].double() - ref).abs()
            assert (err <= eps * ref.abs() + 2.0 ** -20 * mag + 1e-30).all()
            if taps > 1:
                want[slot][:taps - 1] = seq[n:]
        at += n
    assert torch.equal(state.double(), want)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("C", [6144, 6152])
@pytest.mark.parametrize("lens", [[2, 301, 1, 200], [16, 17, 15, 456]])
def test_causal_conv_of_long_prompts(lens, C, taps, dt):
    """Sizes at which a workgroup walks 16 rows, chunks that begin anywhere
    in them."""
    test_causal_conv(lens, C, taps, dt)


@pytest.mark.parametrize("lens,pad", [([130], 0), ([64, 64, 1, 70], 0),
                                      ([7, 200, 9], 5), ([513], 0)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_rglru_segments(lens, pad, dt):
    torch.manual_seed(len(lens))
    W, NB, T = 320, 5, sum(lens) + pad
    bw = W // NB
    starts = [3 * (i % 2) for i in range(len(lens))]
    slots = list(range(len(lens), 0, -1))
    u, y = (torch.randn(T, W, device=DEV).to(dt) for _ in range(2))
    gates = torch.randn(NB, T, 2 * bw, device=DEV) * 3
    gates[0, :3, :2], gates[1, 5, 3] = -200.0, 200.0
    rate = torch.rand(W, device=DEV)
    rate[::7] = 1e-6                      # states that hardly decay
    state = torch.randn(len(lens) + 1, W, device=DEV)
    S0 = state.double()
    cu, sl, st, ts = _layout(lens, starts, slots, pad)
    out = ops.rglru_scan(u, gates, y, rate, state, cu, sl, st, ts)
    g = gates.double().permute(1, 0, 2)
    r = torch.sigmoid(g[..., :bw]).reshape(T, W)
    i = torch.sigmoid(g[..., bw:]).reshape(T, W)
    la = -r * rate.double()
    a, drive = la.exp(), (-torch.expm1(2 * la)).sqrt() * i * u.double()
    tol = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -18
    at = 0
    for n, s, slot in zip(lens, starts, slots):
        S = S0[slot] if s else torch.zeros_like(S0[slot])
        for t in range(at, at + n):
            S = a[t] * S + drive[t]
            ref = S * torch.nn.functional.gelu(y[t].double(),
                                               approximate="tanh")
            err = (out[t].double() - ref).abs()
            assert (err <= tol * ref.abs() + 1e-5 * y[t].double().abs()).all()
        assert ((state[slot].double() - S).abs() <= 1e-5 * (1 + S.abs())).all()
        at += n


def _rows(T, bw, blocks):
    W = bw * blocks
    p = torch.randn(T, 2 * W, device=DEV).bfloat16()    # [y | x]
    u = torch.randn(T, W + 8, device=DEV).bfloat16()[:, :W]
    w = torch.randn(blocks, bw, 2 * bw, device=DEV) * 2 / bw ** 0.5
    bias = torch.randn(blocks, 1, 2 * bw, device=DEV)
    rate = torch.rand(W, device=DEV)
    rate[::7] = 1e-6                      # states that hardly decay
    return u, w, bias, p[:, :W], rate


@pytest.mark.parametrize("bw", [64, 128])
@pytest.mark.parametrize("lens,pad", [
    ([130], 0), ([64, 64, 1, 70], 0), ([7, 200, 9], 5), ([31, 0, 513], 0),
    ([33, 1, 95], 31), ([2500], 0), ([40000, 3, 30000], 1)])
def test_rglru_rows_of_prompts(lens, pad, bw):
    """Gates and recurrence together beside one after the other: the same
    products and steps, sums of 64 rows in another order, of states of up to
    some 2^5 here (f32: 2^-24 by the depth of 64 rows and 1100 segments)."""
    torch.manual_seed(len(lens) + bw)
    T = sum(lens) + pad
    u, w, bias, y, rate = _rows(T, bw, 2)
    u[5, 3], u[70, 9] = float("inf"), float("nan")
    state = torch.randn(len(lens) + 1, 2 * bw, device=DEV)
    starts = [3 * (i % 2) for i in range(len(lens))]
    slots = list(range(len(lens), 0, -1))
    if len(lens) == 4:
        slots[1] = -1                     # rows 64 to 127 are of no chunk
    lay = _layout(lens, starts, slots, pad)
    one, two = state.clone(), state.clone()
    out = ops.rglru(u, w, bias, y, rate, one, *lay)
    ref = ops.rglru_scan(u, ops.rglru_gates(u, w, bias), y, rate, two, *lay)
    at = 0
    for n, slot in zip(lens, slots):
        a, b = out[at:at + n].float(), ref[at:at + n].float()
        at += n
        if slot < 0 or n == 0:
            continue
        assert torch.equal(a.isfinite(), b.isfinite())
        tol = 2.0 ** -7 * b.abs() + 1e-4 * y[at - n:at].float().abs()
        assert ((a - b).abs() <= tol)[b.isfinite()].all()
    assert torch.equal(one.isfinite(), two.isfinite())
    ok = two.isfinite()
    assert ((one - two).abs() <= 1e-4 * (1 + two.abs()))[ok].all()


@pytest.mark.parametrize("T", [65536, 65537, 65600, 70000])
def test_rglru_very_long_steps(T):
    """Both sides of the line from which the carries have a launch of their
    own: the same rows in steps on the short side of it. Sums in another
    order, of states that hardly decay: f32's 2^-24 by the depth of the sums
    (64 rows, 1100 segments)."""
    torch.manual_seed(T)
    W = 64
    lens = [T // 3, 5, T - T // 3 - 5]
    u, y = torch.randn(T, W, device=DEV), torch.randn(T, W, device=DEV)
    gates = torch.randn(1, T, 2 * W, device=DEV)
    rate = torch.rand(W, device=DEV)
    rate[::3] = 1e-6
    state = torch.randn(4, W, device=DEV)
    one, parts = state.clone(), state.clone()
    cu, sl, st, ts = _layout(lens, [0, 3, 0], [1, 2, 3], 0)
    out = ops.rglru_scan(u, gates, y, rate, one, cu, sl, st, ts)
    at = 0
    for n, s, slot in zip(lens, [0, 3, 0], [1, 2, 3]):
        cut = slice(at, at + n)
        cu, sl, st, ts = _layout([n], [s], [slot], 0)
        ref = ops.rglru_scan(u[cut], gates[:, cut].contiguous(), y[cut], rate,
                             parts, cu, sl, st, ts)
        err = (out[cut] - ref).abs()
        assert (err <= 2.0 ** -14 * (ref.abs() + y[cut].abs())).all()
        at += n
    assert ((one - parts).abs() <= 2.0 ** -14 * (1 + parts.abs())).all()


def _decode_of_700(rows, H, G, D):
    """q, pages and the table of rows with 700 keys each."""
    pages = -(-700 // 16)
    kc, vc = (torch.randn(rows * pages, G, 16, D, device=DEV).to(torch.bfloat16)
              for _ in range(2))
    table = torch.arange(rows * pages, dtype=torch.int32,
                         device=DEV).view(rows, pages)
    return torch.randn(rows, H, D, device=DEV).to(torch.bfloat16), kc, vc, \
        table


def _check_decode_of_700(q, kc, vc, table, window):
    """Against f64, with scores beyond f32 as infinities; NaN and infinities
    where the reference has them."""
    (rows, H, D), G, n = q.shape, kc.size(1), 700
    out = ops.window_attention(
        q, kc, vc, table, torch.arange(rows, dtype=torch.int32, device=DEV),
        torch.full((rows,), n - 1, device=DEV), D ** -0.5, 0.0, None, None,
        window)
    lo = n - window if window else 0
    for t in (0, rows - 1):
        k, v = (c[table[t].long()].transpose(1, 2).reshape(-1, G, D)[lo:n]
                .double().repeat_interleave(H // G, 1) for c in (kc, vc))
        s = (k * q[t].double()).sum(-1).T * D ** -0.5
        p = torch.where(s < -1e38, -torch.inf, s).softmax(-1)
        ref = (p.T[:, :, None] * v).sum(0)
        got = out[t].double()
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got[ref.isinf()], ref[ref.isinf()])
        fine = ref.isfinite()
        err = (got - ref).abs()[fine]
        assert (err <= 2.0 ** -8 * ref.abs()[fine] + 2e-5).all()
    return out


@pytest.mark.parametrize("H,G,D", [(3, 3, 64), (8, 1, 128), (4, 1, 256)])
@pytest.mark.parametrize("window,rows", [(0, 2), (300, 2), (0, 300)])
def test_window_decode_infinite_scores(H, G, D, window, rows):
    """Keys whose scores are -infinity weigh nothing, also where a wave has no
    others."""
    torch.manual_seed(D + window)
    q, kc, vc, table = _decode_of_700(rows, H, G, D)
    q[0, :, 0] = 2.0 ** 100
    kc[:table.size(1), :, :, 0] = 0
    kc[512 // 16:640 // 16, :, :, 0] = -2.0 ** 60
    assert _check_decode_of_700(q, kc, vc, table, window).isfinite().all()


@pytest.mark.parametrize("H,G,D", [(3, 3, 64), (8, 1, 128), (4, 1, 256)])
@pytest.mark.parametrize("window,rows", [(0, 2), (300, 2), (0, 300)])
def test_window_decode_infinite_values(H, G, D, window, rows):
    """Infinities in the values come out as such, NaN where two of them meet, as
    a sum of weight times value has it. A window behind them, and rows without
    any, do not see them."""
    torch.manual_seed(D + window)
    q, kc, vc, table = _decode_of_700(rows, H, G, D)
    inf = float("inf")
    for key, dim, v in ((100, 1, inf), (500, 2, -inf), (500, 3, inf),
                        (600, 3, -inf), (699, 4, inf), (450, 5, float("nan"))):
        vc[key // 16, :, key % 16, dim] = v
    out = _check_decode_of_700(q, kc, vc, table, window)
    assert out[1:].isfinite().all()


@pytest.mark.parametrize("H,G,D", [(3, 3, 64), (8, 1, 128), (6, 2, 128),
                                   (8, 2, 256)])
@pytest.mark.parametrize("r2", [1e-7, 3e-6, 1e-3])
def test_window_decode_small_penalties(H, G, D, r2):
    """r1 ln(1 + r2 distance) with r2 distance far below 1 and a large r1: the
    logarithm keeps f32's relative precision. Two equal keys are in the window,
    so that the penalty of the older one alone decides its share."""
    n, BS = 1001, 16
    pages = -(-n // BS)
    kc = torch.zeros(pages, G, BS, D, device=DEV, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    vc[(n - 2) // BS, :, (n - 2) % BS] = 1.
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
    q = torch.ones(1, H, D, device=DEV, dtype=torch.bfloat16)
    r1 = torch.linspace(1, 8, H, device=DEV) / r2
    r2 = torch.full((H,), r2, device=DEV)
    out = ops.window_attention(
        q, kc, vc, table, torch.zeros(1, dtype=torch.int32, device=DEV),
        torch.tensor([n - 1], device=DEV), 1.0, 0.0, r1, r2, 2)
    ref = torch.sigmoid(-r1.double() * torch.log1p(r2.double()))
    # penalties up to 8, of three roundings: shares within 8 * 3 * 2^-24; then
    # one rounding to bf16
    err = (out[0, :, 0].double() - ref).abs()
    assert (err <= (2.0 ** -8 + 2e-6) * ref).all(), err / ref
    assert (out == out[..., :1]).all()


@pytest.mark.parametrize("T", [1, 31, 32, 33, 1100])
@pytest.mark.parametrize("B,bw", [(1, 64), (3, 128), (16, 128), (2, 32)])
def test_rglru_gates(T, B, bw):
    """Rows around the 32 of a tile, several tiles per workgroup; sizes of the
    batched product."""
    torch.manual_seed(T + bw)
    big = torch.randn(T, B * bw + 24, device=DEV).to(torch.bfloat16)
    u = big[:, 8:8 + B * bw]
    w = torch.randn(B, bw, 2 * bw, device=DEV)
    b = torch.randn(B, 1, 2 * bw, device=DEV)
    if T > 1:
        u[T // 2, 3], u[0, 5], u[1, 9] = float("inf"), -float("inf"), \
            float("nan")
    ub = u.reshape(T, B, bw).transpose(0, 1).contiguous()
    ref = torch.baddbmm(b.double(), ub.double(), w.double())
    out = ops.rglru_gates(u, w, b)
    fine = ref.isfinite()
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.double()[ref.isinf()], ref[ref.isinf()])
    # an f32 sum of 3 bw products, every rounding at its worst
    size = torch.baddbmm(b.abs(), ub.float().abs(), w.abs()).double()
    err = (out.double() - ref).abs()
    assert (err[fine] <= 3 * bw * 2.0 ** -24 * size[fine]).all()


@pytest.mark.parametrize("z", [-20.0, -1e4, -1e20, -1e36])
def test_rglru_closed_output_gate(z):
    """gelu of a large negative value is 0, however large."""
    T, W = 256, 64
    u, y = torch.randn(T, W, device=DEV), torch.full((T, W), z, device=DEV)
    gates = torch.randn(1, T, 2 * W, device=DEV)
    state = torch.zeros(2, W, device=DEV)
    cu, sl, st, ts = _layout([T], [0], [1], 0)
    out = ops.rglru_scan(u, gates, y, torch.rand(W, device=DEV), state, cu,
                         sl, st, ts)
    assert out.abs().max().item() < 1e-30


@pytest.mark.parametrize("bw", [64, 128])
def test_rglru_gates_large_weights(bw):
    """Weights that are infinite or beyond the largest bf16, with rows that are
    finite, infinite and NaN, as the f32 product has them."""
    torch.manual_seed(bw)
    T, B = 40, 2
    u = (torch.rand(T, B * bw, device=DEV) / 4 + 0.01).to(torch.bfloat16)
    u[3, 7], u[4, 9], u[5, 11] = float("inf"), -float("inf"), float("nan")
    w = torch.randn(B, bw, 2 * bw, device=DEV)
    big = torch.finfo(torch.float32).max
    w[0, 9, 1], w[0, 20, 2], w[1, 5, 3] = float("inf"), -float("inf"), \
        float("nan")
    w[0, 30, 4], w[1, 30, 5], w[1, 31, 6] = big, -big, 3.395e38
    b = torch.randn(B, 1, 2 * bw, device=DEV)
    ub = u.reshape(T, B, bw).transpose(0, 1).contiguous()
    ref = torch.baddbmm(b.double(), ub.double(), w.double())
    out = ops.rglru_gates(u, w, b)
    fine = ref.isfinite()
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.double()[ref.isinf()], ref[ref.isinf()])
    size = torch.baddbmm(b.double().abs(), ub.double().abs(), w.double().abs())
    err = (out.double() - ref).abs()
    # an f32 sum of 3 bw products, every rounding at its worst
    assert (err[fine] <= 3 * bw * 2.0 ** -24 * size[fine]).all()


@pytest.mark.parametrize("D,H,G", [(64, 3, 3), (128, 8, 1), (128, 6, 2),
                                   (256, 8, 2)])
@pytest.mark.parametrize("window,cap,bias,sink,gated",
                         [(100, 20.0, True, False, False),
                          (0, 0.0, True, True, True),
                          (33, 0.0, False, False, False)])
def test_window_decode_rows(D, H, G, window, cap, bias, sink, gated):
    """Single rows on the matrix cores: lengths around pages, tiles and
    splits, a padding row, slots past a row that hold NaN."""
    torch.manual_seed(D + H)
    lens = [1, 15, 16, 17, 32, 33, 100, 1, 131, 1040]
    T, BS = len(lens), 16
    pages = [-(-n // BS) for n in lens]
    kc = torch.randn(sum(pages), G, BS, D, device=DEV).to(torch.bfloat16)
    vc = torch.randn(sum(pages), G, BS, D, device=DEV).to(torch.bfloat16)
    table = torch.zeros(T, max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        table[b, :pages[b]] = torch.arange(at, at + pages[b])
        at += pages[b]
        if n % BS:
            kc[at - 1, :, n % BS:] = float("nan")
            vc[at - 1, :, n % BS:] = float("nan")
    q = 2 * torch.randn(T, H, D, device=DEV).to(torch.bfloat16)
    r1 = torch.rand(H, device=DEV) if bias else None
    r2 = torch.rand(H, device=DEV) if bias else None
    sinks = torch.randn(H, device=DEV) if sink else None
    gate = torch.randn(T, H, device=DEV).to(torch.bfloat16) if gated else None
    seq = torch.arange(T, dtype=torch.int32, device=DEV)
    seq[7] = -1
    pos = torch.tensor(lens, device=DEV) - 1
    out = ops.window_attention(q, kc, vc, table.to(DEV), seq, pos, D ** -0.5,
                               cap, r1, r2, window, sinks=sinks, gate=gate)
    assert (out[7] == 0).all()
    for t, n in enumerate(lens):
        if t == 7:
            continue
        lo = max(0, n - window) if window else 0
        rows = table[t, :pages[t]].long()
        k, v = (c[rows].transpose(1, 2).reshape(-1, G, D)[lo:n].double()
                .repeat_interleave(H // G, 1) for c in (kc, vc))
        s = (k * q[t].double()).sum(-1).T * D ** -0.5          # [H, keys]
        if cap:
            s = cap * torch.tanh(s / cap)
        if bias:
            dist = torch.arange(n - 1 - lo, -1, -1, device=DEV).double()
            s = s - r1.double()[:, None] * torch.log1p(
                r2.double()[:, None] * dist)
        if sink:
            s = torch.cat([s, sinks.double()[:, None]], 1)
        p = s.softmax(-1)[:, :n - lo]
        ref = (p.T[:, :, None] * v).sum(0)
        if gated:
            ref = ref * torch.sigmoid(gate[t].double())[:, None]
        # rounded once to bf16, half a unit of 8 bits; f32 scores and sums are
        # far below
        err = (out[t].double() - ref).abs()
        assert (err <= 2.0 ** -8 * ref.abs() + 2e-5).all(), (t, n)


@pytest.mark.parametrize("lens", [[1, 2, 3, 4, 5, 9], [31], [8, 64]])
@pytest.mark.parametrize("D,V,a0", [(128, 128, -2.0), (64, 20, 3.0),
                                    (256, 8, -6.0), (12, 12, 0.0)])
def test_delta_rule_steps(lens, D, V, a0):
    """Chunks that four tokens do not divide; slow to very fast decay."""
    torch.manual_seed(D)
    T, G, H, n_seq = sum(lens), 2, 4, len(lens)
    r = lambda *s: torch.randn(*s, device=DEV)
    q, k, v, gate = r(T, G, D), r(T, G, D), r(T, H, V), r(T, H, V)
    a, b = r(T, H), r(T, H)
    a_log, dt_bias, nw = r(H) * 0.5 + a0, r(H), r(V)
    starts = [i % 2 for i in range(n_seq)]
    state = r(n_seq, H, D, V)
    S0 = state.double()
    cu, sl, st, _ = _layout(lens, starts, list(range(n_seq)))
    out = ops.gated_delta_rule(q, k, v, gate, a, b, a_log, dt_bias, nw, state,
                               cu, sl, st, 1e-6, 1e-5)
    qd, kd = q.double(), k.double()
    qd = qd / (qd.square().sum(-1, True) + 1e-6).sqrt() / D ** 0.5
    kd = kd / (kd.square().sum(-1, True) + 1e-6).sqrt()
    qd, kd = (x.repeat_interleave(H // G, 1) for x in (qd, kd))
    dec = torch.exp(-a_log.double().exp() * torch.nn.functional.softplus(
        a.double() + dt_bias.double()))
    beta, vd, gd = torch.sigmoid(b.double()), v.double(), gate.double()
    at = 0
    for i, n in enumerate(lens):
        S = S0[i] if starts[i] else torch.zeros_like(S0[i])
        for t in range(at, at + n):
            S = S * dec[t][:, None, None]
            u = beta[t][:, None] * (vd[t] - (S * kd[t][:, :, None]).sum(1))
            S = S + kd[t][:, :, None] * u[:, None]
            o = (S * qd[t][:, :, None]).sum(1)
            rms = (o.square().mean(-1, True) + 1e-5).sqrt()
            ref = o / rms * nw.double() * gd[t] * torch.sigmoid(gd[t])
            err = (out[t].view(H, V).double() - ref).abs()
            # f32 sums of D terms, relative to the row's rms
            lim = 2e-5 * (nw.double() * gd[t]).abs() / rms.clamp(min=1e-2) \
                * S.abs().amax().clamp(min=1) + 1e-6
            assert (err <= lim).all(), (t, (err / lim).max())
        assert ((state[i].double() - S).abs() <= 1e-5 * (1 + S.abs())).all()
        at += n


@pytest.mark.parametrize("H", [8, 520, 2048, 2056, 4096, 8192, 8200, 100])
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_post_norm(H, pair, dt):
    torch.manual_seed(H)
    T = 3
    x32 = torch.randn(T, H, device=DEV)
    y = torch.randn(T, H + 8, device=DEV).to(dt)[:, :H]
    y2 = torch.randn(T, H, device=DEV).to(dt)
    w, wa, wb = (torch.rand(H, device=DEV) + 0.5 for _ in range(3))
    X, Y, Y2 = x32.double(), y.double(), y2.double()
    kw = dict(y2=y2, w_y=wa, w_y2=wb) if pair else {}
    xa = ops.post_norm_residual(x32, y, w, 1e-5, torch.bfloat16, **kw)
    n = lambda t: t / (t.square().mean(-1, True) + 1e-5).sqrt()
    m = (n(Y) * wa.double() + n(Y2) * wb.double()) / 2 if pair else Y
    ref = X + n(m) * w.double()
    assert ((x32.double() - ref).abs() <= 2e-6 * (1 + ref.abs())).all()
    assert torch.equal(xa, x32.to(torch.bfloat16))


@pytest.mark.parametrize("D", [64, 96])
@pytest.mark.parametrize("n", [1, 40])
def test_delta_rule_of_padding_chunks(n, D):
    """Rows of a chunk without a slot leave zeros, whatever the scratch held
    (one token and 40 a chunk: both forms of the recurrence)."""
    G, H, V = 2, 4, 32
    lens, slots = [n, n, n], [1, -1, 0]
    T = sum(lens)
    r = lambda *s: torch.randn(*s, device=DEV).bfloat16()
    f = lambda *s: torch.randn(*s, device=DEV)
    cu, sl, st, _ = _layout(lens, [0, 0, 3], slots)
    args = (r(T, G, D), r(T, G, D), r(T, H, V), r(T, H, V), r(T, H), r(T, H),
            f(H), f(H), f(V), f(2, H, D, V), cu, sl, st, 1e-6, 1e-6)
    for _ in range(2):
        held = [torch.full((T, H, V), float("nan"), device=DEV)
                for _ in range(8)]
        del held
        out = ops.gated_delta_rule(*args)
        assert out.isfinite().all() and not out[n:2 * n].any()
        assert out[:n].any() and out[2 * n:].any()
