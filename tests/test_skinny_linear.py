"""Linear layers of small decode steps (ops/csrc/skinny.h): rows of x and of
the weight, lengths of K around the steps of the loops, 4-bit groups. Sums
are f32 (their error is far below), results bf16: half a unit of the 8 bits,
and one unit where the sum cancels down to 1/16 of its typical size."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.fx.experimental.proxy_tensor import make_fx

from kaito_amd import ops
from kaito_amd.models.quant import quantize_w4
from kaito_amd.ops import torch_ref as R

DEV = "cuda"


def _close(out, ref):
    assert out.dtype == torch.bfloat16 and torch.isfinite(out).all()
    err = (out.double() - ref).abs()
    rms = ref.square().mean().sqrt()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * rms).all(), err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(1, 8), (7, 64), (300, 520), (33, 2048),
                                 (64, 2056), (129, 4608), (6, 14336)])
def test_rows(M, N, K):
    torch.manual_seed(M * N + K)
    big = torch.randn(M, K + 16, device=DEV).to(torch.bfloat16)
    x = big[:, 8:8 + K]                      # strided rows
    w = torch.randn(2 * N, K, device=DEV).to(torch.bfloat16)
    b = torch.randn(2 * N, device=DEV).to(torch.bfloat16)
    ref = x.double() @ w.double().T
    assert ops._skinny(x, w)
    _close(ops.linear(x, w), ref)
    _close(ops.linear(x, w, b), ref + b.double())
    g, u = ref.chunk(2, -1)
    _close(ops.linear_swiglu(x, w), g * torch.sigmoid(g) * u)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [5, 8, 9, 16, 17, 31, 32])
@pytest.mark.parametrize("N,K", [(16, 64), (48, 192), (64, 256), (112, 1792),
                                 (32, 2048), (16, 2368)])
def test_tiles(M, N, K):
    torch.manual_seed(M * N + K)
    x = torch.randn(M, K + 16, device=DEV).to(torch.bfloat16)[:, 8:8 + K]
    w = torch.randn(2 * N, K, device=DEV).to(torch.bfloat16)
    b = torch.randn(2 * N, device=DEV).to(torch.bfloat16)
    ref = x.double() @ w.double().T
    assert ops._skinny(x, w)
    _close(ops.linear(x, w), ref)
    _close(ops.linear(x, w, b), ref + b.double())
    g, u = ref.chunk(2, -1)
    _close(ops.linear_swiglu(x, w), g * torch.sigmoid(g) * u)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [3, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(6144, 2048), (6168, 2048), (6144, 4096),
                                 (7336, 4096), (2560, 2048), (2568, 2048)])
def test_staying_workgroups(M, N, K):
    """Tiles that workgroups share evenly or not, just enough of them."""
    if M > 16 and K == 4096:
        pytest.skip("the library's")
    test_tiles(M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,glu,streamed", [
    (24, 16384, False, True), (32, 8192, False, True),
    (32, 10240, False, False), (25, 16384, False, False),
    (32, 16384, True, True), (32, 24576, False, True)])
def test_which_rows_of_2048_stream(M, N, glu, streamed):
    x = torch.empty(M, 2048, device=DEV, dtype=torch.bfloat16)
    w = torch.empty(N, 2048, device=DEV, dtype=torch.bfloat16)
    assert ops._skinny(x, w, glu) == streamed


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 3, 4])
@pytest.mark.parametrize("N,K", [(4096, 8192), (4128, 8192), (4104, 8192),
                                 (4128, 8200)])
def test_large_weights(M, N, K):
    """3 and 4 rows on both sides of 2^25 weights, in whole tiles or not."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = torch.randn(N, K, device=DEV).to(torch.bfloat16)
    ref = x.double() @ w.double().T
    _close(ops.linear(x, w), ref)
    g, u = ref.chunk(2, -1)
    _close(ops.linear_swiglu(x, w), g * torch.sigmoid(g) * u)


@pytest.mark.gpu
def test_other_forms_stay_with_the_library():
    x = torch.randn(33, 64, device=DEV).to(torch.bfloat16)
    w = torch.randn(32, 64, device=DEV).to(torch.bfloat16)
    for a, b in [(x, w), (x[:2, :60], w[:, :60]), (x[:2, 1:57], w[:, :56].
                 contiguous()), (x[:2].float(), w.float()), (x[:2, None], w),
                 (x[:0], w), (x[:2], w.T.contiguous().T),
                 (x[:5, :56].contiguous(), w[:, :56].contiguous()),
                 (x[:5], w[:24])]:
        assert not ops._skinny(a, b)
        assert torch.equal(ops.linear(a, b),
                           torch.nn.functional.linear(a, b))
    w.requires_grad_(True)
    assert not ops._skinny(x[:2], w)
    assert ops.linear(x[:2], w).requires_grad


@pytest.mark.gpu
def test_calls_that_torch_transforms_stay_with_the_library():
    x = torch.randn(2, 64, device=DEV).to(torch.bfloat16)
    w = torch.randn(32, 64, device=DEV).to(torch.bfloat16)
    with fwAD.dual_level():
        y = ops.linear(fwAD.make_dual(x, 2 * x), w)
        tangent = fwAD.unpack_dual(y).tangent
    assert torch.equal(tangent, torch.nn.functional.linear(2 * x, w))
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    # biases other than one value per row of W
    one = torch.ones(1, device=DEV, dtype=torch.bfloat16)
    assert torch.equal(ops.linear(x, w, one),
                       torch.nn.functional.linear(x, w, one))
    with pytest.raises(RuntimeError):
        ops.linear(x, w, one[:0])


def test_transformed_calls_are_seen():
    seen = []

    def look(t):
        seen.append(ops._transformed())
        return t * 2

    x = torch.randn(2, 3)
    look(x)
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    make_fx(look)(x)
    with fwAD.dual_level():
        look(fwAD.make_dual(x, x))
    look(x)
    assert seen == [False, True, True, True, True, False]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 14, 16])
@pytest.mark.parametrize("N,K", [(8, 512), (24, 4608), (2056, 1536),
                                 (2080, 2048), (40, 3584), (16, 14336)])
def test_w4_tiles(M, N, K):
    """x in LDS: fewer tiles than workgroups and several each, waves without a
    stage, rings of two and three stages, sizes that do not fit."""
    torch.manual_seed(M * N + K)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    qw, s, z = (t.to(DEV) for t in quantize_w4(torch.randn(2 * N, K), 128))
    w = R.w4a16_unpack(qw.cpu(), s.cpu(), z.cpu(), 128).to(DEV)
    ref = x.double() @ w.double().T
    _close(ops.w4a16_gemv(x, qw, s, z, 128), ref)
    out = ops.w4a16_swiglu(x, qw, s, z, 128)
    assert out is not None or M * K > 34000      # LDS
    if out is not None:
        g, u = ref.chunk(2, -1)
        _close(out, g * torch.sigmoid(g) * u)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(4088, 512), (4096, 512), (4112, 1024),
                                 (8208, 4096), (4112, 5120)])
def test_w4_tiles_of_two_workgroups(M, N, K):
    """Around the 512 tiles from which a CU has two workgroups; waves without a
    stage, more rows than x's room for two."""
    torch.manual_seed(M * N + K)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    packed = [t.to(DEV) for t in quantize_w4(torch.randn(2 * N, K), 128)]
    w = R.w4a16_unpack(*(t.cpu() for t in packed), 128).to(DEV)
    ref = x.double() @ w.double().T
    g, u = ref.chunk(2, -1)
    _close(ops.w4a16_gemv(x, *packed, 128), ref)
    out = ops.w4a16_swiglu(x, *packed, 128)
    if out is not None:
        _close(out, g * torch.sigmoid(g) * u)
    # the same rows as a norm's: the kernel's own
    r = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    norm = torch.randn(K, device=DEV).to(torch.bfloat16)
    y, total = ops.fused_add_rms_norm(x.clone(), r.clone(), norm, 1e-5)
    ref = y.double() @ w.double().T
    g, u = ref.chunk(2, -1)
    for glu, want in ((False, ref), (True, g * torch.sigmoid(g) * u)):
        x0, r0 = x.clone(), r.clone()
        took = ops.w4a16_norm_linear(x, r, norm, 1e-5, *packed, 128, glu)
        assert (took is None) == (M > 2 or (not glu and M == 1 and K % 2048 == 0
                                            and 2 * N < 10240))
        if took is not None:
            _close(took[0], want)
            assert torch.equal(took[1], total)
            assert torch.equal(x, x0) and torch.equal(r, r0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,rows,K,alone,pair", [
    (1, 4096, 4096, False, True), (1, 6144, 4096, False, False),
    (1, 28672, 4096, False, True), (1, 28672, 7168, False, True),
    (1, 5120, 2048, False, True), (1, 6656, 2048, False, False),
    (1, 7168, 2048, False, True),
    (2, 28672, 4096, True, True), (2, 4096, 14336, True, True),
    (2, 12288, 2048, False, True), (2, 57344, 1024, False, True),
    (3, 2048, 2048, False, True), (3, 11008, 2048, True, True),
    (4, 1024, 4096, True, True), (5, 4096, 1024, False, True),
    (5, 22016, 512, False, False), (8, 4096, 2048, True, True),
    (16, 4096, 2048, False, True), (16, 6144, 2048, True, True),
    (16, 4096, 4096, False, False), (17, 4096, 512, False, False)])
def test_which_packed_sizes_take_tiles(M, rows, K, alone, pair):
    """The sides of the lines on which either was measured to be faster."""
    assert ops._K.w4a16_in_tiles(M, rows, K, 128, False) == alone
    assert ops._K.w4a16_in_tiles(M, rows, K, 128, True) == pair
    assert not ops._K.w4a16_in_tiles(M, rows, K, 64, True)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,alone", [
    (4096, 1024, True), (5120, 1024, False), (6144, 512, False),
    (7168, 5120, True), (6144, 4096, False), (20480, 2048, False),
    (28672, 2048, True), (10240, 4096, False), (12288, 4096, True),
    (8192, 8192, False), (10240, 8192, True)])
def test_which_packed_products_take_one_row_s_norm(rows, K, alone):
    """The sides of the lines on which either was measured to be faster."""
    assert ops._K.w4a16_norm_in_tiles(1, rows, K, 128, False) == alone
    assert ops._K.w4a16_norm_in_tiles(1, rows, K, 128, True)
    assert ops._K.w4a16_norm_in_tiles(2, rows, K, 128, False)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K,G", [(1, 64, 64), (40, 128, 128),
                                   (33, 192, 192), (100, 4224, 128),
                                   (17, 2112, 64), (8200, 384, 128),
                                   (16390, 128, 128)])
def test_packed_rows(M, N, K, G):
    torch.manual_seed(M + K)
    qw, s, z = (t.to(DEV) for t in quantize_w4(torch.randn(N, K), G))
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    assert ops.w4a16_streams(x, G)
    w = R.w4a16_unpack(qw.cpu(), s.cpu(), z.cpu(), G).to(DEV)
    _close(ops.w4a16_gemv(x, qw, s, z, G), x.double() @ w.double().T)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K,G", [(40, 2048, 128), (40, 1088, 64)])
def test_packed_sums_keep_f32(M, N, K, G):
    """Integers throughout, small ones beside one pair of +-2^20 in every
    group that cancels. Sums of q x stay below 2^24 and are exact in f32 in
    any order; so is the result up to its rounding to bf16. Sums of terms
    larger than q x are not: at 143 times 2^20 the last 4 bits are lost."""
    torch.manual_seed(M + G)
    q = torch.randint(0, 16, (N, K))
    x = torch.randint(-8, 9, (M, K)).float()
    for g in range(0, K, G):
        at = g + 16 * int(torch.randint(0, G // 16, ()))
        i, j = at + int(torch.randint(0, 8, ())), at + int(
            torch.randint(8, 16, ()))
        x[:, i], x[:, j] = 2.0 ** 20, -2.0 ** 20
        q[:, j] = q[:, i]             # cancels
    words = (q.view(N, K // 8, 8) << (4 * torch.arange(8))).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).int()
    s = torch.ones(N, K // G)
    z = torch.full((N, K // G), 8.0)
    xd = x.to(torch.bfloat16).to(DEV)
    out = ops.w4a16_gemv(xd, words.to(DEV), s.to(DEV), z.to(DEV), G).cpu()
    ref = x.double() @ (q.double() - 8).T
    assert torch.equal(out, ref.to(torch.bfloat16))


@pytest.mark.gpu
def test_swiglu_of_every_gate():
    # all bf16 gates, infinities among them, as the first column of W
    g = torch.arange(-32768, 32768, dtype=torch.int16, device=DEV).view(
        torch.bfloat16)
    w = torch.zeros(2, g.numel(), 8, dtype=torch.bfloat16, device=DEV)
    w[0, :, 0], w[1, :, 0] = g, 1.5
    x = torch.zeros(1, 8, dtype=torch.bfloat16, device=DEV)
    x[0, 0] = 1
    out = ops.linear_swiglu(x, w.view(-1, 8))[0].double()
    v = g.double()
    # beyond the f32 range of exp(-v) the weight is 0
    ref = torch.where(v < -88.8, -0.0 * v.abs(), v * torch.sigmoid(v)) * 1.5
    ref = torch.where(v == -float("inf"), float("nan"), ref)
    ref = torch.where(ref > 2.0 ** 128 - 2.0 ** 119, float("inf"), ref)
    assert torch.equal(out.isnan(), ref.isnan())
    both = ~ref.isnan() & (out != ref)
    err = (out - ref).abs()[both]
    # half a unit of bf16's 8 bits (f32's part, exp(88) included, is below 2^-16),
    # and what is left of results below f32's normal range
    bound = (2.0 ** -8 + 2.0 ** -16) * ref.abs()[both] + 2.0 ** -126
    assert (err <= bound).all(), (err / bound).max()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,N2,K", [
    (16, 48, 64), (48, 16, 256), (320, 48, 2048), (5136, 16, 2048),
    (16, 5136, 2048), (6144, 6160, 4096), (112, 80, 1792)])
def test_pairs(M, N, N2, K):
    """Two products in one launch: the bits of two launches where all three run
    on one kernel (workgroups that stay have sums in another order, and large
    weights of 3 and 4 rows take tiles)."""
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    big = torch.randn(M, K + 16, device=DEV, generator=g).to(torch.bfloat16)
    x, x2 = big[:, 8:8 + K], big[:, 16:16 + K]
    w, w2 = (torch.randn(n, K, device=DEV, generator=g).to(torch.bfloat16)
             for n in (N, N2))
    b, b2 = (torch.randn(n, device=DEV, generator=g).to(torch.bfloat16)
             for n in (N, N2))

    def kernel(n, one=True):
        if M <= 4:
            return "tiles" if M > 2 and n * K > 1 << 25 else "rows"
        stay = n // 16 >= (320 if M > 16 else 768) and (
            K == 2048 or (K == 4096 and M <= 16))
        return "staying" if stay and one else "tiles"

    def new():
        return [torch.full((M, n), float("nan"), dtype=torch.bfloat16,
                           device=DEV) for n in (N, N2)]
    for y in (x, x2):
        if M <= 16 or K == 2048 or N * K <= 3072 * 2048:
            got = ops.linear_pair(x, w, y, w2)
            _close(got[0], x.double() @ w.double().T)
            _close(got[1], y.double() @ w2.double().T)
        out, two = new(), new()
        ops._K.skinny_linear_pair(out[0], x, w, b, out[1], y, w2, b2)
        _close(out[0], x.double() @ w.double().T + b.double())
        _close(out[1], y.double() @ w2.double().T + b2.double())
        ops._K.skinny_linear(two[0], x, w, b)
        ops._K.skinny_linear(two[1], y, w2, b2)
        for o, t, n in zip(out, two, (N, N2)):
            if kernel(N + N2, y is x) == kernel(n):
                assert torch.equal(o, t)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K", [(1, 512), (5, 1024), (64, 2048), (9, 2560),
                                 (30, 4096), (33, 5120), (7, 6144), (3, 6656),
                                 (18, 8192)])
def test_norm_in_the_product(M, N, K):
    """Bit for bit the norm's kernel and the product behind it; the inputs
    stay as they are, the sum is a buffer of its own."""
    torch.manual_seed(M * N + K)
    x, r = (torch.randn(M, K, device=DEV).to(torch.bfloat16) for _ in "xr")
    g, b = (torch.randn(n, device=DEV).to(torch.bfloat16) for n in (K, 2 * N))
    w = torch.randn(2 * N, K, device=DEV).to(torch.bfloat16)
    x0, r0 = x.clone(), r.clone()
    assert ops.norm_fits(x, r, g, w)
    normed, total = ops.fused_add_rms_norm(x, r.clone(), g, 1e-5)
    for bias, glu in ((None, False), (b, False), (None, True)):
        out, stream = ops.add_norm_linear(x, r, g, 1e-5, w, bias, glu)
        want = ops.linear_swiglu(normed, w) if glu \
            else ops.linear(normed, w, bias)
        assert torch.equal(out, want) and torch.equal(stream, total)
        assert torch.equal(x, x0) and torch.equal(r, r0)


@pytest.mark.gpu
def test_norm_beside_the_product():
    """What the one launch does not take goes by the two."""
    g = torch.ones(512, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(16, 512, device=DEV).to(torch.bfloat16)
    for x in (torch.randn(3, 512, device=DEV).to(torch.bfloat16),
              torch.randn(2, 512, device=DEV).to(torch.bfloat16)):
        part = x.size(0) == 2
        v, k = (w[:, :504].contiguous(), 504) if part else (w, 512)
        x, n = x[:, :k].contiguous(), g[:k].contiguous()
        r = torch.randn_like(x)
        assert not ops.norm_fits(x, r, n, v)
        normed, total = ops.fused_add_rms_norm(x, r.clone(), n, 1e-5)
        out, stream = ops.add_norm_linear(x, r, n, 1e-5, v)
        assert torch.equal(out, ops.linear(normed, v))
        assert torch.equal(stream, total)


@pytest.mark.gpu
def test_bias_that_is_trained_beside_the_norm():
    """Its gradient is the sum of the product's, as behind the norm's launch."""
    x, r = (torch.randn(2, 512, device=DEV).bfloat16() for _ in "xr")
    g, w = (torch.randn(*s, device=DEV).bfloat16() for s in ((512,), (16, 512)))
    b = torch.randn(16, device=DEV).bfloat16()
    normed, _ = ops.fused_add_rms_norm(x, r.clone(), g, 1e-5)
    want = normed.double() @ w.double().T + b.double()
    b.requires_grad_()
    out, _ = ops.add_norm_linear(x, r.clone(), g, 1e-5, w, b)
    _close(out.detach(), want)
    out.sum().backward()
    assert torch.equal(b.grad, torch.full_like(b, 2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (2, 32, 2560), (2, 4112, 4096),
                                   (1, 5616, 5120), (2, 48, 8192)])
def test_norm_in_the_packed_product(M, N, K):
    """Bit for bit the norm's kernel and the SwiGLU product behind it."""
    torch.manual_seed(N + K)
    x, r = (torch.randn(M, K, device=DEV).to(torch.bfloat16) for _ in "xr")
    g = torch.randn(K, device=DEV).to(torch.bfloat16)
    packed = quantize_w4(torch.randn(N, K, device=DEV), 128)
    x0, r0 = x.clone(), r.clone()
    normed, total = ops.fused_add_rms_norm(x, r.clone(), g, 1e-5)
    want = ops.w4a16_swiglu(normed, *packed, 128)
    took = ops.w4a16_norm_linear(x, r, g, 1e-5, *packed, 128, True)
    if want is None:                  # one row whose product alone is streamed
        assert M == 1
        w = R.w4a16_unpack(*(t.cpu() for t in packed), 128).to(DEV)
        gate, up = (normed.double() @ w.double().T).chunk(2, -1)
        _close(took[0], gate * torch.sigmoid(gate) * up)
    else:
        assert torch.equal(took[0], want)
    assert torch.equal(took[1], total)
    assert torch.equal(x, x0) and torch.equal(r, r0)
    assert ops.w4a16_norm_linear(x.repeat(3, 1), r.repeat(3, 1), g, 1e-5,
                                 *packed, 128, True) is None


@pytest.mark.parametrize("M,N,one,launch", [
    (1, 25152, False, True), (4, 25152, False, True), (5, 25152, False, False),
    (32, 25152, False, False), (32, 25152, True, True), (32, 9216, False, True)])
def test_pairs_that_share_a_launch(M, N, one, launch):
    """The sides of the line on which either was measured to be faster."""
    assert ops._pair_pays(M, N, one) == launch


def test_pairs_that_torch_transforms():
    """Rows without memory of their own are not asked for its address."""
    x, w = torch.randn(5, 3, 32), torch.randn(16, 32)
    for a, b in zip(torch.func.vmap(lambda r: ops.linear_pair(r, w, r, w))(x),
                    (x @ w.t(),) * 2):
        assert torch.allclose(a, b, atol=1e-5)
