"""Linear layers of batched decode steps (ops/csrc/batch_linear.hip): rows around
the tiles, rows of W that end in a tile, K steps that do not divide by the splits.
Sums are f32, results bf16: half a unit of the 8 bits, and where a sum cancels the
f32 rounding of its terms (K up to 2^12 of them, 2^-24 each at most: below 2^-12 of
the typical sum)."""
import pytest
import torch

from kaito_amd import ops

DEV = "cuda"


def _close(out, ref):
    assert out.dtype == torch.bfloat16 and torch.isfinite(out).all()
    err = (out.double() - ref).abs()
    rms = ref.square().mean().sqrt()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * rms).all(), err.max()


def _inputs(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    big = torch.randn(M, K + 16, device=DEV, generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, device=DEV, generator=g).to(torch.bfloat16)
    b = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
    return big[:, 8:8 + K], w, b             # strided rows


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 9, 16, 17, 32, 33, 64, 65, 128, 129, 192,
                               193, 256])
@pytest.mark.parametrize("N,K", [(16, 64), (80, 192), (144, 1152),
                                 (272, 2048)])
def test_plans(M, N, K):
    x, w, b = _inputs(M, N, K)
    ref = x.double() @ w.double().T
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    none = torch.empty(0, device=DEV)
    for cols in (64, 128):
        for splits in sorted({1, min(3, K // 64), min(16, K // 64)}):
            out.fill_(float("nan"))
            ops._K.batch_linear(out, x, w, none, cols, splits, False)
            _close(out, ref)
            ops._K.batch_linear(out, x, w, b, cols, splits, False)
            _close(out, ref + b.double())
        if N % 32 == 0 or N == 144:
            n = N // 2 // 16 * 16
            g, u = x.double() @ w[:n].double().T, x.double() @ w[
                n:2 * n].double().T
            pair = torch.full((M, n), float("nan"), dtype=torch.bfloat16,
                              device=DEV)
            ops._K.batch_linear(pair, x, w[:2 * n], none, cols, 1, True)
            _close(pair, g * torch.sigmoid(g) * u)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,glu", [
    (9, 1024, 10240, False), (256, 2048, 10240, False),
    (17, 3072, 2880, False), (100, 4112, 2880, False),
    (33, 4096, 4096, False), (250, 6144, 7168, False),
    (33, 12288, 2048, True), (256, 12352, 4096, True)])
def test_route(M, N, K, glu):
    x, w, b = _inputs(M, N, K)
    assert ops._batched(x, w, glu) and not ops._skinny(x, w, glu)
    # larger than a test wants in 64 bits on the device: f32 of the library
    ref = (x.float() @ w.float().T).double()
    if glu:
        g, u = ref.chunk(2, -1)
        _close(ops.linear_swiglu(x, w), g * torch.sigmoid(g) * u)
    else:
        _close(ops.linear(x, w), ref)
        _close(ops.linear(x, w, b), ref + b.double())


def _sides(N, K, glu, ahead, behind):
    for M in ahead:
        assert ops._batched_shape(M, N, K, glu), (M, N, K)
    for M in behind:
        assert not ops._batched_shape(M, N, K, glu), (M, N, K)


@pytest.mark.parametrize("N,K,ahead,behind", [
    (4096, 2880, (17, 128), (129, 256)), (28672, 2880, (17, 128), ()),
    (40960, 2880, (17, 32), (64, 96, 128)), (57344, 2880, (32,), (96, 128)),
    (131072, 3840, (32,), (96, 128)), (201088, 2880, (17, 64, 96), (128,)),
    (262208, 5376, (17, 96), (128,)), (8192, 2816, (17, 64), (96, 128)),
    (3072, 3840, (), (17, 64)), (4096, 2816, (), (17, 64, 128)),
    (12288, 3840, (17,), (64, 128)), (16384, 3840, (17, 64), (96, 128)),
    (3072, 4352, (), (17, 64)), (3072, 5376, (17, 128), ()),
    (8192, 5376, (17, 128), ()), (20480, 5376, (17, 64), (96, 128)),
    (16384, 8960, (17, 128), ()), (20480, 8960, (64,), (128,))])
def test_inner_sizes_in_no_multiple_of_512(N, K, ahead, behind):
    """The sides of the line on which either was measured to be faster."""
    _sides(N, K, False, ahead, behind)


@pytest.mark.parametrize("N,K,ahead,behind", [
    (3072, 4096, (), (17, 32, 64)), (3072, 4608, (), (17, 64, 160)),
    (3072, 5120, (17, 64, 128), ()), (4096, 4096, (17, 64), (128, 192)),
    (4096, 4608, (17, 64, 128, 192), ()), (5120, 4096, (17, 64), ()),
    (4096, 8192, (33, 192), (17, 32)), (8192, 4608, (17, 192), ()),
    (16384, 4096, (17, 64), ()), (32768, 4096, (17, 64), (65,)),
    (36864, 4096, (), (17, 64)), (57344, 4096, (), (17, 64)),
    (36864, 4608, (), (17, 64)), (36864, 5120, (17, 32), (33, 64)),
    (49152, 7168, (17, 32), (64,)), (128256, 4096, (), (17, 64)),
    (1024, 10240, (9, 64), (96, 256)), (1024, 12800, (32,), (128,)),
    (2048, 10240, (9, 96, 256), ()), (1024, 14336, (9, 256), ()),
    (1024, 11008, (9, 128), ())])
def test_inner_sizes_in_multiples_of_512(N, K, ahead, behind):
    _sides(N, K, False, ahead, behind)


@pytest.mark.parametrize("N,K,ahead,behind", [
    (20480, 4096, (17, 96, 128), ()), (20480, 5120, (17, 64, 192), (96, 128)),
    (20480, 8192, (64, 192), (128,)), (22016, 5120, (64,), (128,)),
    (16384, 5120, (17, 128, 256), ()), (22528, 5120, (17, 128, 256), ()),
    (28672, 4096, (17, 128, 256), (16,)), (57344, 4096, (64,), (65, 256))])
def test_sizes_of_pairs(N, K, ahead, behind):
    _sides(N, K, True, ahead, behind)


@pytest.mark.gpu
def test_stays_with_the_library():
    x, w, _ = _inputs(64, 4096, 4096)
    assert ops._batched(x, w)
    for a, b in ((x.float(), w.float()), (x.half(), w.half()),
                 (x[:8], w), (x[:, :4088], w[:, :4088].contiguous()),
                 (x, w[:4088]), (x, w.t().contiguous().t())):
        assert not ops._batched(a, b)
    with torch.enable_grad():
        v = w.clone().requires_grad_()
        assert not ops._batched(x, v)
        y = ops.linear(x, v)
        y.sum().backward()
    assert v.grad is not None
    assert not ops._batched(x.repeat(5, 1), w)


@pytest.mark.gpu
def test_replayed_graph():
    x, w, b = _inputs(40, 2048, 10240)
    x = x.contiguous()
    ops.linear(x, w, b)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(x, w, b)
    for i in range(3):
        x.copy_(torch.randn_like(x) + i)
        eager = ops.linear(x, w, b).clone()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(9, 1024, 10240), (16, 4096, 14336),
                                   (33, 2064, 11008), (250, 4096, 14336),
                                   (130, 8192, 12288), (64, 4096, 4096)])
def test_parts_into_the_norm(M, N, K):
    """Bit for bit the sum's launch and the norm's behind it."""
    torch.manual_seed(M + N)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    r = torch.randn(M, N, device="cuda").bfloat16()
    g = torch.randn(N, device="cuda").bfloat16()
    want, total = ops.fused_add_rms_norm(ops.linear(x, w), r.clone(), g, 1e-5)
    rows = ops.linear_parts(x, w)
    assert isinstance(rows, ops.SplitRows)
    out, stream = rows.add_rms_norm(r.clone(), g, 1e-5)
    assert torch.equal(out, want) and torch.equal(stream, total)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(8, 4096, 14336), (257, 4096, 14336),
                                   (250, 4096, 4096)])
def test_no_parts_elsewhere(M, N, K):
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16()
    assert torch.equal(ops.linear_parts(x, w), ops.linear(x, w))


@pytest.mark.parametrize("what", ["rows", "weight"])
def test_parts_that_the_norm_kernel_does_not_take(what):
    """Residual rows or weights at odd addresses, which the norm of whole rows
    takes: the parts are summed first, to the same bits."""
    def at_odd(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype)[1:].view(
            t.shape).copy_(t)
    torch.manual_seed(3)
    part = torch.randn(3, 20, 64)
    r, g = torch.randn(20, 64).bfloat16(), torch.randn(64).bfloat16()
    rows = ((part[0] + part[1]) + part[2]).bfloat16()
    want, total = ops.fused_add_rms_norm(rows, r.clone(), g, 1e-5)
    if what == "rows":
        r = at_odd(r)
    else:
        g = at_odd(g)
    out, stream = ops.SplitRows(part).add_rms_norm(r, g, 1e-5)
    assert torch.equal(out, want) and torch.equal(stream, total)
