"""Linear layers of prompts on tiles (ops/csrc/tile_linear.hip): rows and columns
that end inside a tile, few K steps, each shape of tiles and several rounds. Sums
of K f32 products, rounded to bf16 once: half a unit of the 8 bits, and where a sum
cancels the f32 rounding of its terms."""
import os
import re
import subprocess

import pytest
import torch

from kaito_amd import ops
from kaito_amd.ops import _build

DEV = "cuda"


def _rand(*shape, std=1.0):
    return (std * torch.randn(*shape, device=DEV)).to(torch.bfloat16)


def _close(out, ref):
    assert torch.isfinite(out).all()
    err = (out.double() - ref).abs()
    rms = ref.square().mean().sqrt()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * rms).all(), err.max()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 64, 64), (127, 192, 128), (257, 320, 192), (300, 2048, 320),
    (1000, 1408, 576), (2050, 2112, 448), (4200, 1600, 256)])
def test_swiglu(M, N, K):
    torch.manual_seed(M)
    x, w = _rand(M, K), _rand(2 * N, K, std=K ** -0.5)
    out = torch.full((M, N), float("nan"), device=DEV).to(torch.bfloat16)
    ops._K.tile_swiglu(out, x, w)
    g, u = (x.double() @ w.double().T).chunk(2, -1)
    _close(out, g * torch.sigmoid(g) * u)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (250, 4160, 448),
                                   (129, 33024, 192), (600, 2112, 320)])
def test_linear(M, N, K):
    torch.manual_seed(M)
    x, w = _rand(M, K), _rand(N, K, std=K ** -0.5)
    out = torch.full((M, N), float("nan"), device=DEV).to(torch.bfloat16)
    ops._K.tile_linear(out, x, w)
    _close(out, x.double() @ w.double().T)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,N2,K,b,b2", [
    (1, 256, 64, 64, True, False), (130, 512, 576, 320, False, True),
    (1000, 3072, 576, 192, True, True), (3001, 768, 1088, 128, False, False),
    (5000, 2048, 2048, 256, False, True)])
@pytest.mark.parametrize("one", [True, False])
def test_pair(M, N, N2, K, b, b2, one):
    torch.manual_seed(M)
    x = _rand(M, K)
    x2 = x if one else _rand(M, K)
    w, w2 = _rand(N, K, std=K ** -0.5), _rand(N2, K, std=K ** -0.5)
    none = torch.empty(0, device=DEV)
    bias, bias2 = _rand(N) if b else none, _rand(N2) if b2 else none
    out, out2 = (torch.full((M, n), float("nan"), device=DEV).to(torch.bfloat16)
                 for n in (N, N2))
    ops._K.tile_pair(out, x, w, bias, out2, x2, w2, bias2)
    _close(out, x.double() @ w.double().T + (bias.double() if b else 0))
    _close(out2, x2.double() @ w2.double().T + (bias2.double() if b2 else 0))


@pytest.mark.gpu
def test_forms_that_tiles_do_not_take():
    """Strided, misaligned and differentiated operands give what they gave."""
    torch.manual_seed(0)
    M, N, K = 1100, 1024, 256
    big, wide = _rand(M, K + 8), _rand(2 * N * K + 8)
    w = wide[:-8].view(2 * N, K)
    forms = [(big[:, 8:], w), (big[:, :K].t().contiguous().t(), w),
             (big[:, :K].contiguous(), wide[4:-4].view(2 * N, K)),
             (big[:, :K].contiguous(), w)]
    for x, v in forms:
        g, u = (x.double() @ v.double().T).chunk(2, -1)
        ref = g * torch.sigmoid(g) * u
        out = ops.linear_swiglu(x, v)
        # gate and up are rounded too where the library makes them
        assert (out.double() - ref).norm() <= 2.0 ** -7 * ref.norm()
        a, b = ops.linear_pair(x, v[:N], x, v[N:])
        assert (a.double() - g).norm() <= 2.0 ** -8 * g.norm()
        assert (b.double() - u).norm() <= 2.0 ** -8 * u.norm()
    x = forms[-1][0].requires_grad_()
    ops.linear_pair(x, w[:N], x, w[N:])[0].sum().backward()
    assert x.grad is not None


@pytest.mark.gpu
def test_rows_without_a_value_stay_among_themselves():
    """A row or a weight row of infinities or NaN, in tiles of finite ones."""
    torch.manual_seed(0)
    M, N, K = 300, 576, 192
    x, w, pair = _rand(M, K), _rand(N, K), _rand(2 * N, K)
    x[5, 7], x[131, 0], x[299] = float("inf"), float("nan"), float("-inf")
    w[64, 3], pair[N + 64, 3] = float("nan"), float("nan")
    rows = torch.ones(M, dtype=torch.bool, device=DEV)
    rows[[5, 131, 299]] = False
    cols = torch.ones(N, dtype=torch.bool, device=DEV)
    cols[64] = False
    out, act = (torch.empty(M, N, device=DEV).to(torch.bfloat16) for _ in "oa")
    ops._K.tile_linear(out, x, w)
    ops._K.tile_swiglu(act, x, pair)
    g, u = (x.double() @ pair.double().T).chunk(2, -1)
    for y, ref in ((out, x.double() @ w.double().T),
                   (act, g * torch.sigmoid(g) * u)):
        _close(y[rows][:, cols], ref[rows][:, cols])
        assert y[131].isnan().all() and y[:, 64].isnan().all()
    assert not out[[5, 299]].isfinite().any()
    # the same rows as two experts'
    off = torch.tensor([0, 131, M], dtype=torch.int32, device=DEV)
    y = torch.empty(M, N, device=DEV)
    ops._K.moe_grouped_down(y, x, w[None].repeat(2, 1, 1), off,
                            torch.empty(0, device=DEV), 0)
    ref = x.double() @ w.double().T
    _close(y[rows][:, cols], ref[rows][:, cols])
    assert y[131].isnan().all() and y[:, 64].isnan().all()


@pytest.mark.gpu
def test_another_stream():
    """What the caller's stream holds is waited for, and no other stream is."""
    torch.manual_seed(0)
    x, w, pair = _rand(3000, 1024), _rand(2112, 1024), _rand(4096, 1024)
    assert ops._uneven_shape(3000, 2112, 1024) and ops._tiled(x, pair)
    want = [ops.linear(x, w), ops.linear_swiglu(x, pair)]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        z = _rand(4096, 4096)
        for _ in range(20):
            z = z @ z * 2 ** -7
        late = torch.empty_like(x).copy_(x)   # behind them
        got = [ops.linear(late, w), ops.linear_swiglu(late, pair)]
    side.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
def test_operands_that_the_kernels_refuse():
    x, w, out = _rand(40, 128), _rand(64, 128), _rand(40, 64)
    wide, none = _rand(40 * 128 + 8), torch.empty(0, device=DEV)
    linear = [
        (out.float(), x, w), (out, x.float(), w), (out, x, w.half()),
        (out, x.cpu(), w), (out[:, ::2], x, w[::2].contiguous()),
        (out, x[:, :64], w[:, :64]), (out, wide[4:-4].view(40, 128), w),
        (out, x[:, :32].contiguous(), w[:, :32].contiguous()),
        (out[:20], x, w), (out, x, w[:32]), (out, x, _rand(64, 192)),
        (_rand(40, 32), x, w[:32].contiguous())]
    for args in linear:
        with pytest.raises(RuntimeError):
            ops._K.tile_linear(*args)
    with pytest.raises(RuntimeError):
        ops._K.tile_swiglu(out, x, w)
    big, big_out = _rand(256, 128), _rand(40, 256)
    pairs = [
        (out, x, w, none, out, x, w, none),           # first not by 256
        (big_out, x, big, _rand(64), out, x, w, none),
        (big_out, x, big, none, out, x, w, torch.zeros(64, device=DEV)),
        (big_out, x, big, none, _rand(41, 64), _rand(41, 128), w, none)]
    for args in pairs:
        with pytest.raises(RuntimeError):
            ops._K.tile_pair(*args)
    ops._K.tile_pair(big_out, x, big, none, out, x, w, none)
    _close(out, x.double() @ w.double().T)


@pytest.mark.parametrize("M,N,K,tiles", [
    (256, 28672, 4096, False), (512, 28672, 4096, True),
    (700, 28672, 4096, False), (8192, 28672, 4096, True),
    (1000, 22016, 4096, False), (1500, 16384, 3072, False),
    (700, 4096, 2048, False), (1000, 4096, 2048, True),
    (1500, 1024, 2048, False), (2048, 1024, 2048, False),
    (2378, 3584, 2048, False), (2635, 3584, 2048, True),
    (4379, 2048, 2048, True)])
def test_which_pairs_take_tiles(M, N, K, tiles):
    """The sides of the line on which either was measured to be faster."""
    assert ops._tiled_shape(M, N, K) == tiles


@pytest.mark.parametrize("M,N,K,tiles", [
    (127, 3648, 2048, False), (128, 3648, 2048, True),
    (8192, 3648, 2048, True), (3000, 7168, 2048, False),
    (6500, 7168, 2048, True), (8192, 2624, 2048, False),
    (168, 832, 2048, False), (154, 2112, 1536, False), (168, 832, 1024, True),
    (241, 3648, 2048, True),
    (1000, 2112, 7168, False)])
def test_which_two_products_take_tiles(M, N, K, tiles):
    assert ops._pair_tiled_shape(M, N, K) == tiles


@pytest.mark.parametrize("M,N,K,tiles", [
    (128, 128256, 4096, False), (129, 128256, 4096, True),
    (256, 128256, 4096, True), (257, 128256, 4096, False),
    (144, 131072, 5120, False), (256, 131072, 5120, True),
    (256, 262144, 2304, False), (200, 32000, 4096, False),
    (160, 100352, 8192, False), (160, 100352, 6144, False),
    (160, 128256, 8192, True), (160, 128256, 7168, True),
    (160, 102400, 7168, False), (256, 102400, 7168, True),
    (144, 151936, 8192, False), (144, 151936, 4096, True)])
def test_which_vocabularies_take_tiles(M, N, K, tiles):
    assert ops._vocabulary_shape(M, N, K) == tiles


@pytest.mark.parametrize("M,N,K,tiles", [
    (8192, 3072, 2048, True), (8192, 2048, 2048, False), (2048, 1024, 512, False),
    (2049, 1024, 512, True), (2049, 1023, 512, False), (8192, 8256, 1024, False),
    (5901, 3072, 4096, True), (8192, 3072, 3136, False),
    (4807, 1024, 1536, False), (2700, 2048, 1536, False),
    (2377, 2496, 2752, False), (6962, 3072, 3072, True),
    (2570, 1024, 256, False), (2570, 1024, 512, True), (2570, 1024, 4096, False),
    (3100, 1024, 4096, True), (4000, 1536, 2048, False), (4000, 1536, 768, True),
    (2826, 2048, 3072, False), (5000, 4096, 128, False)])
def test_which_products_of_prompts_take_tiles(M, N, K, tiles):
    """The sides of the lines on which either was measured to be faster."""
    assert ops._uneven_shape(M, N, K) == tiles


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2049, 1024, 64), (2305, 1088, 192),
                                   (5901, 3072, 128), (8190, 2560, 192),
                                   (2060, 8192, 320), (2305, 1088, 320),
                                   (3000, 2112, 256)])
def test_uneven_products(M, N, K, monkeypatch):
    """Last rounds in quarters and smaller tiles, rows that end inside one."""
    torch.manual_seed(M)
    x, w = _rand(M, K), _rand(N, K, std=K ** -0.5)
    out = torch.full((M, N), float("nan"), device=DEV).to(torch.bfloat16)
    ops._K.tile_linear(out, x, w)
    _close(out, x.double() @ w.double().T)
    assert ops._uneven_shape(M, N, K) == (K >= 256)
    if K >= 256:
        monkeypatch.setattr(torch.nn.functional, "linear", None)
        assert torch.equal(ops.linear(x, w), out)


def _all_close(out, ref, rows=1 << 16):
    for at in range(0, out.size(0), rows):
        _close(out[at:at + rows], ref(slice(at, at + rows)))


# outputs of more than 2 and than 4 GiB, whose last columns end inside a tile
@pytest.mark.gpu
@pytest.mark.parametrize("M", [560000, 746000])
@pytest.mark.parametrize("glu", [False, True])
def test_outputs_of_gigabytes(M, glu):
    torch.manual_seed(M)
    N, K = 2880, 64
    x, w = _rand(M, K), _rand(2 * N if glu else N, K, std=K ** -0.5)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    (ops._K.tile_swiglu if glu else ops._K.tile_linear)(out, x, w)

    def ref(rows):
        y = x[rows].double() @ w.double().T
        if not glu:
            return y
        g, u = y.chunk(2, -1)
        return g * torch.sigmoid(g) * u
    _all_close(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [560000, 746000])
@pytest.mark.parametrize("f32", [False, True])
def test_expert_rows_of_gigabytes(M, f32):
    """Up where rows are bf16, down where they are f32, half as many for as much."""
    torch.manual_seed(M)
    M, N, K = M // (2 if f32 else 1), 2880, 64
    first = M - 130
    off = torch.tensor([0, first, M], dtype=torch.int32, device=DEV)
    none = torch.empty(0, device=DEV)
    x = _rand(M, K)
    w = _rand(2, N if f32 else 2 * N, K, std=K ** -0.5)
    out = torch.full((M, N), float("nan"), device=DEV,
                     dtype=torch.float32 if f32 else torch.bfloat16)
    if f32:
        ops._K.moe_grouped_down(out, x, w, off, none, 0)
    else:
        ids = torch.arange(M, dtype=torch.int32, device=DEV)
        ops._K.moe_grouped_up(out, x, w, ids, off, none, 0, 0, 0.0)

    def ref(rows, e):
        y = x[rows].double() @ w[e].double().T
        if f32:
            return y
        g, u = y.chunk(2, -1)
        return g * torch.sigmoid(g) * u
    _all_close(out[:first], lambda r: ref(slice(r.start, min(r.stop, first)), 0))
    _close(out[first:], ref(slice(first, M), 1))


@pytest.mark.gpu
def test_latent_keys_and_values_of_gigabytes():
    torch.manual_seed(0)
    T, H, D, K = 65600, 128, 128, 64
    c = _rand(T, K)
    wk, wv = _rand(H, D, K, std=K ** -0.5), _rand(H, K, D, std=K ** -0.5)
    assert ops._latent_tiles(T, 2 * H * D, K)
    k, v = ops.latent_kv(c, wk, wv)
    rows = wk.view(H * D, K).double().T
    _all_close(k.reshape(T, H * D), lambda r: c[r].double() @ rows, 1 << 14)
    rows = wv.transpose(0, 1).reshape(K, H * D).double()
    _all_close(v.reshape(T, H * D), lambda r: c[r].double() @ rows, 1 << 14)


@pytest.mark.gpu
def test_rows_too_wide_for_the_tiles():
    """2^22 outputs and more: refused by the kernels, the library's elsewhere."""
    x, w = _rand(1, 64), _rand(1 << 22, 64)
    out = torch.empty(1, 1 << 22, dtype=torch.bfloat16, device=DEV)
    assert not ops._tiles_fit(x, w, 64) and ops._tiles_fit(x, w[:-64], 64)
    with pytest.raises(RuntimeError):
        ops._K.tile_linear(out, x, w)


@pytest.mark.gpu
def test_another_device_is_current(monkeypatch):
    """Prompts whose device is not the current one are torch's, which switches."""
    torch.manual_seed(0)
    x, w, w2 = _rand(2305, 320), _rand(1088, 320), _rand(1024, 320)
    rows, pair = _rand(1000, 2048), _rand(4096, 2048)
    table, where = _rand(300, 64), _rand(70, 64)
    ids = torch.arange(9, device=DEV)
    assert ops._uneven_shape(2305, 1088, 320) and ops._tiles_fit(x, w, 64)
    assert ops._pair_tiled(x, w2, x, w) and ops._tiled(rows, pair)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: x.device.index + 1)
    for op in ("tile_linear", "tile_pair", "tile_swiglu", "embed_positions"):
        monkeypatch.setattr(ops._K, op, None, raising=False)
    F = torch.nn.functional
    assert torch.equal(ops.linear(x, w), F.linear(x, w))
    a, b = ops.linear_pair(x, w2, x, w)
    assert torch.equal(a, F.linear(x, w2)) and torch.equal(b, F.linear(x, w))
    assert torch.equal(ops.linear_swiglu(rows, pair),
                       ops.silu_and_mul(F.linear(rows, pair)))
    assert ops.embed_positions(ids, ids, table, where, 1.0) is None


@pytest.mark.parametrize("group,kernels", [
    ("core", ["tile_linear_kernel"]),
    ("moe", ["moe_grouped_kernel", "latent_kv_kernel"])])
def test_sums_are_the_products_alone(group, kernels, tmp_path):
    """Sums are in accumulation registers by name, unknown to the compiler between
    two statements: in what it built nothing but products writes to one, and nothing
    but the reads of sums looks at one."""
    objdump = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"),
                           "llvm/bin/llvm-objdump")
    lib = _build.so_path(group)
    if not (os.path.exists(objdump) and lib.exists()):
        pytest.skip("nothing built, or no disassembler")
    here = tmp_path / lib.name          # code objects are put beside it
    here.symlink_to(lib)
    subprocess.run([objdump, "--offloading", here.name], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    found = dict.fromkeys(kernels, 0)
    for obj in tmp_path.glob("*amdgcn*"):
        text = subprocess.run([objdump, "-d", obj.name], cwd=tmp_path, check=True,
                              capture_output=True, text=True).stdout
        for body in re.split(r"\n(?=[0-9a-f]+ <)", text):
            name = next((k for k in kernels if k in body.split("\n", 1)[0]), None)
            if name is None:
                continue
            products = 0
            for line in body.split("\n")[1:]:
                code = line.split("//")[0].split(None, 1)
                if len(code) < 2 or not re.search(r"\ba(\d|\[)", code[1]):
                    continue
                assert code[0] in ("v_mfma_f32_16x16x32_bf16",
                                   "v_accvgpr_read_b32"), line
                products += code[0].startswith("v_mfma")
            assert products
            found[name] += 1
    assert all(found.values()), found
