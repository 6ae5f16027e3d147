"""hipattn_linear (x . weight^T + bias + residual for the rows of a generation step) through the C ABI against
the oracle's fp64 product, on the projection shapes of the configured models and on awkward ones."""
import numpy as np
import pytest
import torch

from aici_amd import _native
from aici_amd import kernels as K
from aici_amd._lib import HipAttnError
from oracle import refkernels as ref

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def library_choice():
    yield
    for name in ("linear_tiles", "linear_waves", "linear_splits"):
        K.tuning_set(name, 0)


def operands(M, N, Kd, dtype, seed, ldx=None, ldw=None):
    g = torch.Generator().manual_seed(seed)
    xw = torch.randn((M, ldx or Kd), generator=g).to(dtype)
    ww = (torch.randn((N, ldw or Kd), generator=g) * 0.05).to(dtype)
    return xw[:, :Kd], ww[:, :Kd], g


def check(y: torch.Tensor, x, w, bias=None, residual=None):
    """Distance to the fp64 product at most half a unit in the last place of the data type (2^-9 of the value for
    bf16 with its 8 significant bits, 2^-12 for fp16) at each of the two roundings, plus what fp32 accumulation in
    any order can lose: 2^-22 of sum |x||w|."""
    want = ref.linear(x, w, bias)
    eps = 2.0 ** -8 if x.dtype == torch.bfloat16 else 2.0 ** -11
    slack = (x.double().abs() @ w.double().abs().t()) * 2.0 ** -22
    bound = eps * want.abs() + slack
    if residual is not None:
        # the first rounding moves the value by at most eps * |want|; then the sum is rounded once more
        total = want + residual.double()
        bound = bound + eps * total.abs() + eps * bound
        want = total
    err = (y.cpu().double() - want).abs()
    worst = (err - bound).max().item()
    assert worst <= 0.0, f"off by {err.max().item():.3e}, {worst:.3e} past the bound"


SHAPES = [
    # (M, N, K): the projections of Llama-3-8B, Phi-2 (hidden 2560, FFN 10240) and small / ragged ones
    (128, 4096, 4096), (128, 6144, 4096), (128, 4096, 14336), (128, 28672, 4096),
    (120, 2560, 2560), (124, 7680, 2560), (100, 2560, 10240),
    (1, 64, 256), (7, 48, 512), (16, 16, 256), (17, 272, 768), (128, 4112, 1024),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", SHAPES)
def test_matches_the_fp64_product(device, dtype, shape):
    M, N, Kd = shape
    x, w, _ = operands(M, N, Kd, dtype, seed=M + N + Kd)
    y = K.linear(x.to(device), w.to(device))
    assert y.shape == (M, N) and y.dtype == dtype
    check(y, x, w)


@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("splits", [1, 2, 3, 8, 32])
def test_every_launch_shape(device, tiles, waves, splits):
    K.tuning_set("linear_tiles", tiles)
    K.tuning_set("linear_waves", waves)
    K.tuning_set("linear_splits", splits)
    for (M, N, Kd) in [(128, 4096, 4096), (37, 208, 1792), (128, 1040, 256)]:
        x, w, g = operands(M, N, Kd, torch.bfloat16, seed=tiles * 100 + waves * 10 + splits)
        bias = torch.randn((N,), generator=g).bfloat16()
        res = torch.randn((M, N), generator=g).bfloat16()
        y = K.linear(x.to(device), w.to(device), bias=bias.to(device), residual=res.to(device))
        check(y, x, w, bias, res)


def test_identity_and_one_hot_weights_are_exact(device):
    g = torch.Generator().manual_seed(5)
    x = torch.randn((128, 512), generator=g).bfloat16()
    for splits in (1, 2):
        K.tuning_set("linear_splits", splits)
        y = K.linear(x.to(device), torch.eye(512).bfloat16().to(device))
        assert torch.equal(y.cpu(), x)
        pick = torch.zeros((16, 512))
        cols = torch.randperm(512, generator=g)[:16]
        pick[torch.arange(16), cols] = 1.0
        y = K.linear(x.to(device), pick.bfloat16().to(device))
        assert torch.equal(y.cpu(), x[:, cols])


def test_residual_is_a_second_rounding_and_bias_is_not(device):
    x, w, g = operands(128, 4096, 4096, torch.bfloat16, seed=9)
    res = torch.randn((128, 4096), generator=g).bfloat16()
    bias = torch.randn((4096,), generator=g).bfloat16()
    xd, wd = x.to(device), w.to(device)
    plain = K.linear(xd, wd)
    with_res = K.linear(xd, wd, residual=res.to(device))
    # exactly the separate addition of llama.rs:166: T(T(x . W^T) + residual)
    assert torch.equal(with_res.cpu(), (plain.cpu().float() + res.float()).bfloat16())
    # the bias goes in before the only rounding: closer to the fp64 value than a rounded product plus bias
    check(K.linear(xd, wd, bias=bias.to(device)), x, w, bias)
    both = K.linear(xd, wd, bias=bias.to(device), residual=res.to(device))
    with_bias = K.linear(xd, wd, bias=bias.to(device))
    assert torch.equal(both.cpu(), (with_bias.cpu().float() + res.float()).bfloat16())


def test_row_strides_of_every_operand(device):
    M, N, Kd = 96, 1024, 768
    x, w, g = operands(M, N, Kd, torch.float16, seed=21, ldx=3 * Kd, ldw=Kd + 64)
    assert x.stride(0) == 3 * Kd and w.stride(0) == Kd + 64
    wide_res = torch.randn((M, 2 * N), generator=g).half()
    res = wide_res[:, N:]
    xd = torch.randn((M, 3 * Kd), generator=g).half().to(device)
    xd[:, :Kd] = x.to(device)
    wd = torch.zeros((N, Kd + 64), dtype=torch.float16, device=device)
    wd[:, :Kd] = w.to(device)
    out_wide = torch.full((M, N + 8), 7.0, dtype=torch.float16, device=device)
    K.linear(xd[:, :Kd], wd[:, :Kd], residual=wide_res.to(device)[:, N:], out=out_wide[:, :N])
    check(out_wide[:, :N], x, w, residual=res)
    assert torch.all(out_wide[:, N:] == 7.0)  # nothing written past a row's end


@pytest.mark.parametrize("M,N,ldx,ldw", [(1, 64, 1 << 30, None), (2, 1024, 1 << 28, None), (17, 16384, (1 << 28) + 64, None),
                                         (5, 16, None, 1 << 28), (128, 48, 640, (1 << 28) + 8)])
def test_rows_further_apart_than_32_bits_of_bytes(device, M, N, ldx, ldw):
    """One position per sequence of a long activation; a slice of an enormous weight."""
    Kd = 512
    x, w, g = operands(M, N, Kd, torch.bfloat16, seed=M)

    def spread(t, ld):
        if ld is None:
            return t.to(device)
        far = torch.empty(((t.size(0) - 1) * ld + t.size(1),), dtype=t.dtype, device=device).as_strided(t.shape, (ld, 1))
        return far.copy_(t)
    xd, wd = x.to(device), w.to(device)
    xf, wf = spread(x, ldx), spread(w, ldw)
    assert torch.equal(K.linear(xf, wf), K.linear(xd, wd))
    if N % 32 == 0:
        assert torch.equal(K.linear_silu_and_mul(xf, wf), K.linear_silu_and_mul(xd, wd))
    if N <= 8192:
        nw = torch.ones((N,), dtype=torch.bfloat16, device=device)
        for got, want in zip(K.linear_rms_norm(xf, wf, nw, 1e-5), K.linear_rms_norm(xd, wd, nw, 1e-5)):
            assert torch.equal(got, want)


def test_same_bits_on_every_run_and_rows_do_not_mix(device):
    x, w, _ = operands(128, 4096, 14336, torch.bfloat16, seed=33)
    xd, wd = x.to(device), w.to(device)
    first = K.linear(xd, wd)
    for _ in range(3):
        assert torch.equal(K.linear(xd, wd), first)
    # a row's result does not depend on how many other rows come along
    for m in (1, 5, 64):
        assert torch.equal(K.linear(xd[:m].contiguous(), wd), first[:m])


def test_workspace_from_the_caller(device):
    x, w, _ = operands(128, 4096, 4096, torch.bfloat16, seed=41)
    xd, wd = x.to(device), w.to(device)
    need = K.linear_workspace_size(xd, wd)
    assert need > 0
    ws = torch.empty((need,), dtype=torch.uint8, device=device)
    assert torch.equal(K.linear(xd, wd, workspace=ws), K.linear(xd, wd))
    with pytest.raises(HipAttnError, match="workspace has"):
        K.linear(xd, wd, workspace=ws[: need - 256])
    K.tuning_set("linear_splits", 1)
    assert K.linear_workspace_size(xd, wd) == 0


@pytest.mark.parametrize("M", [1, 16, 17, 128])
@pytest.mark.parametrize("N", [512, 4096, 16384])  # the last: k is not cut
def test_output_over_the_input(device, M, N):
    """out = x's own memory, shifted against it, and between its rows."""
    Kd = 512
    x, w, g = operands(M, N, Kd, torch.bfloat16, seed=M + N)
    wd = w.to(device)
    want = K.linear(x.to(device), wd)
    nw = torch.ones((N,), dtype=torch.bfloat16, device=device)
    want_n = torch.empty_like(want)
    if N <= 8192:
        K.rms_norm(want_n, want, nw, 1e-5)
    for at, ld in [(0, N), (64, N + 64), (Kd, N + Kd)]:  # the last: out's columns behind x's, in the same rows
        def buffer():
            buf = torch.zeros((M * ld + 64 + N,), dtype=torch.bfloat16, device=device)
            xv = buf.as_strided((M, Kd), (ld, 1))
            xv.copy_(x)
            return xv, buf.as_strided((M, N), (ld, 1), at)
        xv, out = buffer()
        assert torch.equal(K.linear(xv, wd, out=out), want)
        if at == Kd:
            assert torch.equal(xv.cpu(), x)
        if N <= 8192:
            xv, out = buffer()
            normed = torch.empty_like(want)
            _native.linear_rms_norm(out, normed, xv, wd, None, None, nw, 1e-5, None)
            assert torch.equal(normed, want_n)
            assert torch.equal(out, want)
        xv, out = buffer()
        half = out[:, : N // 2]
        _native.linear_silu_and_mul(half, xv, wd, None)
        assert torch.equal(half, K.linear_silu_and_mul(x.to(device), wd))


def test_workspace_sized_with_one_row_serves_every_batch(device):
    x, w, _ = operands(128, 4096, 4096, torch.bfloat16, seed=43)
    xd, wd = x.to(device), w.to(device)
    nw = torch.ones((4096,), dtype=torch.bfloat16, device=device)
    ws = torch.empty((K.linear_workspace_size(xd[:1], wd),), dtype=torch.uint8, device=device)
    ws_norm = torch.empty((K.linear_rms_norm_workspace_size(xd[:1], wd),), dtype=torch.uint8, device=device)
    for m in (1, 16, 17, 128):
        want, want_n = K.linear_rms_norm(xd[:m], wd, nw, 1e-5)
        assert torch.equal(K.linear(xd[:m], wd, workspace=ws), want)
        out, normed = K.linear_rms_norm(xd[:m], wd, nw, 1e-5, workspace=ws_norm)
        assert torch.equal(out, want) and torch.equal(normed, want_n)


@pytest.mark.parametrize("M", [1, 2, 16, 17])
@pytest.mark.parametrize("wide", ["out", "norm_out", "both"])
def test_linear_rms_norm_into_rows_that_lie_apart(device, M, wide):
    N, Kd = 1024, 4096
    x, w, g = operands(M, N, Kd, torch.float16, seed=M)
    xd, wd = x.to(device), w.to(device)
    nw = (1.0 + 0.1 * torch.randn((N,), generator=g)).half().to(device)
    res = torch.randn((M, 2 * N), generator=g).half().to(device)[:, N:]
    want, want_n = K.linear_rms_norm(xd, wd, nw, 1e-5, residual=res)
    bufs = [torch.full((M, N + 8 * (wide in (name, "both"))), 7.0, dtype=torch.float16, device=device) for name in ("out", "norm_out")]
    ws = torch.empty((K.linear_rms_norm_workspace_size(xd, wd),), dtype=torch.uint8, device=device)
    for workspace in (None, ws):
        _native.linear_rms_norm(bufs[0][:, :N], bufs[1][:, :N], xd, wd, None, res, nw, 1e-5, workspace)
        assert torch.equal(bufs[0][:, :N], want) and torch.equal(bufs[1][:, :N], want_n)
        assert torch.all(bufs[0][:, N:] == 7.0) and torch.all(bufs[1][:, N:] == 7.0)


@pytest.mark.parametrize("splits", [0, 1, 3, 8])
def test_linear_rms_norm_gives_the_bits_of_the_two_calls(device, splits):
    K.tuning_set("linear_splits", splits)
    for (M, N, Kd, dtype, with_bias) in [(128, 4096, 4096, torch.bfloat16, False), (128, 4096, 14336, torch.bfloat16, False),
                                         (37, 2560, 2560, torch.float16, True), (5, 64, 256, torch.bfloat16, True),
                                         (128, 8192, 512, torch.bfloat16, False)]:
        x, w, g = operands(M, N, Kd, dtype, seed=N + Kd + splits)
        res = torch.randn((M, N), generator=g).to(dtype).to(device)
        bias = torch.randn((N,), generator=g).to(dtype).to(device) if with_bias else None
        nw = (1.0 + 0.1 * torch.randn((N,), generator=g)).to(dtype).to(device)
        xd, wd = x.to(device), w.to(device)
        out, normed = K.linear_rms_norm(xd, wd, nw, 1e-5, bias=bias, residual=res)
        want = K.linear(xd, wd, bias=bias, residual=res)
        assert torch.equal(out, want)
        want_n = torch.empty_like(want)
        K.rms_norm(want_n, want, nw, 1e-5)
        assert torch.equal(normed, want_n)
        # and the norm is the oracle's, from the rounded rows
        o = ref.rms_norm(out.cpu(), nw.cpu(), 1e-5)
        assert (normed.cpu().float() - o.float()).abs().max().item() <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) * max(1.0, o.float().abs().max().item())
    # without a residual, from the caller's workspace, and what is refused
    x, w, g = operands(64, 1024, 768, torch.bfloat16, seed=77)
    nw = torch.ones((1024,), dtype=torch.bfloat16, device=device)
    xd, wd = x.to(device), w.to(device)
    ws = torch.empty((K.linear_rms_norm_workspace_size(xd, wd),), dtype=torch.uint8, device=device)
    assert ws.numel() > 0
    out, normed = K.linear_rms_norm(xd, wd, nw, 1e-6, workspace=ws)
    assert torch.equal(out, K.linear(xd, wd))
    with pytest.raises(HipAttnError, match="at most 8192"):
        K.linear_rms_norm(torch.zeros((8, 256), dtype=torch.bfloat16, device=device),
                          torch.zeros((8208, 256), dtype=torch.bfloat16, device=device),
                          torch.ones((8208,), dtype=torch.bfloat16, device=device), 1e-5)
    with pytest.raises(HipAttnError, match="norm_weight must be"):
        K.linear_rms_norm(xd, wd, nw[:512], 1e-5)


def test_refusals(device):
    def t(*shape, dtype=torch.bfloat16):
        return torch.zeros(shape, dtype=dtype, device=device)
    with pytest.raises(HipAttnError, match="at most 128"):
        K.linear(t(129, 256), t(64, 256))
    with pytest.raises(HipAttnError, match="multiple of 256"):
        K.linear(t(8, 320), t(64, 320))
    with pytest.raises(HipAttnError, match="multiple of 16"):
        K.linear(t(8, 256), t(40, 256))
    with pytest.raises(HipAttnError, match="weight is f16"):
        K.linear(t(8, 256), t(64, 256, dtype=torch.float16))
    with pytest.raises(HipAttnError, match="f16 or bf16"):
        K.linear(t(8, 256, dtype=torch.float32), t(64, 256, dtype=torch.float32))
    with pytest.raises(HipAttnError, match="columns"):
        K.linear(t(8, 256), t(64, 512))
    with pytest.raises(HipAttnError, match="out is"):
        K.linear(t(8, 256), t(64, 256), out=t(8, 32))
    with pytest.raises(HipAttnError, match="residual must be"):
        K.linear(t(8, 256), t(64, 256), residual=t(8, 32))
    with pytest.raises(HipAttnError, match="bias must be"):
        K.linear(t(8, 256), t(64, 256), bias=t(32))
    assert not K.linear_takes(t(129, 256), t(64, 256)) and not K.linear_takes(t(8, 320), t(64, 320))
    assert K.linear_takes(t(8, 256), t(64, 256))
    assert K.linear(t(0, 256), t(64, 256)).shape == (0, 64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,kd", [(16, 256), (2560, 2560), (4096, 1024), (1376, 4352), (14336, 512), (8208, 256)])
def test_linear_silu_and_mul_gives_the_bits_of_the_two_calls(device, n, kd, dtype):
    """Every kernel of the layer (16 rows of x and fewer; up to 32, 64, 96, 128) at its edges, weights whose inner size is
    cut into one to eight ranges, one with a last range that is shorter, and rows that do not fill a workgroup."""
    x, w, _ = operands(128, 2 * n, kd, dtype, seed=n + kd)
    xd, wd = x.to(device), w.to(device)
    for m in (1, 15, 16, 17, 32, 33, 64, 65, 96, 97, 128):
        both = K.linear(xd[:m], wd)
        want = torch.empty((m, n), dtype=dtype, device=device)
        K.silu_and_mul(want, both)
        assert torch.equal(K.linear_silu_and_mul(xd[:m], wd), want), m
        if m == 17:
            check(both, x[:m], w)
        # a row's bits do not depend on the kernel its company selects
        assert torch.equal(both[:1], K.linear(xd[:1], wd)), m
    for waves in (4, 8):
        K.tuning_set("linear_waves", waves)
        for splits in (1, 3):
            K.tuning_set("linear_splits", splits)
            both = K.linear(xd[:50], wd)
            want = torch.empty((50, n), dtype=dtype, device=device)
            K.silu_and_mul(want, both)
            assert torch.equal(K.linear_silu_and_mul(xd[:50], wd), want)


@pytest.mark.parametrize("m", [1, 16, 33, 128])
def test_vocabulary_rows(device, m):
    """Weights of 65536 rows and more: a workgroup of 512 rows, the last one partly empty."""
    x, w, _ = operands(m, 65536 + 80, 256, torch.bfloat16, seed=m)
    y = K.linear(x.to(device), w.to(device))
    check(y, x, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Kd,N,M", [(256, 32, 1), (768, 1056, 4), (4096, 6144, 1), (4096, 4096, 2), (4096, 28672, 3), (2560, 2560, 4),
                                   (8192, 96, 1), (5120, 480, 3), (14336 // 2, 64, 1)])
def test_rms_norm_linear_gives_the_bits_of_the_two_calls(device, dtype, Kd, N, M):
    """The norm inside the projection: the bits of rms_norm and linear (or linear_silu_and_mul) one after the other, from rows
    that lie apart as well, for one range of k and several, rows and weights that end inside a 1 KB piece."""
    g = torch.Generator().manual_seed(Kd + N + M)
    wide = (torch.randn((M, Kd + 24), generator=g) * torch.linspace(0.01, 30, M)[:, None]).to(dtype).to(device)
    x = wide[:, 8:Kd + 8]
    weight = (torch.randn((N, Kd), generator=g) / Kd ** 0.5).to(dtype).to(device)
    norm = (1 + 0.2 * torch.randn((Kd,), generator=g)).to(dtype).to(device)
    h = torch.empty((M, Kd), dtype=dtype, device=device)
    K.rms_norm(h, x.contiguous(), norm, 1e-5)
    assert K.rms_norm_linear_takes(x, norm, weight)
    before = wide.clone()
    for _ in range(2):
        assert torch.equal(K.rms_norm_linear(x, norm, 1e-5, weight), K.linear(h, weight))
        assert torch.equal(K.rms_norm_linear(x, norm, 1e-5, weight, silu_and_mul=True), K.linear_silu_and_mul(h, weight))
    assert torch.equal(wide, before)


def test_rms_norm_linear_refusals(device):
    x = torch.zeros((5, 4096), dtype=torch.bfloat16, device=device)
    w = torch.zeros((64, 4096), dtype=torch.bfloat16, device=device)
    norm = torch.ones((4096,), dtype=torch.bfloat16, device=device)
    assert not K.rms_norm_linear_takes(x, norm, w)
    assert not K.rms_norm_linear_takes(x[:4], torch.ones((4097,), dtype=torch.bfloat16, device=device)[1:], w)
    with pytest.raises(HipAttnError, match="at most 4 rows"):
        K.rms_norm_linear(x, norm, 1e-5, w)
    with pytest.raises(HipAttnError, match="at most 4 rows"):  # 3 rows of 8192: more than 40 KB with the norm's weight
        K.rms_norm_linear(torch.zeros((3, 8192), dtype=torch.bfloat16, device=device), torch.ones(8192, dtype=torch.bfloat16,
                                device=device), 1e-5, torch.zeros((64, 8192), dtype=torch.bfloat16, device=device))
    with pytest.raises(HipAttnError, match="norm_weight must be 4096"):
        K.rms_norm_linear(x[:2], norm[:2048], 1e-5, w)
    square = torch.zeros((4096, 4096), dtype=torch.bfloat16, device=device)
    with pytest.raises(HipAttnError, match="over x"):
        _native.rms_norm_linear(x[:2], x[:2], norm, 1e-5, square, False)


@pytest.mark.parametrize("dtype,index", [(torch.bfloat16, torch.int64), (torch.float16, torch.int32)])
@pytest.mark.parametrize("heads,Kd", [((32, 8, 128), 4096), ((3, 1, 80), 512), ((5, 5, 64), 1024), ((2, 1, 256), 256), ((1, 3, 48), 2560)])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 16, 17, 33, 128])
def test_qkv_linear_gives_the_bits_of_the_calls(device, dtype, index, heads, Kd, M):
    """With and without the norm in front, for tokens in and out of the rotary table and of the cache, blocks of 8, 16 and 32 tokens."""
    Hq, Hkv, d = heads
    g = torch.Generator().manual_seed(M + Kd)
    x = torch.randn((M, Kd), generator=g).to(dtype).to(device)
    norm = (1 + 0.2 * torch.randn((Kd,), generator=g)).to(dtype).to(device)
    weight = (torch.randn(((Hq + 2 * Hkv) * d, Kd), generator=g) / Kd ** 0.5).to(dtype).to(device)
    table = torch.randn((300, d), generator=g).to(dtype).to(device)
    h = torch.empty_like(x)
    K.rms_norm(h, x, norm, 1e-5)
    for bs in (8, 16, 32):
        blocks = 5 + M // bs
        kc = torch.randn((blocks, Hkv, d // 8, bs, 8), generator=g).to(dtype).to(device)
        vc = torch.randn((blocks, Hkv, d, bs), generator=g).to(dtype).to(device)
        pos = torch.randint(0, 300, (M,), generator=g)
        slots = torch.randperm(blocks * bs, generator=g)[:M]
        if M > 4:
            pos[2], pos[3] = 300, -1
            slots[0], slots[1] = -1, blocks * bs
        pos, slots = pos.to(index).to(device), slots.to(index).to(device)
        assert K.qkv_linear_takes(x, weight, table, kc, vc)
        want, wkc, wvc = K.linear(h, weight), kc.clone(), vc.clone()
        q, k, v = want.split([Hq * d, Hkv * d, Hkv * d], dim=1)
        K.rotary_embedding_and_cache(pos, q, k, v.view(M, Hkv, d), d, table, True, wkc, wvc, slots)
        for rows, nw in ((h, None), (x, norm)):
            if nw is not None and not K.rms_norm_linear_takes(x, norm, weight):
                continue
            got_k, got_v = kc.clone(), vc.clone()
            got = K.qkv_linear(rows, nw, 1e-5, weight, pos, table, got_k, got_v, slots)
            assert torch.equal(got, want) and torch.equal(got_k, wkc) and torch.equal(got_v, wvc)


def test_qkv_linear_refusals(device):
    z = lambda *s: torch.zeros(s, dtype=torch.bfloat16, device=device)
    x, w, table, kc, vc = z(4, 256), z(6 * 64, 256), z(32, 64), z(2, 1, 8, 16, 8), z(2, 1, 64, 16)
    at = torch.zeros((4,), dtype=torch.int64, device=device)
    for bad, msg in (((z(17, 256), z(256 * 64, 256), table, kc, vc), "more than 16 rows"), ((x, z(2 * 64, 256), table, kc, vc), "query heads"),
                     ((x, w, z(32, 32), kc, vc), "heads of 64"), ((x, w, table.half(), kc, vc), "must be")):
        assert not K.qkv_linear_takes(*bad)
        idx = torch.zeros((bad[0].size(0),), dtype=torch.int64, device=device)
        with pytest.raises(HipAttnError, match=msg):
            K.qkv_linear(bad[0], None, 0.0, bad[1], idx, bad[2], bad[3], bad[4], idx)
    with pytest.raises(HipAttnError, match="3 positions"):
        K.qkv_linear(x, None, 0.0, w, at[:3], table, kc, vc, at)


def test_operands_off_16_byte_boundaries_are_not_taken(device):
    """Whether a call is accepted is answered for rows, weights and norm weights that start anywhere: what the answer takes runs, what it does
    not take is what the call refuses."""
    def at(offset, *shape):
        n = int(np.prod(shape))
        return torch.zeros((n + 8,), dtype=torch.bfloat16, device=device)[offset:offset + n].view(shape)

    table, kc, vc = at(0, 32, 64), at(0, 2, 1, 8, 16, 8), at(0, 2, 1, 64, 16)
    index = torch.zeros((2,), dtype=torch.int64, device=device)
    for ox, ow, on in ((0, 0, 0), (1, 0, 0), (4, 0, 0), (0, 1, 0), (0, 4, 0), (0, 0, 4)):
        x, w, norm = at(ox, 2, 256), at(ow, 384, 256), at(on, 256)
        assert K.linear_takes(x, w) == (ox == ow == 0)
        assert K.rms_norm_linear_takes(x, norm, w) == (ox == ow == on == 0)
        assert K.qkv_linear_takes(x, w, table, kc, vc) == (ox == ow == 0)
        for taken, call in ((ox == ow == 0, lambda: K.linear(x, w)), (ox == ow == on == 0, lambda: K.rms_norm_linear(x, norm, 1e-5, w)),
                            (ox == ow == 0, lambda: K.qkv_linear(x, None, 0.0, w, index, table, kc, vc, index))):
            if taken:
                call()
            else:
                with pytest.raises(HipAttnError, match="16-byte"):
                    call()
    x, w, norm = at(0, 2, 256), at(0, 384, 256), at(0, 256)
    assert not K.rms_norm_linear_takes(x, norm.half(), w) and not K.rms_norm_linear_takes(x, norm[:128], w)
    assert not K.add_rms_norm_takes(x, x.half(), norm) and not K.add_rms_norm_takes(x, x.clone(), norm.float())


# Weights whose ranges of k begin inside: 2, 4 and 1 ranges, halves of 33, 32, 65 and 64 groups of rows, ranges of 25 stages; and one that is left.
TURNED = [(8448, 2048), (8192, 6400), (16640, 2048), (16384, 6400), (16400, 2048)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,Kd", TURNED)
def test_ranges_that_begin_inside_give_a_row_the_same_bits_in_every_kernel(device, dtype, N, Kd):
    x, w, g = operands(128, N, Kd, dtype, seed=N + Kd)
    xd, wd = x.to(device), w.to(device)
    whole = K.linear(xd, wd)
    check(whole[:40], x[:40], w)
    norm = (1 + 0.2 * torch.randn((Kd,), generator=g)).to(dtype).to(device)
    h = torch.empty_like(xd)
    K.rms_norm(h, xd, norm, 1e-5)
    normed, gated = K.linear(h, wd), K.linear_silu_and_mul(xd, wd) if N % 32 == 0 else None
    if gated is not None:
        act = torch.empty_like(gated)
        K.silu_and_mul(act, whole)
        assert torch.equal(gated, act)
    for m in (1, 2, 4, 5, 16, 17, 33, 65, 97):
        assert torch.equal(K.linear(xd[:m], wd), whole[:m])
        if gated is not None:
            assert torch.equal(K.linear_silu_and_mul(xd[:m], wd), gated[:m])
        if K.rms_norm_linear_takes(xd[:m], norm, wd):
            assert torch.equal(K.rms_norm_linear(xd[:m], norm, 1e-5, wd), normed[:m])
    # ranges of uneven lengths
    for splits in (3, 7):
        K.tuning_set("linear_splits", splits)
        check(K.linear(xd[:17], wd), x[:17], w)


@pytest.mark.parametrize("heads,same", [((48, 8, 128), True), ((120, 4, 64), True), ((32, 2, 256), False), ((88, 4, 96), False)])
def test_qkv_linear_of_many_heads(device, heads, same):
    """Heads that divide the 128 rows that share an order of k: the bits of the calls; others: their own order, the same in every form."""
    Hq, Hkv, d = heads
    Kd, M, N = 2048, 40, (Hq + 2 * Hkv) * d
    x, w, g = operands(M, N, Kd, torch.bfloat16, seed=d)
    xd, wd = x.to(device), w.to(device)
    table = torch.randn((64, d), generator=g).to(torch.bfloat16).to(device)
    caches = [torch.zeros((4, Hkv, d // 8, 16, 8), dtype=torch.bfloat16, device=device),
              torch.zeros((4, Hkv, d, 16), dtype=torch.bfloat16, device=device)]
    pos = torch.randint(0, 64, (M,), generator=g).to(device)
    slots = torch.randperm(64, generator=g)[:M].to(device)
    assert K.qkv_linear_takes(xd, wd, table, *caches) and N >= 8192
    first = [c.clone() for c in caches]
    got = K.qkv_linear(xd, None, 0.0, wd, pos, table, *first, slots)
    for m in (5, 16, 17):
        few = [c.clone() for c in caches]
        assert torch.equal(K.qkv_linear(xd[:m], None, 0.0, wd, pos[:m], table, *few, slots[:m]), got[:m])
    want, wkc, wvc = K.linear(xd, wd), caches[0].clone(), caches[1].clone()
    q, k, v = want.split([Hq * d, Hkv * d, Hkv * d], dim=1)
    K.rotary_embedding_and_cache(pos, q, k, v.view(M, Hkv, d), d, table, True, wkc, wvc, slots)
    if same:
        assert torch.equal(got, want) and torch.equal(first[0], wkc) and torch.equal(first[1], wvc)
    else:
        check(got[:, (Hq + Hkv) * d:], x, w[(Hq + Hkv) * d:])  # values are not rotated
        assert ((got - want).float().norm() / want.float().norm()).item() <= 2.0 ** -8


@pytest.mark.parametrize("d,M", [(128, 1), (128, 4), (64, 3), (128, 16)])
def test_qkv_linear_in_workgroups_of_128_rows(device, d, M):
    Hkv, Kd = 8, 2048
    Hq = 18432 // d - 2 * Hkv
    x, w, g = operands(M, 18432, Kd, torch.bfloat16, seed=d + M)
    xd, wd = x.to(device), w.to(device)
    norm = (1 + 0.2 * torch.randn((Kd,), generator=g)).to(torch.bfloat16).to(device)
    h = torch.empty_like(xd)
    K.rms_norm(h, xd, norm, 1e-5)
    table = torch.randn((64, d), generator=g).to(torch.bfloat16).to(device)
    pos, slots = torch.arange(M, device=device) + 3, torch.arange(M, device=device) * 3
    caches = [torch.zeros((4, Hkv, d // 8, 16, 8), dtype=torch.bfloat16, device=device),
              torch.zeros((4, Hkv, d, 16), dtype=torch.bfloat16, device=device)]
    want, wkc, wvc = K.linear(h, wd), caches[0].clone(), caches[1].clone()
    check(want, h.cpu(), w)
    q, k, v = want.split([Hq * d, Hkv * d, Hkv * d], dim=1)
    K.rotary_embedding_and_cache(pos, q, k, v.view(M, Hkv, d), d, table, True, wkc, wvc, slots)
    for rows, nw in ((h, None), (xd, norm)):
        if nw is not None and not K.rms_norm_linear_takes(xd, norm, wd):
            continue
        kc, vc = caches[0].clone(), caches[1].clone()
        got = K.qkv_linear(rows, nw, 1e-5, wd, pos, table, kc, vc, slots)
        assert torch.equal(got, want) and torch.equal(kc, wkc) and torch.equal(vc, wvc)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,Kd", [((32, 2, 256), 2048), ((88, 4, 96), 2048), ((64, 32, 80), 4096), ((64, 16, 112), 6144),
                                      ((70, 5, 208), 2048)])
def test_qkv_linear_of_heads_that_do_not_divide_128_has_the_bits_of_the_calls(device, dtype, heads, Kd):
    """Weights whose ranges of k begin inside, up to 16 rows also uncut ones; also through rows of out on 8-byte boundaries."""
    Hq, Hkv, d = heads
    M, N = 40, (Hq + 2 * Hkv) * d
    x, w, g = operands(M, N, Kd, dtype, seed=d)
    xd, wd = x.to(device), w.to(device)
    norm = (1 + 0.2 * torch.randn((Kd,), generator=g)).to(dtype).to(device)
    table = torch.randn((64, d), generator=g).to(dtype).to(device)
    empty = [torch.zeros((4, Hkv, d // 8, 16, 8), dtype=dtype, device=device), torch.zeros((4, Hkv, d, 16), dtype=dtype, device=device)]
    pos, slots = torch.randint(0, 64, (M,), generator=g).to(device), torch.randperm(64, generator=g)[:M].to(device)
    for m in (1, 4, 5, 16, 17, 40):
        if not K.qkv_linear_takes(xd[:m], wd, table, *empty):
            assert N >= 16384 and m > 16
            continue
        for nw in (None, norm) if K.rms_norm_linear_takes(xd[:m], norm, wd) else (None,):
            want = K.linear(xd[:m], wd) if nw is None else K.rms_norm_linear(xd[:m], nw, 1e-5, wd)
            q, k, v = want.split([Hq * d, Hkv * d, Hkv * d], dim=1)
            caches = [c.clone() for c in empty]
            K.rotary_embedding_and_cache(pos[:m], q, k, v.view(m, Hkv, d), d, table, True, *caches, slots[:m])
            for out in (torch.empty((m, N), dtype=dtype, device=device), torch.empty((m, N + 8), dtype=dtype, device=device)[:, 4:-4]):
                mine = [c.clone() for c in empty]
                _native.qkv_linear(out, xd[:m], nw, 1e-5, wd, pos[:m], table, *mine, slots[:m])
                assert torch.equal(out, want) and torch.equal(mine[0], caches[0]) and torch.equal(mine[1], caches[1])
