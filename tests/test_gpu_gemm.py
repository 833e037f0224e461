"""fb_gemm (many rows of x) against the exact device-independent decode times x in fp64, at the
edges of its tiles: rows of x and W around the tile sizes, K past and short of a 512-wide span
(the x past K must read as zeros: the memory behind it holds NaN), K-parts, every dtype."""
import ctypes

import pytest
import torch

from if_i_could_turn_back_time_amd import PackedWeight, _capi as C
from oracle import fourbit_oracle as O

DEV = "cuda:0"


def _poisoned(t):
    """t on the GPU, with NaN before and behind it in memory."""
    buf = torch.full((t.numel() + 4096,), float("nan"), dtype=t.dtype, device=DEV)
    v = buf[2048:2048 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,xdt", [("gf4", torch.float16), ("e2m1", torch.bfloat16),
                                     ("e2m1", torch.float16)])
@pytest.mark.parametrize("M,N,K", [
    (17, 1, 128), (32, 64, 512), (33, 63, 640), (48, 129, 384), (64, 300, 1152), (65, 15, 4224),
    (97, 513, 1024), (128, 257, 896), (129, 2050, 512), (333, 1028, 2176), (515, 4100, 640),
    (1025, 6145, 512), (40, 77, 8192)])
def test_gemm_vs_exact_product(fmt, xdt, M, N, K):
    print("gemm", fmt, xdt, M, N, K, flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    pw = PackedWeight.quantize(torch.randn(N, K, generator=g) * 0.02, fmt, device=DEV)
    x = torch.randn(M, K, generator=g).to(xdt)
    w = pw.dequant_host().double().to(DEV)
    xd = _poisoned(x)
    ref = xd.double() @ w.T
    # fp32 sums of K exact products: K roundings of at most 2^-24 of the sum of magnitudes
    bound = K * 2.0 ** -24 * (xd.double().abs() @ w.abs().T)
    for ydt, ulp in ((torch.float32, 2.0 ** -24), (torch.float16, 2.0 ** -11),
                     (torch.bfloat16, 2.0 ** -8)):
        shape = C.make_shape(N, K, M, C.FMT_BY_NAME[fmt], 0, C.DTYPE_CODE[xdt], C.DTYPE_CODE[ydt])
        y = _poisoned(torch.zeros(M, N)).to(ydt)
        C.gemm(pw.wdev, xd, y, shape)
        err = (y.double() - ref).abs()
        # the smallest normal's half ulp where the result is subnormal in 16 bits
        assert bool((err <= bound + ulp * (ref.abs() + bound) + 2.0 ** -25).all()), \
            (ydt, float((err - bound).max()))
        again = torch.empty_like(y)
        C.gemm(pw.wdev, xd, again, shape)
        assert torch.equal(y, again)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,block", [(20, 64, 1024, 256), (130, 96, 4096, 4096),
                                         (67, 40, 11008, 256)])
def test_gemm_rotated_vs_oracle(M, N, K, block):
    g = torch.Generator().manual_seed(M)
    pw = PackedWeight.quantize(torch.randn(N, K, generator=g) * 0.02, "gf4", fwht_block=block,
                               device=DEV)
    x = torch.randn(M, K, generator=g).half()
    shape = C.make_shape(N, K, M, C.FMT_GF4, block, C.DT_F16, C.DT_F32)
    y = torch.full((M, N), float("nan"), device=DEV)
    C.gemm(pw.wdev, _poisoned(x), y, shape)
    ref = O.y_ref("gf4", O.unpack_nibbles(pw.codes.numpy()),
                  pw.meta.numpy().view("uint16"), x, block)
    assert bool(((y.cpu() - ref).abs() <= 1e-2 + 1e-3 * ref.abs()).all())


@pytest.mark.gpu
def test_gemm_special_rows_stay_apart():
    """A row of infinities or NaN reaches its own outputs only."""
    g = torch.Generator().manual_seed(3)
    pw = PackedWeight.quantize(torch.randn(70, 640, generator=g) * 0.02, "gf4", device=DEV)
    x = torch.randn(40, 640, generator=g).half()
    x[3, 5], x[17, 0], x[39, 639] = float("inf"), float("nan"), float("-inf")
    y = torch.empty(40, 70, device=DEV)
    C.gemm(pw.wdev, _poisoned(x), y, C.make_shape(70, 640, 40, C.FMT_GF4, 0, C.DT_F16, C.DT_F32))
    bad = ~torch.isfinite(y).all(dim=1).cpu()
    assert bad.nonzero().flatten().tolist() == [3, 17, 39]


def test_gemm_refusals():
    L = C.lib()
    buf = (ctypes.c_uint8 * 512)()
    p = (ctypes.addressof(buf) + 255) // 256 * 256

    def rc(shape, w=p, x=p, y=p, ws=None, nb=0, bias=None, bdt=0):
        return L.fb_gemm(w, x, y, ctypes.byref(shape), bias, bdt, ws, nb, None)

    big = C.make_shape(64, (1 << 22) + 128, 32)
    assert rc(big) == -2 and L.fb_gemm_workspace_bytes(ctypes.byref(big)) == 0
    ok = C.make_shape(64, 4096, 32, C.FMT_GF4, 4096)
    need = L.fb_gemm_workspace_bytes(ctypes.byref(ok))
    assert need >= 32 * 4096 * 2
    assert rc(ok) == -1                             # the rotated x needs a workspace
    assert rc(ok, ws=p + 16, nb=need) == -7
    assert rc(ok, ws=p, nb=need - 256) == -8
    assert rc(ok, w=None) == -1 and rc(ok, x=p + 2) == -7 and rc(ok, y=p + 2) == -7
    assert rc(C.make_shape(64, 4096, 32, C.FMT_E2M1, 4096, C.DT_BF16)) == -5
    assert rc(C.make_shape(64, 100, 32)) == -2
    plain = C.make_shape(64, 512, 2048)
    assert rc(plain, bias=p, bdt=3) == -5 and rc(plain, bias=p + 2, bdt=2) == -7


@pytest.mark.gpu
@pytest.mark.parametrize("bdt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(33, 70, 512), (40, 132, 8192), (520, 1000, 640)])
def test_gemm_bias(bdt, M, N, K):
    """The bias joins the fp32 sums, in the tile's epilogue or in the K-parts' sum."""
    g = torch.Generator().manual_seed(N)
    pw = PackedWeight.quantize(torch.randn(N, K, generator=g) * 0.02, "gf4", device=DEV)
    x = torch.randn(M, K, generator=g).half().to(DEV)
    bias = torch.randn(N, generator=g).to(bdt).to(DEV)
    for ydt, ulp in ((torch.float32, 2.0 ** -24), (torch.float16, 2.0 ** -11)):
        shape = C.make_shape(N, K, M, C.FMT_GF4, 0, C.DT_F16, C.DTYPE_CODE[ydt])
        y = torch.full((M, N), float("nan"), dtype=ydt, device=DEV)
        C.gemm(pw.wdev, x, y, shape, bias)
        w = pw.dequant_host().double().to(DEV)
        ref = x.double() @ w.T + bias.double()
        bound = (K + 1) * 2.0 ** -24 * (x.double().abs() @ w.abs().T + bias.double().abs())
        assert bool(((y.double() - ref).abs() <= bound + ulp * (ref.abs() + bound)).all())
