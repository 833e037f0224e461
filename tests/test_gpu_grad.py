"""fb_grad_x (the activation gradient) against grad_y times the exact decode in fp64: edges of
its tiles and chunks (rows of gy, of W and of K around them), every way it holds gy and W in 16
bits, K ranges and contraction parts, the rotation, and infinities."""
import pytest
import torch

from if_i_could_turn_back_time_amd import PackedWeight, QuantLinear, _capi as C
from if_i_could_turn_back_time_amd import linear as LN

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _weight(fmt, N, K, g, block=0):
    return PackedWeight.quantize(torch.randn(N, K, generator=g) * 0.02, fmt, fwht_block=block,
                                 device=DEV)


def _run(pw, gy, gx_dtype, f16_exact=True):
    M, N = gy.shape
    shape = C.make_shape(N, pw.K, M, pw.fmt, pw.fwht_block, C.DT_F16, C.DTYPE_CODE[gy.dtype])
    gx = torch.full((M, pw.K), float("nan"), dtype=gx_dtype, device=DEV)
    return C.grad_x(pw.wdev, gy, gx, shape, f16_exact)


@pytest.mark.parametrize("fmt,gdt,exact16", [
    ("gf4", torch.float16, True), ("gf4", torch.bfloat16, True), ("gf4", torch.float32, True),
    ("e2m1", torch.bfloat16, True), ("e2m1", torch.float16, True),
    ("e2m1", torch.float16, False), ("e2m1", torch.float32, True)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 128), (17, 16, 512), (31, 127, 640), (32, 128, 1152),
                                   (65, 264, 384), (129, 1000, 2176), (300, 2051, 4224),
                                   (513, 515, 896), (64, 8200, 128)])
def test_grad_vs_exact_product(fmt, gdt, exact16, M, N, K):
    print("grad", fmt, gdt, exact16, M, N, K, flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    pw = _weight(fmt, N, K, g)
    # magnitudes from 1e-7 (fp16: subnormal) to 1
    gy = torch.randn(M, N, generator=g) * 10.0 ** torch.randint(-7, 1, (M, N), generator=g)
    buf = torch.full((M * N + 4096,), float("nan"), dtype=gdt, device=DEV)
    gd = buf[2048:2048 + M * N].view(M, N)
    gd.copy_(gy)
    w = pw.dequant_host().double().to(DEV)
    ref = gd.double() @ w
    # every product is exact; at most 6 N of them are summed in fp32
    bound = 6 * N * 2.0 ** -24 * (gd.double().abs() @ w.abs()) + 1e-40
    for xdt in (torch.float32, gdt):
        gx = _run(pw, gd, xdt, exact16)
        err = (gx.double() - ref).abs()
        assert bool((err <= bound + ULP[xdt] * (ref.abs() + bound) + 2.0 ** -25 *
                     (xdt == torch.float16)).all()), (xdt, float((err - bound).max()))
        assert torch.equal(gx, _run(pw, gd, xdt, exact16))


@pytest.mark.parametrize("M,N,K,block", [(5, 40, 256, 256), (33, 130, 4096, 4096),
                                         (20, 64, 11008, 256), (18, 48, 6144, 2048),
                                         (17, 32, 384, 128), (17, 32, 256, 2)])
def test_grad_rotated(M, N, K, block):
    g = torch.Generator().manual_seed(block)
    pw = _weight("gf4", N, K, g, block)
    for gdt in (torch.float16, torch.float32):
        gy = torch.randn(M, N, generator=g).to(gdt).to(DEV)
        ref = LN._fwht_last_dim(gy.double().float() @ pw.dequant_host().to(DEV), block).double()
        gx = _run(pw, gy, torch.float32)
        # fp32 sums of N products, then log2(block) additions, on values whose block has this norm
        norm = (gy.double().abs() @ pw.dequant_host().double().abs().to(DEV)).norm(dim=1).max()
        assert float((gx.double() - ref).abs().max()) <= (2 * N + 24) * 2.0 ** -24 * float(norm)


def test_grad_in_k_ranges():
    """A weight whose 16-bit operands pass 256 MiB runs a range of K at a time (here 2 spans of
    100,000 rows, then 1)."""
    N, K = 100000, 1536
    g = torch.Generator().manual_seed(5)
    codes = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
    meta = torch.randint(118, 124, (N, K // 32), generator=g, dtype=torch.uint8)
    pw = PackedWeight("e2m1", N, K, codes, meta, 0, DEV)
    gy = torch.randn(19, N, generator=g).bfloat16().to(DEV)
    shape = C.make_shape(N, K, 19, C.FMT_E2M1, 0, C.DT_BF16, C.DT_BF16)
    import ctypes
    assert C.lib().fb_grad_x_workspace_bytes(ctypes.byref(shape), 1) < N * K * 2
    w = pw.dequant_device().double()
    ref = gy.double() @ w
    gx = _run(pw, gy, torch.float32)
    assert bool(((gx.double() - ref).abs() <= N * 2.0 ** -24 * (gy.double().abs() @ w.abs())).all())


@pytest.mark.parametrize("fmt", ["gf4", "e2m1"])
@pytest.mark.parametrize("gdt", [torch.float16, torch.bfloat16, torch.float32])
def test_grad_infinities_as_in_fp32(fmt, gdt):
    """Non-finite gradients give what an fp32 product gives: +-inf by the weight's sign, NaN
    where the weight is 0, and leave the other rows alone."""
    g = torch.Generator().manual_seed(9)
    pw = _weight(fmt, 48, 256, g)
    gy = torch.randn(20, 48, generator=g)
    gy[2, 7], gy[5, 0], gy[9, 47] = float("inf"), float("-inf"), float("nan")
    if gdt == torch.float32:
        gy[11, 3] = 3.4e38
    gy = gy.to(gdt).to(DEV)
    ref = gy.float() @ pw.dequant_host().to(DEV)
    gx = _run(pw, gy, torch.float32)
    assert torch.equal(torch.isnan(gx), torch.isnan(ref))
    assert torch.equal(gx[[2, 5]], ref[[2, 5]]) or torch.equal(
        torch.nan_to_num(gx[[2, 5]]), torch.nan_to_num(ref[[2, 5]]))
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(gx), fin)
    assert torch.allclose(gx[fin], ref[fin], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("kw", [dict(fmt="gf4"), dict(fmt="gf4", hadamard=256),
                                dict(fmt="e2m1"), dict(fmt="e2m1", fp4_mfma=True)])
def test_layer_gradient_and_its_gradient(kw):
    """The layer's backward (native) equals its differentiable form (torch operations), for an
    expanded grad_y too, and can itself be differentiated."""
    torch.manual_seed(4)
    q = QuantLinear(torch.nn.Linear(768 if "hadamard" in kw else 700, 130), **kw).to(DEV)
    x = torch.randn(37, q.in_features, device=DEV, requires_grad=True)
    for gy in (torch.randn(37, 130, device=DEV), torch.ones(1, 1, device=DEV).expand(37, 130)):
        y = q(x)
        (a,) = torch.autograd.grad(y, x, gy, retain_graph=True)
        g2 = gy.clone().requires_grad_(True)
        (b,) = torch.autograd.grad(y, x, g2, create_graph=True)
        assert a.is_contiguous() and torch.allclose(a, b, rtol=1e-5, atol=1e-5)
        (c,) = torch.autograd.grad(b.sum(), g2)
        assert c.shape == gy.shape and bool(torch.isfinite(c).all())


@pytest.mark.parametrize("gdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [(1, 1), (15, 63), (16, 64), (17, 65), (333, 1000), (2100, 130)])
def test_grad_bias(gdt, M, N):
    """Column sums in fp32 (at most M / 64 + 64 roundings each), and the layer's bias gradient."""
    g = torch.Generator().manual_seed(M)
    gy = torch.randn(M, N, generator=g).to(gdt).to(DEV)
    gb = C.native().linear_grad_bias(gy, torch.float32)
    ref = gy.double().sum(0)
    bound = (M / 64 + 65) * 2.0 ** -24 * gy.double().abs().sum(0)
    assert bool(((gb.double() - ref).abs() <= bound + 1e-40).all())
    q = QuantLinear(torch.nn.Linear(128, N), fmt="gf4").to(DEV)
    x = torch.randn(M, 128, device=DEV, dtype=gdt, requires_grad=True)
    gx, gq = torch.autograd.grad(q(x), (x, q.bias), gy)
    assert gq.dtype == q.bias.dtype and torch.equal(gq, gb)


@pytest.mark.parametrize("gdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [
    (2048, 48), (2049, 48), (2049, 1), (3071, 1), (3073, 2), (4095, 7), (4099, 63), (4096, 64),
    (4103, 65), (9000, 300), (70001, 513), (1 << 18, 48), ((1 << 20) + 3, 1), (1 << 20, 24),
    (12345, 4096), (64, 98305), (65, 98305), (600, 11008), (1537, 4099)])
def test_grad_bias_of_many_rows(gdt, M, N):
    """More than 2048 rows, or 6 Mi values, are summed in parts: at most 256 additions in a row in
    the first pass, 8 in the others and 96 in the last, so at most 400 roundings whatever M is."""
    print("grad bias", gdt, M, N, flush=True)
    buf = torch.full((M * N + 8192,), float("nan"), dtype=gdt, device=DEV)
    for shift in (4096, 4097):  # 16-byte aligned or not, NaN around
        gy = buf[shift:shift + M * N].view(M, N)
        gy.normal_()
        gb = C.native().linear_grad_bias(gy, torch.float32)
        ref = gy.double().sum(0)
        assert bool(((gb.double() - ref).abs() <= 400 * 2.0 ** -24 * gy.double().abs().sum(0)).all())
        assert torch.equal(gb, C.native().linear_grad_bias(gy, torch.float32))
        half = C.native().linear_grad_bias(gy, torch.float16)
        assert torch.equal(half, gb.half())
        gy.fill_(float("nan"))


def test_grad_bias_workspace_contract():
    L = C.lib()
    assert L.fb_grad_bias_workspace_bytes(2048, 300) == 0 == L.fb_grad_bias_workspace_bytes(0, 1)
    assert L.fb_grad_bias_workspace_bytes(64, 1 << 20) == 0 < L.fb_grad_bias_workspace_bytes(65, 1 << 20)
    need = L.fb_grad_bias_workspace_bytes(5000, 300)
    gy = torch.randn(5000, 300, device=DEV)
    gb = torch.empty(300, device=DEV)
    ws = torch.empty(need + 256, dtype=torch.uint8, device=DEV)
    s = torch.cuda.current_stream().cuda_stream

    def rc(ws_ptr, nbytes, g=gy.data_ptr(), dt=C.DT_F32, M=5000):
        return L.fb_grad_bias_ws(g, dt, M, 300, gb.data_ptr(), C.DT_F32, ws_ptr, nbytes, s)

    assert rc(None, 0) == -1 and rc(ws.data_ptr() + 16, need) == -7
    assert rc(ws.data_ptr(), need - 1) == -8
    assert rc(ws.data_ptr(), need, g=None) == -1 and rc(ws.data_ptr(), need, dt=3) == -5
    assert rc(ws.data_ptr(), need, g=gy.data_ptr() + 2) == -7 and rc(None, 0, M=0) == -2
    assert rc(ws.data_ptr(), need) == 0 and rc(None, 0, M=2048) == 0


@pytest.mark.parametrize("ydt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [(1, 300), (3, 77), (16, 4096)])
def test_gemv_bias_is_the_in_place_add(ydt, M, N):
    """The native path's bias of 1 to 16 rows rounds as y.add_(bias.to(y.dtype))."""
    q = QuantLinear(torch.nn.Linear(256, N), fmt="gf4").to(DEV)
    x = torch.randn(M, 256, device=DEV, dtype=ydt)
    with torch.no_grad():
        y = q(x)
        b, q.bias = q.bias, None
        assert torch.equal(y, q(x).add_(b.to(ydt)))


def test_layer_gradient_of_many_rows():
    """More rows than one fb_grad_x call takes (8,192) and a ragged in_features."""
    torch.manual_seed(6)
    q = QuantLinear(torch.nn.Linear(200, 48), fmt="gf4").to(DEV)
    x = torch.randn(8300, 200, device=DEV, dtype=torch.float16, requires_grad=True)
    gy = torch.randn(8300, 48, device=DEV, dtype=torch.float16)
    (gx,) = torch.autograd.grad(q(x), x, gy)
    ref = gy.double() @ q.dequantized_weight().double().to(DEV)
    assert float((gx.double() - ref).abs().max()) <= 2.0 ** -11 * float(ref.abs().max()) * 1.01


def test_step_in_hip_graph_replays_match_eager():
    """Forward (K-parts, a rotated layer) and backward captured in a HIP graph: three replays on
    changed inputs, with eager work between them, equal the eager results."""
    torch.manual_seed(8)
    for kw, M in ((dict(fmt="gf4", hadamard=4096), 40), (dict(fmt="e2m1"), 130)):
        q = QuantLinear(torch.nn.Linear(4096, 200), **kw).to(DEV)
        x = torch.randn(M, 4096, device=DEV, dtype=torch.float16, requires_grad=True)
        gy = torch.randn(M, 200, device=DEV, dtype=torch.float16)

        def step():
            y = q(x)
            return (y, *torch.autograd.grad(y, (x, q.bias), gy))

        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(2):
                step()
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
        for k in range(3):
            with torch.no_grad():
                x.copy_(torch.randn(M, 4096, device=DEV))
                gy.copy_(torch.randn(M, 200, device=DEV))
            graph.replay()
            got = [t.detach().clone() for t in out]
            torch.cuda.synchronize()
            for a, b in zip(got, step()):
                assert torch.equal(a, b)
