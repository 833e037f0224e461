"""More rows of x than one fb_gemm call takes (2^24), or rotates at once (2^29 values)."""
import pytest
import torch

from if_i_could_turn_back_time_amd import PackedWeight, _capi as C
from if_i_could_turn_back_time_amd import linear as LN

DEV = "cuda:0"


@pytest.mark.parametrize("M,block,calls", [(17, 0, [17]), (64, 0, [64]), (65, 0, [64, 1]),
                                           (200, 0, [64, 64, 64, 8]), (100, 256, [48, 48, 4])])
def test_rows_in_slices(M, block, calls, monkeypatch):
    """_gemv_chunks covers the rows once each with calls of at most the limits' rows."""
    K, N = 256, 24
    seen = []

    def gemm(wdev, x, y, shape, bias=None):
        assert shape.B == x.shape[0] == y.shape[0] and x.is_contiguous() and y.is_contiguous()
        seen.append(shape.B)
        y.copy_(x[:, :N].to(y.dtype))
        return y

    monkeypatch.setattr(C, "gemm", gemm)
    monkeypatch.setattr(LN, "MAX_GEMM_ROWS", 64, raising=False)
    monkeypatch.setattr(LN, "MAX_ROTATED_VALUES", 60 * K, raising=False)
    x = torch.randn(M, K).half()
    y = torch.full((M, N), float("nan"))
    LN._gemv_chunks(None, N, K, "gf4", block, x, y)
    assert seen == calls and torch.equal(y, x[:, :N].float())


def test_rows_per_call():
    assert LN.gemm_rows(128, 0) == LN.gemm_rows(1 << 22, 0) == 1 << 24
    assert LN.gemm_rows(128, 128) == 1 << 22 and LN.gemm_rows(8192, 4096) == 1 << 16
    assert LN.gemm_rows(1 << 22, 256) == 128 and LN.gemm_rows(11008, 256) % 16 == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,block", [((1 << 24) + 40, 0), ((1 << 22) + 5, 128)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_layer_of_many_rows(M, block, with_bias):
    """The rows around a slice's end, and the last ones, are what they are on their own."""
    N, K = 16, 128
    pw = PackedWeight.quantize(torch.randn(N, K) * 0.05, "gf4", fwht_block=block, device=DEV)
    bias = torch.randn(N, device=DEV) if with_bias else None
    x = torch.empty(M, K, dtype=torch.float16, device=DEV).normal_()
    cut = LN.gemm_rows(K, block)
    for path in (LN._native_forward, None):  # the native call, then the Python one
        if path:
            y = LN.packed_linear(pw.wdev, N, K, "gf4", block, x, bias)
        else:
            y = LN._forward(x, pw.wdev, N, K, "gf4", block, False, True, False, None, True)
            if with_bias:
                y += bias.half()
        assert bool(torch.isfinite(y).all())
        for r0, r1 in ((0, 40), (cut - 40, cut + 5), (M - 40, M)):
            ref = LN.packed_linear(pw.wdev, N, K, "gf4", block, x[r0:r1], bias)
            # the same fp32 sums of K products, perhaps in another order, rounded to fp16 (and
            # once more with the bias on the Python path)
            assert torch.allclose(y[r0:r1].float(), ref.float(), rtol=2.0 ** -9, atol=2.0 ** -10)
        del y
