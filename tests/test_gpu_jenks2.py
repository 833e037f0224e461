"""GPU two-class Jenks (fb_jenks2_gpu) against the oracle and its host twin, bit for bit: the
split, the GVF and the mask, on the reference's pruned LeNet300 weights (the arrays its
Linear_Mask / Bias_Mask prune, cuda_helpers.py:378-411) and on random arrays across the
256-element block and 65536-element superblock edges; the per-filter version likewise."""
import sys
import time

import numpy as np
import pytest
import torch

from oracle import fourbit_oracle as O
from if_i_could_turn_back_time_amd import _capi as C
from if_i_could_turn_back_time_amd import bias_mask, linear_mask
from model_fixtures import lenet300_from_fixture

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _inputs():
    rng = np.random.default_rng(11)
    net = lenet300_from_fixture()
    for i in (1, 3, 5):
        yield f"lenet300.{i}.weight", net[i].weight.detach().numpy()
        yield f"lenet300.{i}.bias", net[i].bias.detach().numpy()
    for n in (1, 2, 3, 255, 256, 257, 4096, 65535, 65536, 65537, 131073, 1000003):
        w = (rng.standard_normal(n) * 0.02).astype(np.float32)
        if n > 8:
            w[rng.integers(0, n, n // 4)] = 0.0
            w[rng.integers(0, n, n // 8)] = -0.0
        yield f"random{n}", w
    yield "constant", np.full(3000, -0.125, np.float32)
    yield "two-levels", np.repeat(np.array([1.0, -2.0], np.float32), 777)


@pytest.mark.parametrize("case", list(range(20)))
def test_jenks2_gpu_bit_exact_vs_host(case):
    name, w = list(_inputs())[case]
    say("jenks2", name, w.size)
    wt = torch.from_numpy(np.ascontiguousarray(w))
    keep_h, split_h, gvf_h = C.jenks2_host(wt)
    keep_g, split_g, gvf_g = C.jenks2_gpu(wt.to(DEV))
    keep_o, split_o, gvf_o, _ = O.jenks2(w)
    assert split_g == split_h == split_o, name
    assert (np.float64(gvf_g).view(np.int64) == np.float64(gvf_h).view(np.int64)
            == np.float64(gvf_o).view(np.int64)), name
    assert torch.equal(keep_g.cpu(), keep_h), name
    assert np.array_equal(keep_g.cpu().numpy().astype(bool), keep_o), name


def test_linear_mask_on_device_matches_host():
    """linear_mask / bias_mask on ROCm tensors return what they return on the CPU."""
    net = lenet300_from_fixture()
    for i in (1, 3, 5):
        mh, gh = linear_mask(net[i].weight.detach())
        md, gd = linear_mask(net[i].weight.detach().to(DEV))
        assert torch.equal(mh, md) and gh == gd and md.device.type == "cpu"
        bh, _ = bias_mask(net[i].bias.detach())
        bd, _ = bias_mask(net[i].bias.detach().to(DEV))
        assert torch.equal(bh, bd)


def test_jenks2_gpu_large_array():
    """A 32M-value array (an 8192 x 4096 layer): bit-exact against the host twin; the
    GPU time is printed (the reference's one-thread-per-split kernel is O(n^2))."""
    g = torch.Generator().manual_seed(3)
    w = torch.randn(8192 * 4096, generator=g) * 0.02
    w[torch.rand(w.numel(), generator=g) < 0.5] = 0.0
    keep_h, split_h, gvf_h = C.jenks2_host(w)
    wd = w.to(DEV)
    C.jenks2_gpu(wd)                                   # warm-up
    torch.cuda.synchronize()
    t = time.perf_counter()
    keep_g, split_g, gvf_g = C.jenks2_gpu(wd)
    torch.cuda.synchronize()
    say(f"jenks2 gpu 32M values: {(time.perf_counter() - t) * 1e3:.1f} ms (incl. workspace "
        "allocation and the host copy of split / GVF)")
    assert split_g == split_h and gvf_g == gvf_h
    assert torch.equal(keep_g.cpu(), keep_h)


def _filter_inputs():
    """Convolution weights [out, in, kh, kw]: LeNet-5, VGG, AlexNet-stem and ResNet-stem
    filter sizes, the per-filter maximum of 1024 values, ties, signed zeros and constant
    filters."""
    rng = np.random.default_rng(12)
    # one filter per lane for 1024 or more filters of at most 25 values (2100 filters: a
    # partial last workgroup; 1 and 4 values), else one filter per one-wave workgroup (25
    # values in 6 filters; 26 values, the smallest size never run per lane)
    for shape in ((6, 1, 5, 5), (64, 64, 3, 3), (64, 3, 11, 11), (64, 3, 7, 7), (2, 3, 32, 32),
                  (7, 5, 1, 1), (3, 2, 16, 17), (3, 3, 2, 13), (300, 7, 3, 3), (7, 3, 2, 13),
                  (1024, 2, 1, 1), (40, 30, 2, 2), (64, 32, 5, 5)):
        yield f"random{shape}", (rng.standard_normal(shape) * 0.05).astype(np.float32)
    w = (np.round(rng.standard_normal((32, 16, 3, 3)) * 2) / 4).astype(np.float32)
    w[::3] = 0.0
    w[1::5, :, ::2] = -0.0
    w[2] = 0.7
    yield "ties", w


@pytest.mark.parametrize("case", list(range(14)))
def test_jenks2_filters_gpu_bit_exact_vs_host(case):
    """fb_jenks2_filters_gpu (the reference's Conv_Mask, cuda_helpers.py:333-376) against
    the oracle and its host twin, bit for bit, on every filter: split, GVF and mask."""
    name, w = list(_filter_inputs())[case]
    say("jenks2 filters", name)
    w2 = torch.from_numpy(w.reshape(w.shape[0] * w.shape[1], -1))
    keep_h, split_h, gvf_h = C.jenks2_filters_host(w2)
    keep_g, split_g, gvf_g = C.jenks2_filters_gpu(w2.to(DEV))
    torch.cuda.synchronize()
    assert torch.equal(split_g.cpu(), split_h), name
    assert torch.equal(gvf_g.cpu().view(torch.int64), gvf_h.view(torch.int64)), name
    assert torch.equal(keep_g.cpu(), keep_h), name
    keep_o, split_o, gvf_o = O.jenks2_filters(w2.numpy())
    assert np.array_equal(split_g.cpu().numpy(), split_o), name
    assert np.array_equal(gvf_g.cpu().numpy().view(np.int64), gvf_o.view(np.int64)), name
    assert np.array_equal(keep_g.cpu().numpy().astype(bool), keep_o), name


def test_conv_mask_on_device_matches_host():
    """conv_mask keeps the mask on the weights' device (as the reference's Conv_Mask does)
    and gives the host's mask and GVF list; a 512 x 512 x 3 x 3 layer is timed."""
    from if_i_could_turn_back_time_amd import jenks
    g = torch.Generator().manual_seed(5)
    w = torch.randn(512, 512, 3, 3, generator=g) * 0.05
    mh, gh = jenks.conv_mask(w)
    wd = w.to(DEV)
    jenks.conv_mask(wd)                                # warm-up
    torch.cuda.synchronize()
    t = time.perf_counter()
    md, gd = jenks.conv_mask(wd)
    torch.cuda.synchronize()
    say(f"conv_mask 512x512x3x3 on the GPU: {(time.perf_counter() - t) * 1e3:.2f} ms (incl. the "
        "finiteness check and the GVF copy to the host)")
    assert md.device.type == "cuda" and md.dtype == torch.float32
    assert torch.equal(md.cpu(), mh) and gd == gh


def _reference_var_f64(v):
    """The reference kernels' per-split SSD (cuda_helpers.py:85-118, :151-184: serial class
    means, then serial squared deviations), in float64."""
    v = np.asarray(v, np.float64)
    n = v.size
    var = np.zeros(n)
    for idx in range(n):
        m1 = v[:idx].sum() / idx if idx else 0.0
        m2 = v[idx:].sum() / (n - idx)
        var[idx] = ((v[:idx] - m1) ** 2).sum() + ((v[idx:] - m2) ** 2).sum()
    return var


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_jenks2_ssd_gpu_bit_exact_vs_oracle_and_host(dtype):
    """fb_jenks2_ssd_gpu (the per-split SSD the reference's optimizers bind,
    jenks_optimization_cuda / jenks_optimization_biases_cuda) against the oracle's
    jenks2_ssd rounded to the dtype and the host twin, bit for bit, across the block and
    superblock edges, with ties and signed zeros; and within float64 rounding of the
    reference kernels' own two-pass sums on a short array."""
    rng = np.random.default_rng(31)
    npdt = np.float32 if dtype == torch.float32 else np.float64
    for n in (1, 2, 255, 256, 257, 4096, 65535, 65536, 65537, 131073, 1000003):
        say("jenks2 ssd", dtype, n)
        w = (rng.standard_normal(n) * 0.02).astype(npdt)
        if n > 8:
            w[rng.integers(0, n, n // 4)] = 0.0
            w[rng.integers(0, n, n // 8)] = -0.0
        v = np.sort(w, kind="stable")
        vt = torch.from_numpy(v)
        got = C.jenks2_ssd(vt.to(DEV))
        torch.cuda.synchronize()
        assert got.dtype == dtype and got.device.type == "cuda" and got.shape == (n,)
        g = got.cpu().numpy()
        assert np.array_equal(g.view(np.uint8), O.jenks2_ssd(v).astype(npdt).view(np.uint8)), n
        assert np.array_equal(g.view(np.uint8), C.jenks2_ssd(vt).numpy().view(np.uint8)), n
    v = np.sort((rng.standard_t(3, size=300) * 0.05).astype(npdt))
    ref = _reference_var_f64(v)
    got = C.jenks2_ssd(torch.from_numpy(v).to(DEV)).cpu().numpy().astype(np.float64)
    tol = (1e-5 if dtype == torch.float32 else 1e-9) * ref[0]
    assert np.allclose(got, ref, rtol=0, atol=tol)


def test_reference_optimizer_call_pattern_binds_unchanged():
    """The reference's JenksSGD steps (custom_optimizer.py:130-139 for weights, :162-167 for
    biases) and Conv_Mask (cuda_helpers.py:349-359) run as written against module_weights,
    module_bias and module_conv: output shapes, dtypes and devices are the reference's, the
    values are the oracle's per-split SSD, and var.argmin() is the mask path's split."""
    from if_i_could_turn_back_time_amd import module_bias, module_conv, module_weights
    g = torch.Generator().manual_seed(41)
    W = (torch.randn(300, 100, generator=g) * 0.05).to(DEV)
    grad = torch.randn(300, 100, generator=g).to(DEV) * 0.01
    s_W = torch.abs(torch.mul(W, grad))
    WB_cuda_sorted, WB_cuda_indices = s_W.flatten().sort()
    WB_cuda_sorted = WB_cuda_sorted.reshape(s_W.shape)
    var = module_weights.jenks_optimization_cuda(WB_cuda_sorted)
    var_min = var.argmin().item()
    assert var.shape == (30000,) and var.dtype == torch.float32 and var.is_cuda
    srt = WB_cuda_sorted.reshape(-1).cpu().numpy()
    assert np.array_equal(var.cpu().numpy(), O.jenks2_ssd(srt).astype(np.float32))
    _, split, _, _ = O.jenks2(s_W.reshape(-1).cpu().numpy())
    ssd64 = O.jenks2_ssd(srt)
    assert var_min == int(np.argmin(var.cpu().numpy()))
    assert ssd64[var_min] <= ssd64[split] * (1 + 1e-6)        # equal up to the fp32 rounding
    b = (torch.randn(100, generator=g) * 0.05).to(DEV).double()
    B_cuda_sorted, _ = torch.abs(b).sort()
    vb = module_bias.jenks_optimization_biases_cuda(B_cuda_sorted)
    assert vb.shape == (100,) and vb.dtype == torch.float64
    assert np.array_equal(vb.cpu().numpy(), O.jenks2_ssd(B_cuda_sorted.cpu().numpy()))
    Wc = (torch.randn(16, 8, 3, 3, generator=g) * 0.05).to(DEV)
    flat = Wc.view(16 * 8, -1)
    sorted_weights, _ = torch.sort(flat, dim=1)
    weights_sorted = sorted_weights.view(16, 8, 3, 3).contiguous()
    vc = module_conv.jenks_optimization_cuda_conv(weights_sorted)
    assert vc.shape == (16 * 8 * 9,) and vc.dtype == torch.float32
    ref = np.stack([O.jenks2_ssd(r) for r in sorted_weights.cpu().numpy()]).astype(np.float32)
    assert np.array_equal(vc.cpu().numpy().reshape(128, 9), ref)
    _, cs, _ = O.jenks2_filters(flat.cpu().numpy())
    mins = vc.view(16, 8, -1).min(dim=2).indices.cpu().numpy().reshape(-1)
    ssds = [O.jenks2_ssd(r) for r in sorted_weights.cpu().numpy()]
    for f in range(128):
        assert ssds[f][mins[f]] <= ssds[f][cs[f]] * (1 + 1e-6) + 1e-30
    with pytest.raises(RuntimeError, match="contiguous"):
        module_weights.jenks_optimization_cuda(WB_cuda_sorted.t())
    with pytest.raises(RuntimeError, match="not implemented"):
        module_weights.jenks_optimization_cuda(WB_cuda_sorted.half())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_jenks2_ssd_filters_gpu_bit_exact(dtype):
    """fb_jenks2_ssd_filters_gpu against the host twin and the oracle per filter, bit for
    bit, at the per-filter size edges (1, 9, 25, a 256-block and past it, the maximum)."""
    rng = np.random.default_rng(32)
    npdt = np.float32 if dtype == torch.float32 else np.float64
    for nf, n in ((3000, 9), (700, 25), (5, 1), (9, 256), (9, 257), (4, C.JENKS2_FILTER_MAX)):
        say("jenks2 ssd filters", dtype, nf, n)
        w = np.sort((rng.standard_normal((nf, n)) * 0.05).astype(npdt), axis=1)
        w[::7, : n // 2] = 0.0
        got = C.jenks2_ssd_filters(torch.from_numpy(w).to(DEV))
        torch.cuda.synchronize()
        assert got.dtype == dtype and got.is_cuda
        g = got.cpu().numpy()
        host = C.jenks2_ssd_filters(torch.from_numpy(w)).numpy()
        assert np.array_equal(g.view(np.uint8), host.view(np.uint8))
        for f in range(0, nf, max(1, nf // 25)):
            assert np.array_equal(g[f], O.jenks2_ssd(w[f]).astype(npdt)), (nf, n, f)


# ---------------------------------------------------------------- the mask at any split
def _ties_lib():
    import ctypes
    from pathlib import Path
    path = Path(__file__).resolve().parent / "c" / "jenks2_ties.so"
    assert path.exists(), "tests/c/jenks2_ties.so is not built: run __graft_entry__.build()"
    L = ctypes.CDLL(str(path))
    L.ties_scratch_bytes.restype = ctypes.c_int64
    L.ties_scratch_bytes.argtypes = [ctypes.c_int64]
    L.ties_mask.argtypes = [ctypes.c_void_p, ctypes.c_int64] + [ctypes.c_void_p] * 5
    return L


def _mask_at(L, w, srt, split, shift=0):
    n = w.size
    wd = torch.empty(n + shift, dtype=torch.float32, device=DEV)[shift:]
    wd.copy_(torch.from_numpy(w))
    keep = torch.full((n + shift + 8,), 7, dtype=torch.uint8, device=DEV)
    scratch = torch.full((L.ties_scratch_bytes(n),), 255, dtype=torch.uint8, device=DEV)
    sd = torch.from_numpy(srt).to(DEV)
    sp = torch.tensor([split], dtype=torch.int64, device=DEV)
    assert L.ties_mask(wd.data_ptr(), n, sd.data_ptr(), sp.data_ptr(), keep[shift:].data_ptr(),
                       scratch.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    out = keep.cpu().numpy()
    assert (out[:shift] == 7).all() and (out[shift + n:] == 7).all()
    return out[shift:shift + n]


# segments of 16384 values are counted one by one; n around their edges, and many of them
@pytest.mark.parametrize("n", [1, 2, 5, 16383, 16384, 16385, 32768, 49152 + 7, 300001])
@pytest.mark.parametrize("kind", ["few values", "zeros", "constant", "clustered", "distinct"])
def test_mask_of_a_split_inside_equal_values(n, kind):
    """At every kind of position (first, inside and last of a run of equal values, -0.0 and +0.0
    among them) the mask is that of the stable ascending order."""
    say("mask", n, kind)
    L = _ties_lib()
    rng = np.random.default_rng(n)
    if kind == "few values":
        w = rng.integers(-2, 3, n).astype(np.float32) / 4
        w[rng.random(n) < 0.3] = -0.0
    elif kind == "zeros":  # nearly all zeros of either sign
        w = np.where(rng.random(n) < 0.01, rng.standard_normal(n), 0.0).astype(np.float32)
        w[rng.random(n) < 0.5] *= -1
    elif kind == "constant":
        w = np.full(n, -0.125, np.float32)
    elif kind == "clustered":  # the equal values in a few neighbouring places
        w = rng.standard_normal(n).astype(np.float32)
        for c in (0, 16380, 16384, n - 3):
            w[max(0, min(c, n)):max(0, min(c + 9, n))] = 0.5
    else:
        w = rng.permutation(n).astype(np.float32) - n // 2
    order = np.argsort(w, kind="stable")
    srt = w[order]
    runs = np.flatnonzero(np.r_[True, srt[1:] != srt[:-1]])  # -0.0 == 0.0
    ends = np.r_[runs[1:], n]
    longest = np.argsort(ends - runs)[-4:]
    splits = {0, n - 1, n // 2}
    for r in longest:
        a, b = int(runs[r]), int(ends[r])
        splits |= {a, min(a + 1, b - 1), (a + b) // 2, b - 1, int(rng.integers(a, b))}
        # the first kept one at a segment's edge in index order
        idx = order[a:b]
        for edge in (16383, 16384, 32767, 32768, (n - 1) // 16384 * 16384):
            p = int(np.searchsorted(idx, edge))
            if p < b - a:
                splits.add(a + p)
    for split in sorted(splits):
        ref = np.zeros(n, np.uint8)
        ref[order[split:]] = 1
        assert np.array_equal(_mask_at(L, w, srt, split), ref), split
    # the sort by key bits has -0.0 before +0.0; and pointers that allow no 4-value accesses
    bits = np.sort(w.view(np.int32) ^ ((w.view(np.int32) >> 31) & 0x7FFFFFFF))
    by_bits = (bits ^ ((bits >> 31) & 0x7FFFFFFF)).view(np.float32)
    for shift in (1, 2, 3):
        assert np.array_equal(_mask_at(L, w, by_bits, split, shift), ref)


@pytest.mark.parametrize("n", [1, 2, 257, 65537])
@pytest.mark.parametrize("bad", [(np.inf,), (-np.inf,), (np.inf, -np.inf), (np.nan,), (-np.nan,),
                                 (np.inf, np.nan)])
def test_jenks2_gpu_rejects_nonfinite(n, bad):
    """Wherever they stand, infinities and NaN raise, as on the host; the largest finite values do
    not."""
    rng = np.random.default_rng(n)
    for at in {0, n // 2, n - 1}:
        w = rng.standard_normal(n).astype(np.float32)
        for i, v in enumerate(bad):
            w[(at + i) % n] = v
        for fn in (C.jenks2_gpu, linear_mask, bias_mask):
            with pytest.raises(RuntimeError):
                fn(torch.from_numpy(w).to(DEV))
        with pytest.raises(RuntimeError):
            C.jenks2_host(torch.from_numpy(w))
    w = np.where(rng.random(n) < 0.5, 3.4028234e38, -3.4028234e38).astype(np.float32)
    kh, sh, gh = C.jenks2_host(torch.from_numpy(w))
    kg, sg, gg = C.jenks2_gpu(torch.from_numpy(w).to(DEV))
    assert sg == sh and gg == gh and torch.equal(kg.cpu(), kh)


@pytest.mark.parametrize("n", [3, 255, 65537])
def test_jenks2_gpu_takes_any_address(n):
    """A view that starts 4 bytes into its buffer."""
    w = torch.randn(n + 1) * 0.02
    kh, sh, gh = C.jenks2_host(w[1:].contiguous())
    kg, sg, gg = C.jenks2_gpu(w.to(DEV)[1:])
    assert sg == sh and gg == gh and torch.equal(kg.cpu(), kh)
