"""The GPU packers' class search and the GPU form of fb_to_device against the host's bytes."""
import pytest
import torch

from if_i_could_turn_back_time_amd import PackedWeight, QuantLinear, _capi as C

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("kind", ["normal", "heavy", "few values", "tiny", "wide", "masked"])
def test_gf4_classes_over_many_groups(kind):
    """16-class breaks of 6,144 groups a kind: the division by reciprocal and the order of the
    candidates decide near-ties, so every byte is compared."""
    print("pack", kind, flush=True)
    g = torch.Generator().manual_seed(len(kind))
    w = torch.randn(768, 1024, generator=g)
    keep = None
    if kind == "heavy":
        w = w / torch.randn(768, 1024, generator=g).abs().clamp_min(1e-3)
    elif kind == "few values":
        w = (w * 3).round() / 8
    elif kind == "tiny":
        w = w * 1e-42  # fp32 subnormals
    elif kind == "wide":
        w = w * 10.0 ** torch.randint(-30, 31, w.shape, generator=g)
    elif kind == "masked":
        keep = torch.rand(768, 1024, generator=g) < torch.rand(768, 1, generator=g)
    hc, hb = C.quantize_gf4(w, 8, keep)
    dc, db = C.quantize_gf4_gpu(w.to(DEV), None if keep is None else keep.to(DEV))
    assert torch.equal(dc.cpu(), hc) and torch.equal(db.cpu(), hb)


@pytest.mark.parametrize("fmt", ["gf4", "e2m1"])
@pytest.mark.parametrize("N,K", [(1, 128), (15, 384), (16, 512), (17, 640), (100, 1152), (65, 4224)])
def test_layout_on_the_gpu_is_the_hosts(fmt, N, K):
    g = torch.Generator().manual_seed(N)
    codes = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
    meta = (torch.randint(-2**15, 2**15, (N, K // 128, 16), generator=g, dtype=torch.int16)
            if fmt == "gf4" else
            torch.randint(0, 256, (N, K // 32), generator=g, dtype=torch.uint8))
    shape = C.make_shape(N, K, 1, C.FMT_BY_NAME[fmt])
    dev = C.to_device_layout_gpu(codes.to(DEV), meta.to(DEV), shape)
    assert torch.equal(dev.cpu(), C.to_device_layout(codes, meta, shape))


@pytest.mark.parametrize("fmt", ["gf4", "e2m1"])
@pytest.mark.parametrize("device", [None, DEV])
def test_quantize_on_gpu_or_cpu_weights(fmt, device):
    """packer='gpu' takes w from either side and leaves the stream where packer='host' does."""
    g = torch.Generator().manual_seed(2)
    w = torch.randn(40, 256, generator=g) * 0.02
    host = PackedWeight.quantize(w, fmt, device=device)
    for src in (w, w.to(DEV), w.to(DEV).t().contiguous().t()):
        pw = PackedWeight.quantize(src, fmt, device=device, packer="gpu")
        for a, b in ((pw.codes, host.codes), (pw.meta, host.meta), (pw.wdev, host.wdev)):
            assert a.device == b.device and torch.equal(a, b)


@pytest.mark.parametrize("kw", [dict(fmt="gf4"), dict(fmt="e2m1"), dict(fmt="gf4", hadamard=128)])
def test_checkpoint_loads_to_the_same_stream_on_gpu_and_cpu(kw):
    torch.manual_seed(3)
    lin = torch.nn.Linear(384 if "hadamard" in kw else 300, 70)
    src = QuantLinear(lin, **kw)
    for dev in ("cpu", DEV):
        q = QuantLinear(lin, pack=False).to(dev)
        q.load_state_dict(src.state_dict())
        assert q.wdev.device.type == torch.device(dev).type
        assert torch.equal(q.wdev.cpu(), src.wdev) and q._f16_exact == src._f16_exact


@pytest.mark.parametrize("fmt", ["gf4", "e2m1"])
@pytest.mark.parametrize("offset", [1, 2, 4, 8, 16])
def test_checkpoint_of_views_loads_at_any_offset(fmt, offset):
    """load_state_dict(assign=True) keeps views of one flat buffer, at addresses that are no
    multiple of 16 (codebooks: of 2 at least)."""
    lin = torch.nn.Linear(300, 70)
    src = QuantLinear(lin, fmt=fmt)
    sd = {k: v.to(DEV) for k, v in src.state_dict().items()}
    for name in ("codes", "meta"):
        t = sd[name]
        at = offset * t.element_size()
        flat = torch.zeros(at + t.numel() * t.element_size(), dtype=torch.uint8, device=DEV)
        sd[name] = flat[at:].view(t.dtype).view(t.shape).copy_(t)
    q = QuantLinear(lin, pack=False).to(DEV)
    q.load_state_dict(sd, assign=True)
    assert q.codes.data_ptr() % 16 == offset % 16
    assert torch.equal(q.wdev.cpu(), src.wdev)
