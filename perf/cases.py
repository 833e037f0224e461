"""What this framework is timed on: the 4-bit linear layer in every way a program calls it
(one token, a small batch, a prompt, a training step), the GPU packer that makes its weights
and the pruning mask over a whole weight matrix.

The layer shapes are the benchmark's (the 4096 / 11008 and 8192 / 28672 projections and the
784 -> 300 layer of the pruned LeNet300); ``draw`` spreads sizes, formats and activation
types over the same ranges.  Layers are built the way a packed checkpoint is loaded: codes
and codebooks (or scales) go into ``QuantLinear(pack=False)`` through ``load_state_dict``,
drawn with the distribution that packing normally distributed weights gives.
"""
from __future__ import annotations

import math

import torch

from if_i_could_turn_back_time_amd import PackedWeight, QuantLinear, linear_mask

DEV = "cuda"
DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIGMA = 0.02
# the 16 centroids of a unit normal's optimal 16-class partition (Lloyd-Max), positive half
_HALF = [0.1284, 0.3881, 0.6568, 0.9424, 1.2562, 1.6181, 2.0690, 2.7326]
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]
MOST_MACS = 2048 * 8192 * 28672


def _linear(name, fmt, K, N, M, xdt, rot=0, bias=False, fp4=False):
    return {"name": name, "kind": "linear", "fmt": fmt, "K": K, "N": N, "M": M, "xdt": xdt,
            "rot": rot, "bias": bias, "fp4": fp4}


def listed():
    return [
        # the first layer of the pruned LeNet300 on one image: fp32 activations as its
        # program has them, in_features that need padding, a bias; all launch cost
        _linear("lenet_784x300_m1", "gf4", 784, 300, 1, "f32", bias=True),
        # one decoded token through a 7B model's attention projection
        _linear("gf4_4096x4096_m1", "gf4", 4096, 4096, 1, "f16"),
        # one decoded token through a 70B model's MLP: the headline benchmark's layer
        _linear("gf4_8192x28672_m1", "gf4", 8192, 28672, 1, "f16"),
        # the same through a rotated 7B MLP layer
        _linear("gf4rot_4096x11008_m1", "gf4", 4096, 11008, 1, "f16", rot=4096),
        # sixteen sequences decoded together, OCP MXFP4 weights
        _linear("e2m1_8192x28672_m16", "e2m1", 8192, 28672, 16, "bf16"),
        # a prompt of 512 tokens through a 7B MLP layer
        _linear("gf4_4096x11008_m512", "gf4", 4096, 11008, 512, "f16"),
        # a prompt of odd length through the down projection, with a bias
        _linear("e2m1_11008x4096_m333", "e2m1", 11008, 4096, 333, "bf16", bias=True),
        # a short prompt on the native FP4 option
        _linear("e2m1fp4_8192x8192_m96", "e2m1", 8192, 8192, 96, "bf16", fp4=True),
        # a long prompt (or several) through a rotated 70B MLP layer: the largest call
        _linear("gf4rot_8192x28672_m2048", "gf4", 8192, 28672, 2048, "f16", rot=4096),
        # one calibration / fine-tuning step below a frozen 4-bit layer: forward, then the
        # gradient of the activations and of the bias
        {"name": "train_gf4_4096x4096_m256", "kind": "train", "fmt": "gf4", "K": 4096,
         "N": 4096, "M": 256, "xdt": "f16", "rot": 0, "bias": True},
        # packing a projection on the GPU
        {"name": "pack_gf4_4096x4096", "kind": "pack", "fmt": "gf4", "K": 4096, "N": 4096},
        # the pruning mask of a projection
        {"name": "mask_4096x4096", "kind": "mask", "rows": 4096, "cols": 4096},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "train", "pack",
                       "mask"])
    if kind == "pack":
        fmt = rng.choice(["gf4", "gf4", "e2m1"])
        K = 128 * _log(rng, 4, 64)
        return {"kind": "pack", "fmt": fmt, "K": K, "N": _log(rng, 300, max(301, (1 << 25) // K))}
    if kind == "mask":
        cols = _log(rng, 300, 8192)
        return {"kind": "mask", "rows": _log(rng, 300, max(301, (1 << 25) // cols)), "cols": cols}
    fmt = rng.choice(["gf4", "e2m1"])
    xdt = rng.choice(["f16", "f16", "bf16", "f32"] if fmt == "gf4" else ["bf16", "bf16", "f16"])
    rot = rng.choice([0, 0, 0, 256, 1024, 4096]) if fmt == "gf4" else 0
    fp4 = kind != "train" and fmt == "e2m1" and rng.random() < 0.25
    if kind == "decode":
        M, lo, hi = rng.choice([1, 1, 1, 2, 3, 4, 6, 8, 13, 16]), 300, 28672
    elif kind == "prefill":
        M, lo, hi = _log(rng, 17, 2048), 1024, 28672
    else:
        M, lo, hi = _log(rng, 17, 1024), 784, 11008
    K = _log(rng, lo, hi)
    if rot:  # a rotation takes whole blocks
        K = max(rot, K // rot * rot)
    elif rng.random() < 0.7:  # most layers are a multiple of the group wide, some are not
        K = max(256, K // 128 * 128)
    most = 8192 * 28672 if kind == "decode" else MOST_MACS // 2 // M
    N = _log(rng, lo, min(hi, max(lo + 1, most // K)))
    if rng.random() < 0.6:
        N = max(16, N // 16 * 16)
    if kind == "train":
        return {"kind": "train", "fmt": fmt, "K": K, "N": N, "M": M, "xdt": xdt, "rot": rot,
                "bias": True}
    return {"kind": "linear", "fmt": fmt, "K": K, "N": N, "M": M, "xdt": xdt, "rot": rot,
            "bias": rng.random() < 0.3, "fp4": fp4}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _packed(case, g):
    """Codes uint8 [N, K'/2] and codebooks int16 [N, K'/128, 16] or scales uint8 [N, K'/32]
    of a packed weight, K' = K rounded up to whole groups."""
    N, K = case["N"], (case["K"] + 127) // 128 * 128
    codes = torch.empty(N, K // 2, dtype=torch.uint8, device=DEV)
    step = max(1, (1 << 25) // K)
    half = torch.tensor(_HALF, device=DEV)
    if case["fmt"] == "gf4":
        cent = torch.cat([-half.flip(0), half])
        meta = torch.empty(N, K // 128, 16, dtype=torch.int16, device=DEV)
    else:
        cent = torch.tensor(_E2M1, device=DEV)
        meta = torch.empty(N, K // 32, dtype=torch.uint8, device=DEV)
    mids = (cent[1:] + cent[:-1]) / 2
    for r0 in range(0, N, step):
        r1 = min(N, r0 + step)
        z = torch.randn(r1 - r0, K, generator=g, device=DEV)
        if case["fmt"] == "gf4":
            c = torch.bucketize(z, mids).to(torch.uint8)
            # each group's codebook: the normal centroids, moved as 128 samples move them
            spread = 1 + 0.06 * torch.randn(r1 - r0, K // 128, 1, generator=g, device=DEV)
            book = cent * spread + 0.03 * torch.randn(r1 - r0, K // 128, 16, generator=g,
                                                      device=DEV)
            meta[r0:r1] = (SIGMA * book.sort(-1).values).half().view(torch.int16)
        else:
            # a 32-group's largest value (about 2.1 sigma on average, 1.3 to 5) sets its scale
            amax = z.abs().reshape(r1 - r0, -1, 32).amax(-1, keepdim=True)
            e = torch.floor(torch.log2(SIGMA * amax)) - 2
            q = (SIGMA * z.reshape(r1 - r0, -1, 32) * torch.exp2(-e)).reshape(r1 - r0, K)
            c = (torch.bucketize(q.abs(), mids) + 8 * (q < 0)).to(torch.uint8)
            meta[r0:r1] = (e.squeeze(-1) + 127).to(torch.uint8)
        codes[r0:r1] = c[:, ::2] | (c[:, 1::2] << 4)
    return codes, meta


def _inputs(case, seed):
    g = _gen(seed)
    codes, meta = _packed(case, g)
    M, N, K, xdt = case["M"], case["N"], case["K"], DT[case["xdt"]]
    x = torch.randn(M, K, generator=g, device=DEV)
    x[:, torch.randperm(K, generator=g, device=DEV)[:max(1, K // 1000)]] *= 20  # outlier channels
    bias = 0.1 * torch.randn(N, generator=g, device=DEV) if case["bias"] else None
    gy = torch.randn(M, N, generator=g, device=DEV) / M if case["kind"] == "train" else None
    return codes, meta, x.to(xdt), bias, None if gy is None else gy.to(xdt)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pack":
        w = SIGMA * torch.randn(case["N"], case["K"], generator=_gen(seed), device=DEV)
        return {"kind": kind, "fmt": case["fmt"], "w": w}
    if kind == "mask":
        w = SIGMA * torch.randn(case["rows"], case["cols"], generator=_gen(seed), device=DEV)
        return {"kind": kind, "w": w}
    codes, meta, x, bias, gy = _inputs(case, seed)
    fp4 = bool(case.get("fp4"))
    with torch.device(DEV):
        lin = torch.nn.utils.skip_init(torch.nn.Linear, case["K"], case["N"],
                                       bias=bias is not None, device=DEV)
        layer = QuantLinear(lin, fmt=case["fmt"], hadamard=case["rot"], pack=False, fp4_mfma=fp4)
    del lin
    book = meta.view(torch.uint8) if case["fmt"] == "e2m1" else meta
    state = {"codes": codes, "meta": book, "fb_header": layer.fb_header}
    if bias is not None:
        state["bias"] = bias
    layer.load_state_dict(state, strict=False)
    if kind == "train":
        x.requires_grad_(True)
    return {"kind": kind, "layer": layer, "x": x, "gy": gy}


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "pack":
        pw = PackedWeight.quantize(state["w"], state["fmt"], device=state["w"].device,
                                   packer="gpu")
        return {"codes": pw.codes, "meta": pw.meta, "wdev": pw.wdev}
    if kind == "mask":
        mask, gvf = linear_mask(state["w"])
        return {"mask": mask, "gvf": gvf}
    layer, x = state["layer"], state["x"]
    if kind == "train":
        y = layer(x)
        gx, gb = torch.autograd.grad(y, (x, layer.bias), state["gy"])
        return {"y": y.detach(), "grad_x": gx, "grad_bias": gb}
    with torch.no_grad():
        return layer(x)


# ------------------------------------------------------------------ what it cannot do without
def work(case):
    kind = case["kind"]
    if kind == "mask":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n + 4 * n, "flops": 10 * n}
    N, K = case["N"], case["K"]
    kp = (K + 127) // 128 * 128
    packed = N * kp // 2 + (N * (kp // 128) * 32 if case["fmt"] == "gf4" else N * (kp // 32))
    if kind == "pack":  # codes, codebooks or scales, and the same in the kernels' layout
        # gf4: every class break of every prefix of a sorted 128-group
        return {"bytes": 4 * N * K + 2 * packed,
                "flops": N * K * (15 * 64 * 2 if case["fmt"] == "gf4" else 10)}
    M, e = case["M"], 4 if case["xdt"] == "f32" else 2
    b = packed + M * K * e + M * N * e + (4 * N if case["bias"] else 0)
    f = 2 * M * N * K
    if case["rot"]:
        f += M * K * int(math.log2(case["rot"]))
    if kind == "train":  # gy and the weight again, grad_x, grad_bias
        b += packed + M * N * e + M * K * e + 4 * N
        f = 2 * f + M * N
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] in ("pack", "mask"):
        return "exact"
    # what the output's type gives (about half an ulp of rounding, with another order of
    # the fp32 sums moving some results to the neighbouring value); a rotated x is held in
    # fp16, so one rounding of it may fall the other way
    rel = {"f16": 1e-3, "bf16": 8e-3, "f32": 1e-5}[case["xdt"]]
    if case["rot"]:
        rel = max(rel, 1.5e-3)
    return {"rel": rel}


# ------------------------------------------------------------------ the same in 64 bits
def _decode(case, codes, meta):
    c = torch.stack((codes & 15, codes >> 4), dim=-1).reshape(codes.shape[0], -1)
    if case["fmt"] == "gf4":
        book = meta.view(torch.float16).double()
        n, g = book.shape[:2]
        w = torch.empty(n, g, 128, dtype=torch.float64, device=codes.device)
        step = max(1, (1 << 26) // (g * 128))
        for r in range(0, n, step):  # the gather's 64-bit indices are large
            w[r:r + step] = book[r:r + step].gather(
                -1, c[r:r + step].reshape(-1, g, 128).long())
        w = w.reshape(n, -1)
    else:
        grid = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=codes.device)
        w = torch.empty(c.shape, dtype=torch.float64, device=codes.device)
        step = max(1, (1 << 26) // c.shape[1])
        for r in range(0, c.shape[0], step):
            w[r:r + step] = grid[c[r:r + step].int()]
        w.view(w.shape[0], -1, 32).mul_(torch.exp2(meta.double() - 127)[..., None])
    return w[:, :case["K"]]


def _rotate(v, block):
    shape, h = v.shape, 1
    while h < block:
        v = v.reshape(-1, 2, h)
        v = torch.stack((v[:, 0] + v[:, 1], v[:, 0] - v[:, 1]), dim=1)
        h *= 2
    return v.reshape(shape) / math.sqrt(block)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("pack", "mask"):  # whole values (and one ratio of sums that decides them)
        return None
    codes, meta, x, bias, gy = _inputs(case, seed)
    w = _decode(case, codes, meta)
    xr = x.double()
    if case["rot"]:
        xr = _rotate(xr, case["rot"])
    y = xr @ w.T
    if bias is not None:
        y += bias.double()
    if kind != "train":
        return y
    gx = gy.double() @ w
    if case["rot"]:
        gx = _rotate(gx, case["rot"])
    return {"y": y, "grad_x": gx, "grad_bias": gy.double().sum(0)}
