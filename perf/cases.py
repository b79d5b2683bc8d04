"""The calls that a user of this package makes, as measurable cases over their real ranges.

Five kinds of call, each through the public entry point that a program uses:

* ``attn``    FlashDeformAttnFunction: multi-scale deformable attention over 3-D volumes, the main
              path (training step, or forward alone for inference);
* ``offsets`` FlashDeformAttnFromOffsets: the same with locations formed from a projection's
              offsets and fp32 reference points (what the FlashDeformAttn3D module calls);
* ``dcn``     dcnv4_3d: deformable 3-D convolution;
* ``roi``     roi_align_3d: region features of detected boxes;
* ``nms``     nms_nd: greedy suppression of scored boxes.

A case is a dict of plain values.  ``train`` says whether the pass is forward and backward
(gradients returned) or the forward alone.  Levels are written "16x32x128,8x16x64" (D x H x W,
finest first); ``queries`` 0 means self-attention (one query per voxel of every level).
"""
from __future__ import annotations

import math

import torch

from ops3d_amd import FlashDeformAttnFromOffsets, FlashDeformAttnFunction
from ops3d_amd.dcnv4 import dcnv4_3d
from ops3d_amd.nms import nms_nd
from ops3d_amd.roi_align import roi_align_3d

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
IM2COL_STEP = 64


def _attn(name, levels, dtype, train, batch=1, queries=0, heads=8, channels=32, points=4, outside=0.0,
          kind="attn", ref_levels=1):
    return {"name": name, "kind": kind, "levels": levels, "dtype": dtype, "train": train, "batch": batch,
            "queries": queries, "heads": heads, "channels": channels, "points": points, "outside": outside,
            "ref_levels": ref_levels}


def _roi(name, size, dtype, train, batch, channels, rois, pooled, ratio, order=1, scale=1.0, min_ext=4.0,
         max_ext=32.0):
    return {"name": name, "kind": "roi", "size": size, "dtype": dtype, "train": train, "batch": batch,
            "channels": channels, "rois": rois, "pooled": pooled, "ratio": ratio, "order": order, "scale": scale,
            "min_ext": min_ext, "max_ext": max_ext}


def _dcn(name, size, dtype, train, batch, heads, channels, kernel=3, stride=1, dilation=1, remove_center=False,
         softmax=True, offset_scale=1.0):
    return {"name": name, "kind": "dcn", "size": size, "dtype": dtype, "train": train, "batch": batch,
            "heads": heads, "channels": channels, "kernel": kernel, "stride": stride, "dilation": dilation,
            "remove_center": remove_center, "softmax": softmax, "offset_scale": offset_scale}


def _nms(name, boxes, side, threshold):
    return {"name": name, "kind": "nms", "boxes": boxes, "side": side, "threshold": threshold}


def listed():
    return [
        # the smallest calls: a training step on a tiny crop, where launches and host time count
        _attn("attn_tiny_fp32_train", "4x8x16,2x4x8", "fp32", True),
        # a decoder's cross-attention: few object queries over a three-level volume, some samples
        # outside it
        _attn("attn_cross_bf16_train", "16x32x64,8x16x32,4x8x16", "bf16", True, batch=2, queries=200, outside=0.1),
        # an encoder layer's self-attention over a tiled light-sheet volume at strides 16 and 32
        _attn("attn_self_bf16_train", "16x32x128,8x16x64", "bf16", True),
        # the same at strides 8, 16 and 32: the largest training step
        _attn("attn_large_bf16_train", "32x64x256,16x32x128,8x16x64", "bf16", True),
        # a ragged volume in full precision, 6 heads of 48 channels, a batch of two crops
        _attn("attn_ragged_fp32_train", "11x27x45,6x14x23,3x7x12", "fp32", True, batch=2, heads=6, channels=48),
        # inference in half precision: wide heads, four odd levels, eight points
        _attn("attn_ragged_fp16_infer", "13x37x61,7x19x31,4x10x16,2x5x8", "fp16", False, channels=64, points=8),
        # the attention module's own step: offsets from a projection, gradients of the reference
        # points too
        _attn("offsets_self_bf16_train", "16x32x128,8x16x64", "bf16", True, kind="offsets"),
        # a deformable convolution block of a 3-D backbone, training
        _dcn("dcn_block_bf16_train", "32x64x64", "bf16", True, 2, 8, 32),
        # region features of a detector, training
        _roi("roi_head_bf16_train", "32x64x64", "bf16", True, 2, 256, 512, 7, 2),
        # the same at inference: full precision, an odd volume at half scale, adaptive sampling
        _roi("roi_adaptive_fp32_infer", "21x45x77", "fp32", False, 1, 120, 150, 7, 0, scale=0.5, min_ext=8.0,
             max_ext=48.0),
        # suppression of one crop's boxes
        _nms("nms_crop", 4096, 100.0, 0.3),
        # suppression of a whole volume's boxes
        _nms("nms_volume", 50001, 230.0, 0.3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _volume(rng, voxels):
    """A box of about `voxels` voxels, flatter in z than in x, odd sizes as they come."""
    side = voxels ** (1.0 / 3.0)
    d = max(2, int(round(side * rng.uniform(0.35, 0.9))))
    h = max(2, int(round(side * rng.uniform(0.7, 1.2))))
    return d, h, max(2, int(round(voxels / (d * h))))


def _pyramid(rng, voxels, levels):
    d, h, w = _volume(rng, voxels)
    out = []
    for _ in range(levels):
        out.append("%dx%dx%d" % (d, h, w))
        d, h, w = (d + 1) // 2, (h + 1) // 2, (w + 1) // 2
    return ",".join(out)


def draw(rng):
    case = _drawn(rng)
    del case["name"]
    return case


def _drawn(rng):
    kind = rng.choices(["attn", "offsets", "dcn", "roi", "nms"], weights=[8, 3, 3, 4, 3])[0]
    if kind in ("attn", "offsets"):
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        channels = rng.choice([16, 32, 32, 32, 48, 64])
        heads = rng.choice([4, 6, 8, 8, 8])
        points = rng.choice([4, 4, 4, 8])
        levels = rng.choice([1, 2, 2, 3, 3, 4])
        cross = rng.random() < 0.25
        # below the largest listed step: under half of its sample rows times channels in 16 bits
        most = 250000 * 8 * 32 * 12 / (heads * channels * points * levels * (2 if dtype == "fp32" else 1))
        voxels = _log_int(rng, 500, min(480000, most))
        return _attn("", _pyramid(rng, voxels, levels), dtype, rng.random() < 0.75,
                     batch=rng.choice([1, 2]) if voxels < 100000 else 1,
                     queries=_log_int(rng, 50, 900) if cross else 0, heads=heads, channels=channels, points=points,
                     outside=0.1 if cross else 0.0, kind=kind, ref_levels=rng.choice([1, levels]))
    if kind == "dcn":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        voxels = _log_int(rng, 1000, 110000 if dtype != "fp32" else 50000)
        return _dcn("", "%dx%dx%d" % _volume(rng, voxels), dtype, rng.random() < 0.7, rng.choice([1, 2]),
                    rng.choice([4, 8]), rng.choice([16, 32]), stride=rng.choice([1, 1, 2]),
                    dilation=rng.choice([1, 1, 2]), remove_center=rng.random() < 0.25, softmax=rng.random() < 0.6)
    if kind == "roi":
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        voxels = _log_int(rng, 8000, 130000)
        d, h, w = _volume(rng, voxels)
        scale = rng.choice([1.0, 0.5, 0.25])
        low = rng.uniform(2.0, 5.0)
        order = rng.choice([1, 1, 1, 0])   # nearest takes one sample per bin, as the RoIAlign module has it
        return _roi("", "%dx%dx%d" % (d, h, w), dtype, rng.random() < 0.6, rng.choice([1, 2]),
                    rng.choice([32, 64, 96, 128, 250, 256]), _log_int(rng, 16, 512), rng.choice([3, 5, 7, 7]),
                    rng.choice([0, 2, 2, 3]) if order else 1, order=order, scale=scale, min_ext=low / scale,
                    max_ext=max(low + 1.0, 0.8 * min(d, h, w)) / scale)
    boxes = _log_int(rng, 50, 60000)
    return _nms("", boxes, round(100.0 * (boxes / 4096.0) ** (1.0 / 3.0) * rng.uniform(0.7, 1.4), 3),
                rng.choice([0.1, 0.25, 0.3, 0.5]))


# ---------------------------------------------------------------------------- inputs


def _sizes(text):
    return [tuple(int(v) for v in s.split("x")) for s in text.split(",")]


def _shape(case):
    """B, S, Q, G, D, L, K and the levels of an attn / offsets case."""
    levels = _sizes(case["levels"])
    S = sum(d * h * w for d, h, w in levels)
    return case["batch"], S, case["queries"] or S, case["heads"], case["channels"], len(levels), case["points"], levels


def _dcn_geometry(case):
    size = _sizes(case["size"])[0]
    k, s, dil = case["kernel"], case["stride"], case["dilation"]
    pad = dil * (k - 1) // 2
    out = tuple((n + 2 * pad - (dil * (k - 1) + 1)) // s + 1 for n in size)
    taps = k ** 3 - (1 if case["remove_center"] else 0)
    padded = (case["heads"] * 4 * taps + 7) // 8 * 8
    return size, out, pad, taps, padded


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device=dev)

    if kind == "nms":
        n, side = case["boxes"], case["side"]
        clusters = max(1, n // 20)
        centre = rand(clusters, 3) * side
        pick = torch.randint(0, clusters, (n,), generator=g, device=dev)
        c = centre[pick] + 3.0 * randn(n, 3)
        e = 2.0 + 10.0 * rand(n, 3)
        score = torch.round(rand(n, 1) * 1000.0) / 1000.0
        return {"case": case, "dets": torch.cat([c - e / 2, c + e / 2, score], 1).contiguous(),
                "kept": torch.empty(n, dtype=torch.int64, device=dev)}

    dt = DTYPES[case["dtype"]]
    train = case["train"]
    if kind in ("attn", "offsets"):
        B, S, Q, G, D, L, K, levels = _shape(case)
        n = L * K
        st = {"case": case, "shapes": torch.tensor(levels, dtype=torch.int64, device=dev)}
        counts = [d * h * w for d, h, w in levels]
        st["starts"] = torch.tensor([sum(counts[:i]) for i in range(L)], dtype=torch.int64, device=dev)
        st["value"] = randn(B, S, G, D).to(dt).requires_grad_(train)
        logits = randn(B, Q, G, n)
        if kind == "attn":
            loc = rand(B, Q, G, n, 3)
            if case["outside"] > 0:
                wide = rand(B, Q, G, n, 3) * 1.2 - 0.1
                loc = torch.where(rand(B, Q, G, n, 1) < case["outside"], wide, loc)
            rows = loc.reshape(B, Q, G, 3 * n)
        else:
            rows = 2.0 * randn(B, Q, G, 3 * n)   # voxels
            st["ref"] = rand(B, Q, case["ref_levels"], 3).requires_grad_(train)
        st["packed"] = torch.cat([rows, logits], -1).to(dt).contiguous().requires_grad_(train)
        if train:
            st["grad"] = randn(B, Q, G * D).to(dt)
        return st
    if kind == "dcn":
        size, out, _, taps, padded = _dcn_geometry(case)
        B, G, D = case["batch"], case["heads"], case["channels"]
        st = {"case": case, "value": randn(B, *size, G * D).to(dt).requires_grad_(train),
              "offset": randn(B, *out, padded).to(dt).requires_grad_(train)}
        if train:
            st["grad"] = randn(B, *out, G * D).to(dt)
        return st
    size = _sizes(case["size"])[0]
    N, C, R, p = case["batch"], case["channels"], case["rois"], case["pooled"]
    st = {"case": case, "features": randn(N, C, *size).to(dt).requires_grad_(train)}
    whole = torch.tensor([size[2], size[1], size[0]], dtype=torch.float32, device=dev) / case["scale"]
    ext = torch.minimum(case["min_ext"] + (case["max_ext"] - case["min_ext"]) * rand(R, 3), whole)
    lo = rand(R, 3) * (whole - ext)
    item = torch.randint(0, N, (R, 1), generator=g, device=dev).float()
    st["rois"] = torch.cat([item, lo, lo + ext], 1).to(dt)
    if train:
        st["grad"] = randn(R, C, p, p, p).to(dt)
    return st


# ---------------------------------------------------------------------------- one pass


def _call(st):
    """The entry point's output, and the tensors whose gradients a training step takes."""
    case = st["case"]
    kind = case["kind"]
    if kind == "attn":
        out = FlashDeformAttnFunction.apply(st["value"], st["shapes"], st["starts"], st["packed"], IM2COL_STEP,
                                            case["points"], True)
        return out, (st["value"], st["packed"])
    if kind == "offsets":
        out = FlashDeformAttnFromOffsets.apply(st["value"], st["shapes"], st["starts"], st["packed"], st["ref"],
                                               IM2COL_STEP, case["points"])
        return out, (st["value"], st["packed"], st["ref"])
    if kind == "dcn":
        k, s, dil = case["kernel"], case["stride"], case["dilation"]
        pad = _dcn_geometry(case)[2]
        out = dcnv4_3d(st["value"], st["offset"], (k, k, k), (s, s, s), (pad, pad, pad), (dil, dil, dil),
                       case["heads"], case["channels"], case["offset_scale"], IM2COL_STEP,
                       1 if case["remove_center"] else 0, case["softmax"])
        return out, (st["value"], st["offset"])
    p = case["pooled"]
    return roi_align_3d(st["features"], st["rois"], (p, p, p), case["scale"], case["ratio"], case["order"]), (
        st["features"],)


def run(st):
    case = st["case"]
    if case["kind"] == "nms":   # the kept boxes in score order, padded to a fixed length
        keep = nms_nd(st["dets"], case["threshold"])[0]
        st["kept"].fill_(-1)[:keep.shape[0]] = keep
        return st["kept"]
    if not case["train"]:
        with torch.no_grad():
            return _call(st)[0]
    out, leaves = _call(st)
    return (out.detach(), *torch.autograd.grad(out, leaves, st["grad"]))


# ---------------------------------------------------------------------------- what a pass needs


def work(case):
    """Every input read once and every output written once; two operations per multiply-add of the
    interpolation (8 corners of a sample, and in a training step twice that again for the corner
    products and the values' gradient; RoI: the two nearest voxels per axis and bin; NMS: none of
    the pairs has to be looked at, so the boxes themselves)."""
    kind = case["kind"]
    if kind == "nms":
        n = case["boxes"]
        return {"bytes": 28 * n + 8 * n, "flops": 20 * n}
    e = 4 if case["dtype"] == "fp32" else 2
    train = case["train"]
    if kind in ("attn", "offsets"):
        B, S, Q, G, D, L, K, _ = _shape(case)
        v, r, o = B * S * G * D, B * Q * G * 4 * L * K, B * Q * G * D
        ref = B * Q * case["ref_levels"] * 12 if kind == "offsets" else 0
        rows = B * Q * G * L * K * 8 * D
    elif kind == "dcn":
        size, out, _, taps, padded = _dcn_geometry(case)
        B, G, D = case["batch"], case["heads"], case["channels"]
        q = B * out[0] * out[1] * out[2]
        v, r, o, ref = B * size[0] * size[1] * size[2] * G * D, q * padded, q * G * D, 0
        rows = q * G * taps * 8 * D
    else:
        size = _sizes(case["size"])[0]
        v = case["batch"] * case["channels"] * size[0] * size[1] * size[2]
        o = case["rois"] * case["channels"] * case["pooled"] ** 3
        r, ref, rows = 7 * case["rois"], 0, 8 * o
        if train:   # features' gradient written, the output's read
            return {"bytes": e * (v + o + r) + e * (v + o + r), "flops": 2 * 2 * rows}
    fwd = e * (v + r + o) + ref
    if not train:
        return {"bytes": fwd, "flops": 2 * rows}
    return {"bytes": fwd + e * (2 * v + 2 * r + o) + 2 * ref, "flops": 3 * 2 * rows}


def tolerance(case):
    """About four times the distance from exact(), which is the rounding of the results (all sums are
    fp32): 1.7e-3 in bf16 and 2.1e-4 in fp16 wherever measured, at most 6.6e-7 in fp32 with its
    largest in the gradients summed over many samples, where the order of the sums counts."""
    if case["kind"] == "nms":
        return "exact"
    return {"rel": {"fp32": 4e-6, "fp16": 8.5e-4, "bf16": 7e-3}[case["dtype"]]}


# ---------------------------------------------------------------------------- in 64 bits


def _trilinear(value, size, pix):
    """value [V, D] float64 rows of a D x H x W volume, pix [n, 3] float64 (x, y, z) -> [n, D]; zero
    outside the volume, weights x - floor(x)."""
    d, h, w = size
    base = pix.detach().floor()
    frac = pix - base
    base = base.long()
    out = 0
    for corner in range(8):
        idx, wt, ok = 0, 1, True
        for axis, extent, stride in ((0, w, 1), (1, h, w), (2, d, w * h)):
            up = (corner >> axis) & 1
            i = base[:, axis] + up
            ok = ok & (i >= 0) & (i < extent)
            idx = idx + i.clamp(0, extent - 1) * stride
            wt = wt * (frac[:, axis] if up else 1 - frac[:, axis])
        out = out + value.index_select(0, idx) * (wt * ok).unsqueeze(1)
    return out


_EXACT_ROWS = 1 << 26   # sampled elements at a time (rows times channels)


def _deform_exact(value, levels, pixels, weights, grad):
    """value [S, D], weights [Q, n], both float64 and pixels a list (per level) of [Q, k, 3]: the
    weighted sum of the samples [Q, D], and with grad [Q, D] the gradients of value, pixels and
    weights."""
    S, D = value.shape
    Q, n = weights.shape
    out = value.new_empty(Q, D)
    train = grad is not None
    gv = torch.zeros_like(value) if train else None
    gp = [torch.empty_like(p) for p in pixels]
    gw = torch.empty_like(weights)
    step = max(1, _EXACT_ROWS // (n * D))
    for q0 in range(0, Q, step):
        q = slice(q0, min(q0 + step, Q))
        col, start, total = 0, 0, 0
        for size, pix, gpix in zip(levels, pixels, gp):
            count, k = size[0] * size[1] * size[2], pix.shape[1]
            v = value[start:start + count].detach().requires_grad_(train)
            p = pix[q].detach().requires_grad_(train)
            a = weights[q, col:col + k].detach().requires_grad_(train)
            with torch.set_grad_enabled(train):
                rows = _trilinear(v, size, p.reshape(-1, 3)).view(p.shape[0], k, D)
                o = (rows * a.unsqueeze(2)).sum(1)
            if train:
                dv, dp, da = torch.autograd.grad(o, (v, p, a), grad[q])
                gv[start:start + count] += dv
                gpix[q] = dp
                gw[q, col:col + k] = da
            total = total + o.detach()
            col, start = col + k, start + count
        out[q] = total
    return out, gv, gp, gw


def _softmax_backward(prob, grad):
    return prob * (grad - (prob * grad).sum(-1, keepdim=True))


def _exact_attn(st):
    """Sampling positions are rounded in fp32 as the operator defines them (grid_sample's steps on
    2 loc - 1; in offset mode loc = ref + offset / size first); everything after in 64 bits."""
    case = st["case"]
    B, S, Q, G, D, L, K, levels = _shape(case)
    n = L * K
    train, offsets = case["train"], case["kind"] == "offsets"
    value = st["value"].detach().double()
    rec = st["packed"].detach()
    logits = rec[..., 3 * n:].double()
    prob = torch.softmax(logits, -1)
    sizes = [torch.tensor([w, h, d], dtype=torch.float32, device=rec.device) for d, h, w in levels]
    grad = st["grad"].double().view(B, Q, G, D) if train else None
    out = value.new_empty(B, Q, G, D)
    if train:
        gvalue, grec = torch.empty_like(value), value.new_empty(rec.shape)
        gref = value.new_zeros(B, Q, case["ref_levels"], 3) if offsets else None
    for b in range(B):
        for h in range(G):
            pixels = []
            for lv in range(L):
                loc = rec[b, :, h, 3 * lv * K:3 * (lv + 1) * K].float().view(Q, K, 3)
                if offsets:
                    loc = st["ref"].detach()[b, :, min(lv, case["ref_levels"] - 1)].unsqueeze(1) + loc / sizes[lv]
                grid = 2.0 * loc - 1.0
                pixels.append((((grid + 1.0) * sizes[lv] - 1.0) / 2.0).double())
            o, gv, gp, gw = _deform_exact(value[b, :, h].contiguous(), levels, pixels, prob[b, :, h],
                                          grad[b, :, h].contiguous() if train else None)
            out[b, :, h] = o
            if train:
                gvalue[b, :, h] = gv
                grec[b, :, h, 3 * n:] = _softmax_backward(prob[b, :, h], gw)
                for lv in range(L):
                    gloc = gp[lv] * sizes[lv].double()
                    grec[b, :, h, 3 * lv * K:3 * (lv + 1) * K] = (gp[lv] if offsets else gloc).reshape(Q, 3 * K)
                    if offsets:
                        gref[b, :, min(lv, case["ref_levels"] - 1)] += gloc.sum(1)
    out = out.view(B, Q, G * D)
    if not train:
        return out
    return (out, gvalue, grec) + ((gref,) if offsets else ())


def _exact_dcn(st):
    """Positions rounded in fp32 step by step: (start - half * scale) + (tap + offset) * scale; a
    sample counts when every coordinate lies in (-1, size)."""
    case = st["case"]
    size, out_size, pad, K, padded = _dcn_geometry(case)
    B, G, D = case["batch"], case["heads"], case["channels"]
    k, stride, dil, train = case["kernel"], case["stride"], case["dilation"], case["train"]
    scale = torch.tensor(case["offset_scale"], dtype=torch.float32, device=st["value"].device)
    Q = out_size[0] * out_size[1] * out_size[2]
    value = st["value"].detach().double().view(B, -1, G, D)
    rec = st["offset"].detach()[..., :G * 4 * K].reshape(B, Q, G, 4 * K)
    dev = value.device
    half = (dil * (k - 1)) >> 1
    taps = [(i, j, t) for i in range(k) for j in range(k) for t in range(k)
            if not (case["remove_center"] and i == j == t == k // 2)]
    taps = torch.tensor(taps, dtype=torch.float32, device=dev) * dil
    zo, yo, xo = torch.meshgrid(*(torch.arange(s, device=dev) for s in out_size), indexing="ij")
    start = torch.stack([xo, yo, zo], -1).reshape(Q, 1, 3).float() * stride + float(half - pad) - float(half) * scale
    extent = torch.tensor([size[2], size[1], size[0]], dtype=torch.float32, device=dev)
    grad = st["grad"].double().view(B, Q, G, D) if train else None
    out = value.new_empty(B, Q, G, D)
    gvalue = torch.empty_like(value) if train else None
    grec = value.new_empty(B, Q, G, 4 * K) if train else None
    for b in range(B):
        for h in range(G):
            pix = start + (taps + rec[b, :, h, :3 * K].float().view(Q, K, 3)) * scale
            inside = ((pix > -1.0) & (pix < extent)).all(-1).double()
            mask = rec[b, :, h, 3 * K:].double()
            prob = torch.softmax(mask, -1) if case["softmax"] else mask
            o, gv, gp, gw = _deform_exact(value[b, :, h].contiguous(), [size], [pix.double()], prob * inside,
                                          grad[b, :, h].contiguous() if train else None)
            out[b, :, h] = o
            if train:
                gvalue[b, :, h] = gv
                gw = gw * inside
                grec[b, :, h, 3 * K:] = _softmax_backward(prob, gw) if case["softmax"] else gw
                grec[b, :, h, :3 * K] = (gp[0] * scale.double()).reshape(Q, 3 * K)
    out = out.view(B, *out_size, G * D)
    if not train:
        return out
    full = value.new_zeros(B, *out_size, padded)
    full[..., :G * 4 * K] = grec.view(B, *out_size, G * 4 * K)
    return out, gvalue.view(B, *size, G * D), full


def _axis_weights(lo, hi, size, p, ratio, order):
    """[R, p, size] float64: the averaged sample weights of every bin on every voxel of one axis;
    sample positions rounded in fp32 step by step."""
    extent = torch.clamp(hi - lo, min=1.0)
    step = extent / torch.full_like(extent, float(p))   # a division, not a product with 1 / p
    R = lo.shape[0]
    grid = torch.full((R,), float(ratio), device=lo.device) if ratio > 0 else torch.ceil(step)
    out = torch.zeros(R, p, size, dtype=torch.float64, device=lo.device)
    bins = torch.arange(p, dtype=torch.float32, device=lo.device).unsqueeze(0)
    for i in range(int(grid.max().item()) if R else 0):
        c = (lo.unsqueeze(1) + bins * step.unsqueeze(1)) + (float(i) + 0.5) * step.unsqueeze(1) / grid.unsqueeze(1)
        ok = (c >= -1.0) & (c <= float(size)) & (i < grid).unsqueeze(1)
        c = c.clamp(min=0.0)
        i0 = c.floor().long().clamp(max=size - 1)
        frac = torch.where(i0 >= size - 1, torch.zeros_like(c), c - i0.float())   # exact in fp32
        low = 1.0 - frac
        if order == 0:
            low = (low >= 0.5).float()
            frac = 1.0 - low
        i1 = (i0 + 1).clamp(max=size - 1)
        out.scatter_add_(2, i0.unsqueeze(2), (low.double() * ok).unsqueeze(2))
        out.scatter_add_(2, i1.unsqueeze(2), (frac.double() * ok).unsqueeze(2))
    return out / grid.double().view(R, 1, 1)


def _exact_roi(st):
    case = st["case"]
    d, h, w = _sizes(case["size"])[0]
    p, R, C = case["pooled"], case["rois"], case["channels"]
    rois = st["rois"].float()
    lo, hi = rois[:, 1:4] * case["scale"], rois[:, 4:7] * case["scale"]
    wx, wy, wz = (_axis_weights(lo[:, a], hi[:, a], s, p, case["ratio"], case["order"])
                  for a, s in ((0, w), (1, h), (2, d)))
    feat = st["features"].detach().double()
    grad = st["grad"].double() if case["train"] else None
    out = feat.new_empty(R, C, p, p, p)
    gfeat = torch.zeros_like(feat) if case["train"] else None
    items = rois[:, 0].long().tolist()
    for r in range(R):
        spans = []
        for m in (wz[r], wy[r], wx[r]):   # the voxels that the roi's bins reach
            hit = torch.nonzero(m.abs().sum(0)).flatten()
            spans.append(slice(int(hit[0]), int(hit[-1]) + 1) if hit.numel() else slice(0, 1))
        z, y, x = spans
        az, ay, ax = wz[r][:, z], wy[r][:, y], wx[r][:, x]
        f = feat[items[r], :, z, y, x]
        t = torch.tensordot(torch.tensordot(torch.tensordot(f, ax, ([3], [1])), ay, ([2], [1])), az, ([1], [1]))
        out[r] = t.permute(0, 3, 2, 1)   # [C, x, y, z] -> [C, z, y, x]
        if grad is not None:
            t = torch.tensordot(torch.tensordot(torch.tensordot(grad[r], ax, ([3], [0])), ay, ([2], [0])), az,
                                ([1], [0]))
            gfeat[items[r], :, z, y, x] += t.permute(0, 3, 2, 1)
    return out if gfeat is None else (out, gfeat)


def exact(case, seed):
    if case["kind"] == "nms":   # indices: decisions in fp32, no 64-bit value
        return None
    st = prepare(case, seed)
    if case["kind"] in ("attn", "offsets"):
        return _exact_attn(st)
    return _exact_dcn(st) if case["kind"] == "dcn" else _exact_roi(st)
