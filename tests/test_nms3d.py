"""3-D NMS: the CPU oracle pinned (closed-form IoUs, the reference's own test cases, an
independent pairwise formulation), and the GPU kernels against it (marked gpu).

Reference tests: tests/test_nms.py:17-49 (1000 duplicates of one box -> only the top box;
two disjoint boxes -> both kept)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import nms3d as O


def _clustered(n, seed, spread=30.0, size=(2.0, 12.0)):
    """Boxes in a few clusters (so suppression happens), random scores with some ties."""
    r = np.random.default_rng(seed)
    centres = r.uniform(0, 100, size=(max(1, n // 20), 3))
    c = centres[r.integers(0, len(centres), n)] + r.normal(0, spread / 10, size=(n, 3))
    e = r.uniform(*size, size=(n, 3))
    boxes = np.concatenate([c - e / 2, c + e / 2], 1).astype(np.float32)
    scores = np.round(r.uniform(0, 1, n), 2).astype(np.float32)   # two decimals: ties
    return boxes, scores


# --- oracle pinning (CPU) --------------------------------------------------------------------
def test_iou_closed_forms():
    a = [0, 0, 0, 2, 2, 2]
    assert O.iou3d(a, [a])[0] == 1.0
    assert O.iou3d(a, [[3, 3, 3, 4, 4, 4]])[0] == 0.0                      # disjoint
    assert O.iou3d(a, [[2, 0, 0, 4, 2, 2]])[0] == 0.0                      # touching faces
    assert np.isclose(O.iou3d(a, [[1, 0, 0, 3, 2, 2]])[0], 4 / 12)         # half shifted along x
    assert np.isclose(O.iou3d([0, 0, 0, 4, 4, 4], [[1, 1, 1, 3, 3, 3]])[0], 8 / 64)   # nested
    assert np.isclose(O.iou3d(a, [[1, 1, 1, 3, 3, 3]])[0], 1 / 15)        # corner overlap
    # zero-volume pair: 0/0 -> NaN, never above a threshold
    assert np.isnan(O.iou3d([1, 1, 1, 1, 1, 1], [[1, 1, 1, 1, 1, 1]])[0])


def test_oracle_reference_cases():
    box0 = [0, 0, 0, 100, 100, 100]
    boxes = np.tile(np.asarray(box0, np.float32), (1000, 1))
    scores = np.zeros(1000, np.float32)
    scores[0] = 0.9
    assert O.nms3d(boxes, scores, 0.1).tolist() == [0]
    two = np.asarray([[0, 0, 0, 10, 10, 10], [20, 20, 20, 30, 30, 30]], np.float32)
    assert O.nms3d(two, np.asarray([0.6, 0.7]), 0.5).tolist() == [1, 0]   # both, by score


def test_oracle_against_pairwise_definition():
    """The greedy pass restated from a full float64 IoU matrix: box i is kept iff no kept box
    before it (in score order) has IoU above the threshold with it.  Boxes whose IoU lies within
    1e-5 of the threshold are excluded so that fp32 and fp64 decide alike."""
    for seed in range(5):
        boxes, scores = _clustered(300, seed)
        order = np.argsort(-scores.astype(np.float64), kind="stable")
        b = boxes[order].astype(np.float64)
        lo, hi = np.maximum(b[:, None, :3], b[None, :, :3]), np.minimum(b[:, None, 3:], b[None, :, 3:])
        inter = np.prod(np.clip(hi - lo, 0, None), -1)
        vol = np.prod(b[:, 3:] - b[:, :3], -1)
        iou = inter / (vol[:, None] + vol[None, :] - inter)
        thr = 0.3
        if np.any(np.abs(iou - thr) < 1e-5):
            continue
        kept = []
        for i in range(len(b)):
            if all(iou[k, i] <= thr for k in kept):
                kept.append(i)
        assert O.nms3d(boxes, scores, thr).tolist() == order[kept].tolist()


# --- GPU ---------------------------------------------------------------------------------------
@pytest.mark.gpu
def test_gpu_reference_cases(gpu_device):
    from ops3d_amd import _C

    box0 = torch.tensor([0, 0, 0, 100, 100, 100], device=gpu_device, dtype=torch.float32)
    boxes = box0.unsqueeze(0).repeat(1000, 1)
    scores = torch.cat([torch.tensor([0.9], device=gpu_device), torch.zeros(999, device=gpu_device)])
    assert _C.nms_3d(boxes, scores, 0.1).cpu().tolist() == [0]
    two = torch.tensor([[0, 0, 0, 10, 10, 10], [20, 20, 20, 30, 30, 30]], device=gpu_device, dtype=torch.float32)
    assert set(_C.nms_3d(two, torch.tensor([0.6, 0.7], device=gpu_device), 0.5).cpu().tolist()) == {0, 1}
    empty = _C.nms_3d(torch.empty(0, 6, device=gpu_device), torch.empty(0, device=gpu_device), 0.5)
    assert empty.dtype == torch.long and empty.numel() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("n,thr,seed", [(1, 0.5, 0), (63, 0.3, 1), (64, 0.3, 2), (65, 0.3, 3), (1000, 0.1, 4),
                                        (1000, 0.5, 5), (4097, 0.3, 6), (20000, 0.3, 7)])
def test_gpu_matches_oracle(gpu_device, n, thr, seed):
    from fda_helpers import log

    from ops3d_amd.nms import nms_nd

    log(f"[case] nms3d n={n} thr={thr} seed={seed}")
    boxes, scores = _clustered(n, seed)
    dets = torch.from_numpy(np.concatenate([boxes, scores[:, None]], 1)).to(gpu_device)
    keep, _ = nms_nd(dets, thr)
    want = O.nms3d(boxes, scores, thr)
    assert keep.dtype == torch.long
    assert keep.cpu().numpy().tolist() == want.tolist()


@pytest.mark.gpu
def test_gpu_degenerate_and_thresholds(gpu_device):
    from ops3d_amd import _C

    boxes, scores = _clustered(500, 9)
    boxes[::7, 3:] = boxes[::7, :3]     # zero-volume boxes: IoU NaN with each other
    b = torch.from_numpy(boxes).to(gpu_device)
    s = torch.from_numpy(scores).to(gpu_device)
    for thr in (0.0, 0.3, 1.0):
        got = _C.nms_3d(b, s, thr).cpu().numpy().tolist()
        assert got == O.nms3d(boxes, scores, thr).tolist(), thr
    with pytest.raises(RuntimeError, match="CPU"):
        _C.nms_3d(torch.from_numpy(boxes), torch.from_numpy(scores), 0.5)


# --- the pair path (ops3d_nms3d_pairs) against the mask path (ops3d_nms3d) ---------------------
def test_pairs_host_rules():
    """Which calls the pair path takes, and its refusals before any device work (no GPU needed)."""
    from ops3d_amd import _C

    lib = _C._lib
    assert lib.ops3d_nms3d_pairs_workspace_bytes(0) == 0
    assert lib.ops3d_nms3d_pairs_workspace_bytes((1 << 18) + 1) == 0
    assert [lib.ops3d_nms3d_pairs_ranks(n) for n in (0, 1, 8192, 8193)] == [0, 1, 1, 0]
    for n in (1, 64, 8192, 8193, 1 << 18):
        # boxes in score order, padded to blocks of 64 (32 bytes each), and the pair lists
        assert lib.ops3d_nms3d_pairs_workspace_bytes(n) >= (n + 63) // 64 * 64 * 32 + n * 64 * 8
    p = 256

    def call(n, thr, order=None, scores=p, ws=p, wsb=1 << 40):
        return lib.ops3d_nms3d_pairs(p, 6, 1, scores, 1, order, n, thr, ws, wsb, p, p, None)

    bad = (call(10, -0.5), call(10, float("nan")), call((1 << 18) + 1, 0.5, order=p), call(9000, 0.5),
           call(10, 0.5, order=p), call(10, 0.5, scores=None), call(10, 0.5, wsb=64), call(10, 0.5, ws=p + 8))
    assert set(bad) == {1}   # EINVAL


def test_pair_block_enumeration():
    """The pair kernel's folded grid (row blocks p and last - p share last + 2 column blocks) visits
    every block pair on or above the diagonal once."""
    for nblk in (1, 2, 3, 8, 63, 64, 65, 128):
        seen = []
        for bid in range((nblk + 1) // 2 * (nblk + 1)):
            p, k = divmod(bid, nblk + 1)
            if k < nblk - p:
                seen.append((p, p + k))
            elif nblk - 1 - p != p:
                rb = nblk - 1 - p
                seen.append((rb, rb + k - (nblk - p)))
        assert sorted(seen) == [(r, c) for r in range(nblk) for c in range(r, nblk)]
    # and its row index of pair p among nr x nc, formed in fp32, is p // nc
    p = np.arange(64 * 64)
    for nc in range(1, 65):
        inv = np.float32(1) / np.float32(nc)
        got = ((p.astype(np.float32) + np.float32(0.5)) * inv).astype(np.int64)
        assert np.array_equal(got, p // nc), nc


def _mask_path(boxes, scores, thr):
    """Kept indices by torch's stable sort and the mask kernels, through the C ABI."""
    from ops3d_amd import _C

    lib, n = _C._lib, boxes.shape[0]
    order = torch.sort(scores, stable=True, descending=True)[1]
    b = boxes.index_select(0, order).float().contiguous()
    wsb = lib.ops3d_nms3d_workspace_bytes(n)
    ws = torch.empty(wsb, dtype=torch.uint8, device=boxes.device)
    keep = torch.empty(n, dtype=torch.long, device=boxes.device)
    num = torch.empty(1, dtype=torch.int32, device=boxes.device)
    st = torch.cuda.current_stream().cuda_stream
    assert lib.ops3d_nms3d(b.data_ptr(), order.data_ptr(), n, thr, ws.data_ptr(), wsb, keep.data_ptr(),
                           num.data_ptr(), st) == 0
    return keep[: int(num.item())].cpu().tolist()


def _chain(n):
    """Overlapping boxes in a row: each depends on the one before."""
    lo = np.zeros((n, 3), np.float32)
    lo[:, 0] = np.arange(n)
    return np.concatenate([lo, lo + np.float32([2.2, 1, 1])], 1).astype(np.float32), np.ones(n, np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,thr", [
    ("random", 2, 0.3), ("random", 127, 0.0), ("random", 4096, 0.1), ("random", 8192, 0.3), ("random", 8193, 0.3),
    ("random", 65537, 0.5), ("random", 1 << 18, 0.5), ("random", (1 << 18) + 1, 0.5), ("dense", 3000, 0.1), ("dense", 9001, 0.2), ("chain", 40, 0.2), ("chain", 3000, 0.2),
    ("chain", 10000, 0.2), ("special", 1000, 0.25), ("special", 9000, 0.0), ("random", 700, -0.5),
    ("strided", 500, 0.3), ("half", 500, 0.3), ("double", 500, 0.3), ("double", 9000, 0.3)])
def test_gpu_pairs_same_as_mask(gpu_device, kind, n, thr):
    """Every route of nms_3d gives the mask path's list: ranks by counting and by torch's sort, the
    cell order, lists that overflow (dense) and chains beyond the rounds (both fall back), scores
    with ties, NaN, infinities and both zeros, boxes with NaN, infinite, inverted and zero extents,
    strided and other types."""
    from fda_helpers import log

    from ops3d_amd import _C

    log(f"[case] nms3d pairs {kind} n={n} thr={thr}")
    boxes, scores = _chain(n) if kind == "chain" else _clustered(n, 3)
    if kind == "dense":
        boxes[:, :3] = boxes[:, :3] * np.float32(0.01)
        boxes[:, 3:] = boxes[:, :3] + np.float32(5.0)
    if kind == "special":
        boxes[::9, 0] = np.nan
        boxes[1::31, 4] = np.inf
        boxes[2::37, :3] = -np.inf
        boxes[3::11, 3:] = boxes[3::11, :3]
        boxes[4::13, 3:] = boxes[4::13, :3] - 1
        scores[::17] = np.nan
        scores[1::19] = np.inf
        scores[2::23] = -np.inf
        scores[3::5] = 0.0
        scores[4::10] = -0.0
    b, s = torch.from_numpy(boxes).to(gpu_device), torch.from_numpy(scores).to(gpu_device)
    if kind == "strided":
        b = torch.cat([b, b], 1).t().contiguous().t()[:, 6:12]
        s = torch.stack([s, -s], 1)[:, 0]
    if kind == "half":
        b, s = b.half(), s.half()
    if kind == "double":
        b, s = b.double(), s.double()
    assert _C.nms_3d(b, s, thr).cpu().tolist() == _mask_path(b, s, thr)


def _pairs_path(boxes, scores, thr):
    """ops3d_nms3d_pairs itself: the kept indices, or None where it gave up (num_keep = -1)."""
    from ops3d_amd import _C

    lib, n = _C._lib, boxes.shape[0]
    order = None if lib.ops3d_nms3d_pairs_ranks(n) else torch.sort(scores, stable=True, descending=True)[1]
    wsb = lib.ops3d_nms3d_pairs_workspace_bytes(n)
    ws = torch.empty(wsb, dtype=torch.uint8, device=boxes.device)
    keep = torch.full((n,), -7, dtype=torch.long, device=boxes.device)
    num = torch.full((1,), -7, dtype=torch.int32, device=boxes.device)
    rc = lib.ops3d_nms3d_pairs(boxes.data_ptr(), boxes.stride(0), boxes.stride(1),
                               None if order is not None else scores.data_ptr(), scores.stride(0),
                               None if order is None else order.data_ptr(), n, thr, ws.data_ptr(), wsb,
                               keep.data_ptr(), num.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    kept = int(num.item())
    assert -1 <= kept <= n
    return keep[:kept].cpu().tolist() if kept >= 0 else None


def _clusters(n, m):
    """Clusters of m boxes that overlap each other, far apart."""
    r = np.random.default_rng(n)
    c = (np.arange(n) % -(-n // m) * 100.0)[:, None] + r.uniform(-0.3, 0.3, (n, 3))
    return np.concatenate([c - 5, c + 5], 1).astype(np.float32), r.uniform(size=n).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(64, 25), (64, 64), (128, 25), (128, 64), (300, 25), (1000, 25), (2000, 50),
                                 (1000, 100), (4096, 120), (9000, 100)])
def test_gpu_pairs_crowded_blocks(gpu_device, n, m):
    """The pair path itself (no fallback to the mask behind it) holds the pairs of a few crowded blocks,
    down to a call of a single one: they are spread over all lists."""
    from fda_helpers import log

    log(f"[case] nms3d pair path, clusters of {m} among {n}")
    boxes, scores = _clusters(n, m)
    b, s = torch.from_numpy(boxes).to(gpu_device), torch.from_numpy(scores).to(gpu_device)
    got = _pairs_path(b, s, 0.3)
    assert got is not None
    assert got == _mask_path(b, s, 0.3)


def _row(n, reach, thr):
    """Boxes in a row, each above the threshold with the next `reach`, scores falling along the row."""
    lo = np.zeros((n, 3), np.float32)
    lo[:, 0] = np.arange(n)
    width = (reach + 0.5) * (1 + thr) / (1 - thr)
    return np.concatenate([lo, lo + np.float32([width, 1, 1])], 1).astype(np.float32), -np.arange(n, dtype=np.float32)


def _raster(shape):
    """Boxes of edge 8 on a grid of step 2, equal scores: ranked in raster order."""
    lo = np.stack(np.meshgrid(*[np.arange(k) for k in shape], indexing="ij"), -1).reshape(-1, 3) * np.float32(2)
    return np.concatenate([lo, lo + 8], 1).astype(np.float32), np.ones(len(lo), np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,arg", [
    ("random", 1, 0.3), ("random", 64, 0.0), ("random", 4096, 0.1), ("random", 8192, 0.3), ("random", 8193, 0.3),
    ("random", 1 << 18, 0.5), ("chain", 40, 0.2), ("chain", 3000, 0.2), ("chain", 10000, 0.2), ("row", 65, 3),
    ("row", 2000, 25), ("row", 9000, 28), ("row", 20011, 12), ("raster", 0, (12, 12, 12)), ("raster", 0, (4, 4, 500)),
    ("raster", 0, (25, 25, 25))])
def test_gpu_pairs_take_chains(gpu_device, kind, n, arg):
    """The pair path itself (no fallback to the mask behind it) decides independent scores and chains
    of any length -- a row, equal scores in raster order -- with the mask path's list."""
    from fda_helpers import log

    log(f"[case] nms3d pair path {kind} n={n} {arg}")
    thr = arg if kind in ("random", "chain") else 0.3
    boxes, scores = {"random": lambda: _clustered(n, 5), "chain": lambda: _chain(n),
                     "row": lambda: _row(n, arg, thr), "raster": lambda: _raster(arg)}[kind]()
    b, s = torch.from_numpy(boxes).to(gpu_device), torch.from_numpy(scores).to(gpu_device)
    got = _pairs_path(b, s, thr)
    assert got is not None
    assert got == _mask_path(b, s, thr)


@pytest.mark.gpu
@pytest.mark.parametrize("n,row,reach,gives_up", [(1000, 1000, 40, True), (4096, 4096, 60, True), (9001, 9001, 50, True),
                                                  (2000, 160, 40, None), (9600, 120, 60, None)])
def test_gpu_pairs_leave_long_lists_of_chains(gpu_device, n, row, reach, gives_up):
    """Rows with more than 32 pairs per box: one chain is left to the mask path (a box is not blocked by
    an eighth of the pairs with (7/8)^reach < 1 %), many short ones may be decided either way."""
    from fda_helpers import log

    from ops3d_amd import _C

    log(f"[case] nms3d pair path, rows of {row} among {n} reaching {reach}")
    boxes, scores = _row(n, reach, 0.3)
    boxes[:, [1, 4]] += np.float32(5) * (np.arange(n) // row)[:, None].astype(np.float32)
    b, s = torch.from_numpy(boxes).to(gpu_device), torch.from_numpy(scores).to(gpu_device)
    got, want = _pairs_path(b, s, 0.3), _mask_path(b, s, 0.3)
    assert got is None or (gives_up is None and got == want)
    assert _C.nms_3d(b, s, 0.3).cpu().tolist() == want


@pytest.mark.gpu
@pytest.mark.parametrize("n", [300, 3000, 9001])
def test_gpu_mask_after_pairs(gpu_device, n):
    """More overlapping pairs than the lists hold: the pair path says so, and the mask path that goes on
    from its workspace (boxes and order) gives the mask path's list."""
    from ops3d_amd import _C

    lib, r = _C._lib, np.random.default_rng(1)
    lo = r.uniform(0, 1, (n, 3)).astype(np.float32)
    b = torch.from_numpy(np.concatenate([lo, lo + r.uniform(3, 5, (n, 3)).astype(np.float32)], 1)).to(gpu_device)
    s = torch.rand(n, device=gpu_device)
    order = None if lib.ops3d_nms3d_pairs_ranks(n) else torch.sort(s, stable=True, descending=True)[1]
    op = None if order is None else order.data_ptr()
    sizes = lib.ops3d_nms3d_pairs_workspace_bytes(n), lib.ops3d_nms3d_workspace_bytes(n)
    pws, ws = (torch.empty(v, dtype=torch.uint8, device=gpu_device) for v in sizes)
    keep = torch.empty(n, dtype=torch.long, device=gpu_device)
    num = torch.empty(1, dtype=torch.int32, device=gpu_device)
    st = torch.cuda.current_stream().cuda_stream
    out = (keep.data_ptr(), num.data_ptr(), st)
    assert lib.ops3d_nms3d_pairs(b.data_ptr(), 6, 1, None if op else s.data_ptr(), 1, op, n, 0.2, pws.data_ptr(), sizes[0],
                                 *out) == 0
    assert int(num.item()) == -1
    assert lib.ops3d_nms3d_after_pairs(pws.data_ptr(), sizes[0], op, n, 0.2, ws.data_ptr(), sizes[1], *out) == 0
    assert keep[: int(num.item())].cpu().tolist() == _mask_path(b, s, 0.2)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [500, 9000])
def test_gpu_negated_views(gpu_device, n):
    """Boxes and scores that are negated views (the imaginary part of a conjugate), through both
    modules: the values count, not what lies in memory."""
    import importlib

    from ops3d_amd import _C

    boxes, scores = _clustered(n, 4)
    want = O.nms3d(boxes, scores, 0.3).tolist()

    def view(a):
        t = torch.from_numpy(a).to(gpu_device)
        v = torch.complex(t, -t).conj().imag
        assert v.is_neg() and torch.equal(v, t)
        return v

    for module in (_C, importlib.import_module("ops3d_amd._fda_torch")):
        assert module.nms_3d(view(boxes), view(scores), 0.3).cpu().tolist() == want
