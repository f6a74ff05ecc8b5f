"""The dispatch tables of batches above 64 tokens, against their definition:
the (t, j) picks grouped by expert, in token order within an expert.  Batches
at the edges of the 64-token masks and of the one-workgroup form (2048
tokens, and expert counts whose masks outgrow its LDS)."""
import numpy as np
import pytest

import llmpager_amd as lp
from _gpu import DeviceLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k", [(3, 1), (64, 6), (128, 8), (257, 16), (1024, 2)])
@pytest.mark.parametrize("T", [65, 127, 128, 129, 203, 1024, 2047, 2049])
def test_dispatch_tables(cuda, T, E, k):
    L = DeviceLayer(cuda, H=64, I=32, E=E, k=k, group=32, seed=E, gating=lp.GATING_SIGMOID, renorm=False,
                    min_weight=0.6, bias=np.zeros(E, np.float32))
    rng = np.random.default_rng(T + E)
    logits = (rng.standard_normal((T, E)) * 2 + np.linspace(2, -2, E) - rng.uniform(0, 8, (T, 1))).astype(np.float32)
    lay = lp.ws_layout(L.desc, T)
    ws = cuda.alloc_device(lay.total)
    dl = cuda.upload(logits)
    L.layer.route_logits(dl, T, ws)
    ids = cuda.download(ws + lay.ids, (T, k), np.int32)
    cnt = cuda.download(ws + lay.cnt, (T,), np.int32)
    assert np.array_equal((ids >= 0).sum(1), cnt) and (cnt < k).any()
    want = [[t * k + j for t, j in zip(*np.nonzero(ids == e))] for e in range(E)]
    gs = cuda.download(ws + lay.gs, (E + 1,), np.int32)
    n = np.array([len(w) for w in want])
    assert np.array_equal(gs, np.concatenate([[0], np.cumsum(n)]))
    perm = cuda.download(ws + lay.perm, (T * k,), np.int32)[: n.sum()]
    assert np.array_equal(perm, np.concatenate([np.array(w, np.int32) for w in want]))
    inv = np.full(T * k, -1, np.int32)
    inv[perm] = np.arange(len(perm))
    assert np.array_equal(cuda.download(ws + lay.inv, (T * k,), np.int32), inv)
    uniq = np.nonzero(n)[0]
    meta = cuda.download(ws + lay.meta, (3,), np.int32)
    assert meta[:2].tolist() == [len(uniq), 0]
    assert np.array_equal(cuda.download(ws + lay.uniq, (len(uniq),), np.int32), uniq)
    et = cuda.download(ws + lay.et, (min(T * k, E), 8), np.int32)
    for u, row in enumerate(et):
        toks = [p // k for p in want[uniq[u]][:4]] if u < len(uniq) else []
        blob = row[:2].copy().view(np.uint64)[0]
        assert (blob != 0) == (u < len(uniq))
        assert row[2:4].tolist() == ([gs[uniq[u]], n[uniq[u]]] if u < len(uniq) else [0, 0])
        assert row[4:].tolist() == toks + [-1] * (4 - len(toks))
    # the tile list of the kernels that take the experts in blocks: the GEMM's
    # of 128 tokens (16 pairs per expert), lp_mid.hip's of 32 (x's images in y)
    block = 128 if T * k >= 16 * min(E, T * k) else 32 if lay.xf == lay.y else 0
    if block:
        tiles = [(u << 16) | b for u, e in enumerate(uniq) for b in range((n[e] + block - 1) // block)]
        assert meta[2] == len(tiles)
        assert cuda.download(ws + lay.tiles, (len(tiles),), np.int32).tolist() == tiles
    for p in (ws, dl):
        cuda.free_device(p)
    L.free()


# experts with exactly a block's tokens, one short of it, one past it, and
# several blocks: both block sizes, the one-workgroup dispatch and (2049
# tokens) the three-launch one; 48 tokens: the list of a decode-sized GEMM
@pytest.mark.parametrize("T,E,counts", [
    (203, 40, [32, 31, 33, 64, 1]), (2049, 300, [32, 96, 31, 33, 1]), (700, 6, [128, 127, 129, 256, 1]),
    (2049, 9, [128, 256, 127, 129, 1]), (48, 2, [31]), (48, 3, [16, 32])])
def test_tile_list_edges(cuda, T, E, counts):
    L = DeviceLayer(cuda, H=64, I=32, E=E, k=1, group=32, seed=E)
    logits = np.full((T, E), -5.0, np.float32)
    logits += 0.1 * np.random.default_rng(T).standard_normal((T, E)).astype(np.float32)
    at = 0
    for e, c in enumerate(counts):
        logits[at:at + c, e] = 5.0
        logits[at + c:, e] = -50.0
        at += c
    lay = lp.ws_layout(L.desc, T)
    gemm = T >= 16 * E
    assert gemm or lay.xf == lay.y
    block = 128 if gemm else 32
    ws = cuda.alloc_device(lay.total)
    dl, dx, dh = cuda.upload(logits), cuda.upload(np.ones((T, 64), np.float32)), cuda.alloc_device(T * 64 * 4)
    L.layer.route_logits(dl, T, ws)
    L.layer.experts(dx, dh, T, ws)
    n = np.bincount(logits.argmax(1), minlength=E)
    assert n[:len(counts)].tolist() == counts
    want = [(u << 16) | b for u, e in enumerate(np.nonzero(n)[0]) for b in range((n[e] + block - 1) // block)]
    assert cuda.download(ws + lay.meta, (3,), np.int32).tolist() == [np.count_nonzero(n), 0, len(want)]
    assert cuda.download(ws + lay.tiles, (len(want),), np.int32).tolist() == want
    for p in (ws, dl, dx, dh):
        cuda.free_device(p)
    L.free()
