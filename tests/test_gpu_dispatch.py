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
    assert cuda.download(ws + lay.meta, (2,), np.int32).tolist() == [len(uniq), 0]
    assert np.array_equal(cuda.download(ws + lay.uniq, (len(uniq),), np.int32), uniq)
    et = cuda.download(ws + lay.et, (min(T * k, E), 8), np.int32)
    for u, row in enumerate(et):
        toks = [p // k for p in want[uniq[u]][:4]] if u < len(uniq) else []
        blob = row[:2].copy().view(np.uint64)[0]
        assert (blob != 0) == (u < len(uniq))
        assert row[2:4].tolist() == ([gs[uniq[u]], n[uniq[u]]] if u < len(uniq) else [0, 0])
        assert row[4:].tolist() == toks + [-1] * (4 - len(toks))
    for p in (ws, dl):
        cuda.free_device(p)
    L.free()
