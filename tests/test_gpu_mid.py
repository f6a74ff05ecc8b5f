"""Batches between decode and prefill: the grouped projections of more than 64
tokens below the prefill GEMM's average per expert, and the shared MLP of
every batch above 64 tokens, against the CPU oracle."""
import numpy as np
import pytest

import llmpager_amd as lp
import _oracle as O
from _gpu import DeviceLayer, rel_l2

pytestmark = pytest.mark.gpu

# x and act enter as 22-bit hi + lo images (2^-22 each); the sums over the
# sub-groups are fp32 multiply-adds, one per 32 columns (at most 128 of them
# here), where the oracle's are fp32 throughout: both within 128 2^-24.
TOL = 2.0 ** -21 + 2 * 128 * 2.0 ** -24


def _run(cuda, L, x, h, logits=None):
    T = x.shape[0]
    lay = lp.ws_layout(L.desc, T)
    ws, dx, dh = cuda.alloc_device(lay.total), cuda.upload(x), cuda.upload(h)
    if logits is None:
        L.layer.forward(dx, dh, T, ws)
    else:
        dl = cuda.upload(logits)
        L.layer.route_logits(dl, T, ws)
        L.layer.experts(dx, dh, T, ws)
        cuda.sync()
        cuda.free_device(dl)
    got = cuda.download(dh, x.shape, np.float32)
    glog = cuda.download(ws + lay.logits, (T, L.E), np.float32)
    err = L.layer.status(ws, T)[1]
    for p in (ws, dx, dh):
        cuda.free_device(p)
    return got, glog, err


def _check(cuda, L, T, seed, logits=None, blobs=None, scale=1.0, want_err=0):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((T, L.H)) * scale).astype(np.float32)
    h = np.zeros((T, L.H), np.float32)
    got, glog, err = _run(cuda, L, x, h, logits)
    assert err == want_err
    want = O.moe_layer(L.oracle_desc(), blobs or L.oracle_blobs(), x, h.copy(), logits_in=glog, threads=8,
                       shared_blob=L.shared)[0]
    assert rel_l2(got, want) <= TOL
    per_token = [rel_l2(got[t], want[t]) for t in range(T)]
    assert max(per_token) <= 4 * TOL


# widths around the stages of 128 columns and the 128-column / 256-row blocks:
# one sub-group past, a lone one, rows short of a block; every group size; a
# token count just past the decode sizes; averages from 2 (rows wider than the
# balanced kernels take, or more token groups than CUs) to just below 16
@pytest.mark.parametrize("H,I,E,k,group,T", [
    (2048, 768, 128, 8, 32, 81), (2048, 768, 128, 8, 32, 203), (2048, 1408, 64, 6, 32, 100), (160, 96, 16, 2, 32, 65),
    (384, 32, 32, 4, 32, 100), (288, 544, 24, 3, 32, 127), (192, 128, 16, 2, 64, 90), (512, 384, 10, 1, 128, 77),
    (4096, 256, 16, 2, 32, 66), (128, 128, 12, 1, 32, 191), (2176, 64, 32, 1, 32, 66), (64, 64, 300, 4, 32, 70),
    (128, 128, 32, 2, 32, 96), (128, 128, 32, 2, 32, 95)])
def test_mid_layer(cuda, H, I, E, k, group, T):
    L = DeviceLayer(cuda, H=H, I=I, E=E, k=k, group=group, seed=H + I)
    assert T > 64 and T * k < 16 * E, "between decode and the prefill GEMM"
    _check(cuda, L, T, T)
    L.free()


# one expert with 1, 16, 17, 32, 33 and 70 tokens (token tiles and the group
# loop), the others sharing the rest
@pytest.mark.parametrize("heavy", [1, 16, 17, 32, 33, 70])
def test_mid_skewed(cuda, heavy):
    E, T = 16, 110
    L = DeviceLayer(cuda, H=256, I=128, E=E, k=2, group=32, seed=heavy)
    logits = np.random.default_rng(heavy).standard_normal((T, E)).astype(np.float32)
    logits[:, 5] = -20.0
    logits[np.random.default_rng(1).permutation(T)[:heavy], 5] = 20.0
    _check(cuda, L, T, 3, logits=logits)
    L.free()


# exponents: rows of very different size, a zero row's neighbours, and act
# sub-groups far apart
@pytest.mark.parametrize("scale", [1e-6, 30.0])
def test_mid_scaled(cuda, scale):
    L = DeviceLayer(cuda, H=256, I=128, E=16, k=2, group=32, seed=8)
    rows = (10.0 ** np.random.default_rng(2).integers(-3, 4, (100, 1))).astype(np.float32)
    rows[7] = 0.0
    _check(cuda, L, 100, 4, scale=scale * rows)
    L.free()


def test_mid_missing_expert(cuda):
    # an expert without a slot contributes zero and raises the flag
    slots = np.arange(16, dtype=np.int32)
    slots[[2, 9]] = -1
    L = DeviceLayer(cuda, H=256, I=160, E=16, k=2, group=32, seed=5, slots=slots)
    zero = next(b for b in L.oracle_blobs() if b is not None).copy()
    for off, rows, cols in zip(lp.blob_offsets(256, 160, 32), (160, 160, 256), (256, 256, 160)):
        sb = rows * (cols // 32) * 2
        zero[off + sb: off + sb + rows * cols // 2] = 0x88
    _check(cuda, L, 96, 6, blobs=[b if b is not None else zero for b in L.oracle_blobs()], want_err=1)
    L.free()


# the shared MLP above 64 tokens, beside routed experts through the decode
# kernels (70 tokens, few per expert), this path and the prefill GEMM (whose
# fp16 operands set the bound there)
@pytest.mark.parametrize("T,E,k,Is,sg", [(70, 64, 2, 352, 32), (90, 16, 2, 128, 64), (65, 16, 1, 1408, 32),
                                         (300, 16, 2, 256, 128), (1100, 8, 1, 96, 32)])
def test_mid_shared(cuda, T, E, k, Is, sg):
    L = DeviceLayer(cuda, H=256, I=128, E=E, k=k, group=32, seed=T, shared=(Is, sg))
    rng = np.random.default_rng(T)
    x, h = rng.standard_normal((T, 256)).astype(np.float32), np.zeros((T, 256), np.float32)
    got, glog, err = _run(cuda, L, x, h)
    want = O.moe_layer(L.oracle_desc(), L.oracle_blobs(), x, h.copy(), logits_in=glog, threads=8,
                       shared_blob=L.shared)[0]
    gemm = T * k >= 16 * E
    assert err == 0 and rel_l2(got, want) <= (1e-3 if gemm else 1e-4)
    L.free()


# ... and where x's images and the shared MLP's exponents sit in parts that the
# routed experts write after it: beside the balanced decode kernels (with rows
# short of 128 columns and one pick, x's images begin in act), and beside
# routed experts of this path with x's images past y's end
@pytest.mark.parametrize("H,I,T,E,k,Is", [(256, 256, 70, 64, 2, 352), (160, 256, 70, 64, 1, 128), (288, 96, 100, 10, 1, 160),
                                          (2048, 1408, 130, 64, 6, 2816)])
def test_mid_shared_workspace(cuda, H, I, T, E, k, Is):
    L = DeviceLayer(cuda, H=H, I=I, E=E, k=k, group=32, seed=T + H, shared=(Is, 32))
    rng = np.random.default_rng(T)
    x, h = rng.standard_normal((T, H)).astype(np.float32), np.zeros((T, H), np.float32)
    got, glog, err = _run(cuda, L, x, h)
    want = O.moe_layer(L.oracle_desc(), L.oracle_blobs(), x, h.copy(), logits_in=glog, threads=8,
                       shared_blob=L.shared)[0]
    assert err == 0 and rel_l2(got, want) <= 1e-4
    L.free()
