"""GPU parity of the 1:1 launchers (kernels.rs hot-path methods) against the
CPU oracle.  Tolerances are the reference's own (gemv_bench.rs:61-71,
kernels_bench.rs:136-161) unless the build's order makes the result exact."""
import numpy as np
import pytest

import llmpager_amd as lp
import _oracle as O
from _gpu import align, rel_l2, worst_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,group,experts,x_stride", [
    (768, 2048, 32, 8, 0),      # gate/up, config 1
    (2048, 768, 32, 8, 768),    # down, config 1 (x per expert)
    (768, 2048, 64, 8, 0),      # the reference's own q4g64 packs
    (64, 128, 64, 2, 128),      # write_test_checkpoint shape (lib.rs:341-423)
    (100, 96, 32, 3, 96),       # ragged rows, unaligned nibble rows: VALU path
    (100, 128, 32, 3, 128),     # ragged rows on the MFMA tile
    (48, 96, 32, 2, 96),        # a partial last sub-group step (cols/32 = 3)
    (40, 64, 8, 2, 64),         # group 8: generic VALU path
])
def test_q4_gemv_batch(cuda, rows, cols, group, experts, x_stride):
    rng = np.random.default_rng(rows * 7 + cols)
    H, I = (cols, rows) if rows <= cols else (rows, cols)
    qb = lp.q4_bytes(rows, cols, group)
    span = align(qb + 64)
    host = np.zeros(experts * span, np.uint8)
    regions = []
    for e in range(experts):
        w = rng.standard_normal(rows * cols).astype(np.float32) * 0.05
        buf, _ = O.q4_quantize(w, rows, cols, group)
        host[e * span + 32: e * span + 32 + qb] = buf
        regions.append(buf)
    nx = cols if x_stride == 0 else x_stride * experts
    x = rng.standard_normal(nx).astype(np.float32)
    arena = cuda.upload(host)
    ptrs = np.array([arena + e * span for e in range(experts)], np.uint64)
    d_ptrs = cuda.upload(ptrs)
    d_x = cuda.upload(x)
    d_y = cuda.alloc_device(experts * rows * 4)
    k = lp.Kernels(cuda)
    k.q4g64_gemv_batch(d_ptrs, 32, d_x, x_stride, d_y, rows, cols, group, experts)
    y = cuda.download(d_y, (experts, rows), np.float32)
    for e in range(experts):
        want = O.q4_gemv(regions[e], x[e * x_stride: e * x_stride + cols], rows, cols, group)
        assert worst_rel(y[e], want) <= 1e-3
        # the MFMA path carries x as 16-bit fixed point per 32 columns
        # (within 2^-16 of each sub-group's largest magnitude): rel-L2 ~2e-5
        assert rel_l2(y[e], want) <= 1e-4
    # single-matrix form
    k.q4g64_gemv(arena + 32, d_x, d_y, rows, cols, group)
    y1 = cuda.download(d_y, (rows,), np.float32)
    want = O.q4_gemv(regions[0], x[:cols], rows, cols, group)
    assert rel_l2(y1, want) <= 1e-4
    for p in (arena, d_ptrs, d_x, d_y):
        cuda.free_device(p)


@pytest.mark.parametrize("rows,cols", [(128, 2048), (64, 128), (7, 13), (4096, 4096)])
def test_bf16_gemv(cuda, rows, cols):
    rng = np.random.default_rng(rows + cols)
    w = lp.synth_bf16(rows * cols, 0.02, 5, rows)
    x = rng.standard_normal(cols).astype(np.float32)
    d_w, d_x = cuda.upload(w), cuda.upload(x)
    d_y = cuda.alloc_device(rows * 4)
    lp.Kernels(cuda).bf16_gemv(d_w, d_x, d_y, rows, cols)
    y = cuda.download(d_y, (rows,), np.float32)
    want = O.bf16_gemv(w, x, rows, cols)
    assert worst_rel(y, want) <= 1e-4          # kernels_bench.rs:148-149
    if cols % 8 == 0:
        # the canonical router order: bit-identical to the oracle's restatement
        canon = np.array([O.router_logits(w[r * cols:(r + 1) * cols], x, 1, cols)[0]
                          for r in range(rows)], np.float32)
        assert np.array_equal(y.view(np.uint32), canon.view(np.uint32))
    for p in (d_w, d_x, d_y):
        cuda.free_device(p)


def test_silu_add_reduce(cuda):
    rng = np.random.default_rng(3)
    n = 1000
    a = rng.standard_normal(n).astype(np.float32) * 3
    b = rng.standard_normal(n).astype(np.float32)
    k = lp.Kernels(cuda)
    da, db, dout = cuda.upload(a), cuda.upload(b), cuda.alloc_device(n * 4)
    k.silu_mul(da, db, dout, n)
    assert worst_rel(cuda.download(dout, (n,), np.float32), O.silu_mul(a, b)) <= 1e-4
    k.add(da, db, n)
    assert worst_rel(cuda.download(da, (n,), np.float32), O.add(a, b)) <= 1e-5
    # moe_reduce: same fused order as the oracle restatement -> bit-exact
    E, H = 8, 2048
    eo = rng.standard_normal((E, H)).astype(np.float32)
    wt = rng.random(E).astype(np.float32)
    h = rng.standard_normal(H).astype(np.float32)
    deo, dwt, dh = cuda.upload(eo), cuda.upload(wt), cuda.upload(h)
    k.moe_reduce(deo, dwt, dh, E, H)
    got = cuda.download(dh, (H,), np.float32)
    assert np.array_equal(got, O.moe_reduce(eo, wt, h))
    for p in (da, db, dout, deo, dwt, dh):
        cuda.free_device(p)


def _device_expf(cuda, first, stride, n):
    out = cuda.alloc_device(n * 4)
    assert lp.lib().lp_route_expf_device(cuda.ctx, first, stride, n, out, None) == 0
    got = cuda.download(out, (n,), np.float32)
    cuda.free_device(out)
    return got


@pytest.mark.parametrize("first,stride,n", [
    (0, 9973, (1 << 32) // 9973),     # a spread over every float
    (0x42b00000 - 2048, 1, 4096),     # around 88.0 (the special-case cut)
    (0x42b17218 - 2048, 1, 4096),     # around the overflow threshold
    (0xc2cff1b4 - 2048, 1, 4096),     # around the underflow threshold
    (0x7f800000 - 2048, 1, 4096),     # largest finite, +inf, NaNs
    (0xff800000 - 2048, 1, 4096),     # most negative finite, -inf, NaNs
    (0x00000000, 1, 8192),            # +0 and denormals
    (0x80000000, 1, 8192),            # -0 and negative denormals
    (0x3f800000 - 4096, 1, 8192),     # around 1.0
])
def test_device_expf_matches_glibc(cuda, first, stride, n):
    # The routing kernels' expf (glibc's method, table in registers) against
    # this host's glibc expf, bit for bit.
    got = _device_expf(cuda, first, stride, n)
    want = O.expf_sweep(first, stride, n)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), hex((first + stride * int(np.argmin(same))) & 0xffffffff)


# The 1:1 launchers' edges: rows around a wave's and a workgroup's register
# form of rmsnorm, widths that make no 16-byte pieces; bf16 GEMV widths around
# four chunks of 64 lanes; q4 GEMV tiles of one chunk, of two and of more, on
# one wave per workgroup and on four.  Bounds: fp32 sums of n terms.
@pytest.mark.parametrize("rows,n", [(1, 1024), (5, 1023), (3, 1028), (2, 4096), (2, 4100), (7, 20), (9, 30)])
def test_rmsnorm_edges(cuda, rows, n):
    rng = np.random.default_rng(n)
    K = lp.Kernels(cuda)
    x, w = rng.standard_normal(rows * n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    dx, dw = cuda.upload(x), cuda.upload(w)
    K.rmsnorm(dx, dw, dx, rows, n, 1e-6)
    x64 = x.reshape(rows, n).astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6) * w
    got = cuda.download(dx, (rows, n), np.float32)
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1.0)) <= n * 2.0 ** -24 + 4 * 2.0 ** -23
    cuda.free_device(dx)
    cuda.free_device(dw)


@pytest.mark.parametrize("rows,cols", [(5, 8), (4, 2040), (3, 2048), (6, 2056), (2, 4096), (1, 4104), (3, 12288), (4, 2047)])
def test_bf16_gemv_edges(cuda, rows, cols):
    K = lp.Kernels(cuda)
    w = lp.synth_bf16(rows * cols, 0.05, 3, cols)
    x = np.random.default_rng(cols).standard_normal(cols).astype(np.float32)
    dw, dx, dy = cuda.upload(w), cuda.upload(x), cuda.alloc_device(rows * 4)
    K.bf16_gemv(dw, dx, dy, rows, cols)
    w64 = (w.astype(np.uint32) << 16).view(np.float32).astype(np.float64).reshape(rows, cols)
    got = cuda.download(dy, (rows,), np.float32)
    bound = (cols / 64 + 8) * 2.0 ** -24 * (np.abs(w64) @ np.abs(x.astype(np.float64)))
    assert np.all(np.abs(got - w64 @ x) <= bound)
    for p in (dw, dx, dy):
        cuda.free_device(p)


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("rows,cols,experts", [(16, 128, 1), (33, 1024, 2), (768, 1152, 8), (48, 2048, 3), (64, 2176, 2),
                                               (2048, 768, 8), (5000, 256, 4)])
def test_q4_gemv_batch_edges(cuda, rows, cols, experts, group):
    rng = np.random.default_rng(rows + cols)
    K = lp.Kernels(cuda)
    w = rng.standard_normal((experts, rows * cols)).astype(np.float32) * 0.05
    blobs = [O.q4_quantize(w[e], rows, cols, group)[0] for e in range(experts)]
    dev = [cuda.upload(b) for b in blobs]
    dptr = cuda.upload(np.array([int(d) for d in dev], np.uint64))
    x = rng.standard_normal((experts, cols)).astype(np.float32)
    dx, dy = cuda.upload(x), cuda.alloc_device(experts * rows * 4)
    K.q4g64_gemv_batch(dptr, 0, dx, cols, dy, rows, cols, group, experts)
    W = np.stack([O.q4_dequantize(b, rows, cols, group) for b in blobs]).astype(np.float64)
    got = cuda.download(dy, (experts, rows), np.float32)
    for e in range(experts):
        want = W[e] @ x[e].astype(np.float64)
        # x to 2^-16 of each 32 columns' largest (at most max |x|), and fp32 sums
        bound = (2.0 ** -16 * np.abs(x[e]).max() + 2.0 ** -24 * cols / 32 * np.abs(x[e]).max()) * np.abs(W[e]).sum(1)
        assert np.all(np.abs(got[e] - want) <= bound)
    for p in dev + [dptr, dx, dy]:
        cuda.free_device(p)
