"""lp_attn_fused and lp_attn_block past the splits that a KV head's last
arrival merges: one workgroup per query head merges up to 64 records."""
import os

import numpy as np
import pytest

import llmpager_amd as lp
import test_gpu_step as step

pytestmark = pytest.mark.gpu

# 33 and 64 chunks of 64 positions (one per split), 65 and 130 (two and three
# per split); a scratch that holds 32 records (the last arrival's merge), then 33
LONG = [(8, 2, 2111, 8192), (16, 1, 4095, 8200), (4, 4, 4096, 8448), (8, 1, 8300, 16384), (8, 2, 4000, 32 * 132 + 32),
        (8, 2, 4000, 33 * 132 + 32)]


@pytest.mark.parametrize("heads,kvh,pos,ms", LONG)
def test_attn_block_long(cuda, heads, kvh, pos, ms):
    step.test_attn_block(cuda, lp.Kernels(cuda), heads, kvh, pos, ms, 512)


@pytest.mark.parametrize("heads,kvh,pos,ms", LONG)
def test_attn_fused_long(cuda, heads, kvh, pos, ms):
    for _ in range(2):  # the counters reset themselves
        step.test_attn_fused(cuda, lp.Kernels(cuda), heads, kvh, pos, ms, True)


@pytest.mark.parametrize("block", [False, True])
def test_merge_wait_that_gives_up_is_reported(cuda, block):
    # a context whose bound on the waits is one poll (set from the host): the
    # merges of 44 splits give up, the launch still ends, lp_step_errors_sync
    # reports it and clears the counters, so the next launch on that stream
    # (16 splits, whose last arrival merges) is right again
    os.environ["LLMPAGER_HIP_STEP_SPIN"] = "1"
    try:
        c = lp.Cuda(0)
    finally:
        del os.environ["LLMPAGER_HIP_STEP_SPIN"]
    K = lp.Kernels(c)
    heads, kvh, hd, pos, ms, hidden = 16, 1, 128, 8300, 16384, 512
    rng = np.random.default_rng(3)
    sizes = [heads * hd, kvh * hd, kvh * hd, hidden * heads * hd // 2, kvh * ms * hd // 2, kvh * ms * hd // 2, heads * hd,
             heads * ms, hidden, hidden, hidden]
    dq, dk, dv, dwo, dkc, dvc, dout, dscr, dh, dln, dhn = bufs = [
        c.upload((rng.standard_normal(n) if i < 3 else np.zeros(n)).astype(np.float32)) for i, n in enumerate(sizes)]
    args = (dq, dk, dv, 0, 0, 1e-6, 1e6, dkc, dvc, dout, dscr, heads, kvh, hd, pos, ms, 0.09)
    if block:
        K.attn_block(*args, dwo, dh, dln, dhn, hidden)
    else:
        K.attn_fused(*args)
    assert c.step_errors() > 0
    step.test_attn_fused(c, K, 32, 4, 1023, 4096, True)
    assert c.step_errors() == 0
    for p in bufs:
        c.free_device(p)
    c.close()
