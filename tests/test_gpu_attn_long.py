"""lp_attn_fused and lp_attn_block past the splits that a KV head's last
arrival merges: one workgroup per query head merges up to 64 records."""
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
