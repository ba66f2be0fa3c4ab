"""Which sequences overlap="auto" runs the memory branch beside Polar for: the lengths where that was measured faster."""

import pytest
import torch

pytestmark = pytest.mark.gpu
F32, B16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("dtype,B,T,want", [
    (F32, 1, 2048, False), (F32, 1, 2304, True), (F32, 1, 3000, True), (F32, 1, 6000, True), (F32, 1, 6001, False),
    (F32, 1, 8191, False), (F32, 1, 8192, True), (F32, 2, 4096, False),   # (two sequences' recurrences fill half the device)
    (B16, 1, 3000, False), (B16, 1, 8191, False), (B16, 1, 8192, True), (B16, 2, 8192, True), (B16, 8, 8192, False)])
def test_auto(dev, dtype, B, T, want):
    from atma_amd.layers.global_attention import PolarAttention
    layer = PolarAttention(1024, head_dim=128, num_kv_heads=2)
    assert layer._overlapped(B, T, dtype, dev) is want
    assert not layer._overlapped(B, T, dtype, dev, training=True)
    layer.overlap = False
    assert not layer._overlapped(B, T, dtype, dev)
    layer.overlap = True
    assert layer._overlapped(B, T, dtype, dev)
