"""Decode + dequantize in one kernel: how many elements go out at a time depends on K or V, code lengths and tile sizes.
Head sizes that leave every remainder, tiles on both sides of the size up to which K writes whole cache lines, size hints
absent; against decode followed by dequantization, bit for bit."""
import pytest
import torch

from tests import _synth as S
from tests.test_gpu_ctx import _config

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("is_k", [True, False])
@pytest.mark.parametrize("H,D", [(8, 8), (8, 24), (2, 64), (8, 72), (2, 96), (8, 104), (8, 120), (1, 128)])
@pytest.mark.parametrize("eb", [0.2, 0.03, 1.0 / 120.0])            # K tiles of 128 channels: 2, 5 and 7 KB
@pytest.mark.parametrize("hints", [True, False])
def test_equals_decode_then_dequant(is_k, H, D, eb, hints):
    from kvcomp_amd.ctx import KVCompCtx
    _config(k_mode="ChannelQuant", v_mode="TokenQuant")
    g = torch.Generator().manual_seed(D)
    x = (torch.rand(256, 1, H, D, generator=g) * 2.0 - 1.0).to(torch.float16).to(DEV)
    ctx = KVCompCtx(is_k, 1, H, D, eb)
    ctx.store(x)
    if not hints:
        ctx.max_tile_bytes = ctx.max_stream_bytes = 0
    try:
        one, _ = ctx.get_only_compressed()
        KVCompCtx.fused_get = False
        two, _ = ctx.get_only_compressed()
    finally:
        KVCompCtx.fused_get = True
    assert one.shape == (256, 1, H, D) and torch.equal(one.view(torch.int16), two.view(torch.int16))
