"""The dense caches' two entry points at the sizes where they can go wrong: kvc_append_dense against PyTorch's fp16
rotation (bit for bit), kvc_quant_in_place against the CPU restatement of the reference's simulated quantization."""
import pytest
import torch

from tests import _synth as S
from tests.test_gpu_cache import _rope, _sim_cpu

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _no_quant():
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic
    KVCompCacheConfigStatic.extract_cache = None
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", None, None, None, None, None, None, None, None, enable_quant=False)


# groups of every layout: head_dim off 16 elements, blocks that do not fit a thread's registers, tokens that take a
# wave's registers (up to 8192 elements), a workgroup's (two sizes) and more than those
@pytest.mark.parametrize("mode,B,H,T,D,bs", [
    ("ChannelQuant", 2, 3, 192, 72, 64), ("ChannelQuant", 1, 2, 256, 64, 128), ("VectorQuant", 2, 3, 64, 72, 64),
    ("VectorQuant", 1, 5, 128, 128, 64), ("TokenQuant", 2, 3, 64, 40, 64), ("TokenQuant", 1, 17, 64, 128, 64),
    ("TokenQuant", 1, 64, 64, 128, 64), ("TokenQuant", 1, 80, 64, 104, 64), ("TokenQuant", 1, 260, 64, 128, 64),
    ("TokenQuant", 1, 520, 64, 128, 64), ("BlockQuant", 3, 5, 192, 72, 64), ("BlockQuant", 1, 2, 256, 128, 128),
    ("ChannelQuant", 1, 2, 64, 36, 64)])
def test_quantized_where_it_lies(mode, B, H, T, D, bs):
    from kvcomp_amd.compute import QuantMode, quant_in_place
    x = S.synth_k(T + 24, B, H, D).permute(1, 2, 0, 3).contiguous()
    cache = x.to(DEV).clone()
    quant_in_place(cache[:, :, 8:8 + T], bs, 0.1, QuantMode(mode))
    got = cache.cpu()
    assert torch.equal(got[:, :, :8], x[:, :, :8]) and torch.equal(got[:, :, 8 + T:], x[:, :, 8 + T:])
    assert torch.equal(got[:, :, 8:8 + T].view(torch.int16), _sim_cpu(x[:, :, 8:8 + T].contiguous(), bs, 0.1, mode).view(torch.int16))


@pytest.mark.parametrize("offset", [40.0, 12.0])
@pytest.mark.parametrize("mode", ["ChannelQuant", "TokenQuant", "VectorQuant", "BlockQuant"])
def test_quantized_where_it_lies_far_from_zero(mode, offset):
    from kvcomp_amd.compute import QuantMode, quant_in_place
    x = (torch.rand(1, 8, 128, 64, generator=torch.Generator().manual_seed(5)) * 0.5 + offset).to(torch.float16)
    got = x.to(DEV).clone()
    quant_in_place(got, 64, 0.1, QuantMode(mode))
    assert torch.equal(got.cpu().view(torch.int16), _sim_cpu(x, 64, 0.1, mode).view(torch.int16))


# 16-byte, 8-byte and single loads; keys as [B, T, H, D] memory; angles per batch entry; no rotation
@pytest.mark.parametrize("B,H,T,D,at", [(2, 3, 5, 128, 7), (1, 4, 1, 96, 0), (2, 2, 9, 72, 3), (1, 3, 4, 50, 2), (3, 1, 300, 64, 1)])
@pytest.mark.parametrize("angles", ["shared", "per entry", "none"])
def test_appended_rows_equal_the_rotation_in_pytorch(B, H, T, D, at, angles):
    from kvcomp_amd.compute import append_dense, apply_rotary_pos_emb_single
    k = S.synth_k(T, B, H, D).permute(1, 2, 0, 3).contiguous().to(DEV)
    v = S.synth_v(T, B, H, D).permute(1, 0, 2, 3).contiguous().to(DEV).transpose(1, 2)       # rows of a token adjacent
    cos, sin = (t.to(DEV) for t in _rope(T + 40, D))
    if angles == "none":
        cos = sin = None
        want = k
    else:
        pick = [torch.arange(T) + (7 * b if angles == "per entry" else 3) for b in range(B if angles == "per entry" else 1)]
        cos, sin = torch.stack([cos[0, p] for p in pick]), torch.stack([sin[0, p] for p in pick])
        want = apply_rotary_pos_emb_single(k, cos, sin)
    kc = torch.full((B, H, at + T + 3, D), 7.0, dtype=torch.float16, device=DEV)
    vc = kc.clone()
    assert append_dense(k, v, cos, sin, kc, vc, at)
    for cache, rows in ((kc, want), (vc, v)):
        assert torch.equal(cache[:, :, at:at + T].contiguous().view(torch.int16), rows.contiguous().view(torch.int16))
        assert (cache[:, :, :at] == 7).all() and (cache[:, :, at + T:] == 7).all()
    assert not append_dense(k, v, cos, sin, kc[:, :, :, :D - 2], vc[:, :, :, :D - 2], at)    # a cache of another shape


@pytest.mark.parametrize("wide", ["cos", "sin", "both"])
def test_angles_in_fp32_keep_the_keys_in_fp32(wide):
    """The rotation of fp16 keys by fp32 angles is fp32 in PyTorch, and the history holds it as it is."""
    from kvcomp_amd.cache import KVCompCachePytorchQuant
    from kvcomp_amd.compute import apply_rotary_pos_emb_single
    _no_quant()
    k = S.synth_k(12, 2, 3, 64).permute(1, 2, 0, 3).contiguous().to(DEV)
    cos, sin = (t.to(DEV).float() if wide in (n, "both") else t.to(DEV) for t, n in zip(_rope(12, 64), ("cos", "sin")))
    cache = KVCompCachePytorchQuant(2, 3, 64, 1)
    for lo, hi in ((0, 10), (10, 11), (11, 12)):
        keys, values = cache.update(k[:, :, lo:hi], k[:, :, lo:hi], 0, {"cos": cos[:, lo:hi], "sin": sin[:, lo:hi]})
    want = apply_rotary_pos_emb_single(k, cos, sin)
    assert want.dtype is torch.float32 and torch.equal(keys, want) and keys.dtype is torch.float32 and torch.equal(values, k)


def test_angles_of_several_sequences_spread_the_keys_of_one():
    from kvcomp_amd.cache import KVCompCachePytorchQuant
    from kvcomp_amd.compute import apply_rotary_pos_emb_single
    _no_quant()
    k = S.synth_k(5, 1, 3, 64).permute(1, 2, 0, 3).contiguous().to(DEV)
    cos, sin = (torch.cat([t[:, :5], t[:, 5:10]]).to(DEV) for t in _rope(10, 64))
    keys, _ = KVCompCachePytorchQuant(1, 3, 64, 1).update(k, k, 0, {"cos": cos, "sin": sin})
    assert torch.equal(keys, apply_rotary_pos_emb_single(k, cos, sin))
