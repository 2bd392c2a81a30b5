"""Codebooks with codes of more than 7 bits on the matrix-core and expansion kernels of their own (an escape list beside a
7-bit table): symbols drawn so that long codes are common, rare or absent, code lengths up to 15 and beyond the generic
table's 10 bits, against the decode path that reads the table one symbol at a time and against fp32 products of it."""
import pytest
import torch

from tests import _synth as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _contexts(T, B, H, D, shape, k_mode="BlockQuant", v_eb=0.2):
    """K whose symbols follow `shape`: a geometric ladder (long codes common), one level nearly always (long codes rare) or
    the synthetic keys at a fine bound (the longest codes belong to symbols that never occur)."""
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode(k_mode), QuantMode.TokenQuant, 64, 128, 64, 128, 0.05, v_eb)
    g = torch.Generator().manual_seed(7)
    if shape == "fine":
        k = S.synth_k(T, B, H, D)
    else:
        u = torch.rand(T, B, H, D, generator=g)
        level = torch.floor(-torch.log2(u) * (1.0 if shape == "ladder" else 0.6)).clamp(max=18)
        k = (level / 20.0).to(torch.float16)
        k[::64, 0, 0, 0], k[1::64, 0, 0, 0] = 0.0, 1.0          # every block spans 0 .. 1: the step is 0.05
    v = S.synth_v(T, B, H, D)
    ctxs = KVCompCtx(True, B, H, D, 0.05), KVCompCtx(False, B, H, D, v_eb)
    for c, x in zip(ctxs, (k, v)):
        c.codebook_smoothing = True
        c.store(x.to(DEV), want_symbols=False)
    return ctxs


@pytest.mark.parametrize("shape,k_mode", [("ladder", "BlockQuant"), ("rare", "BlockQuant"), ("fine", "BlockQuant"), ("fine", "ChannelQuant")])
@pytest.mark.parametrize("B,H,rep,D", [(1, 2, 1, 128), (2, 3, 2, 64), (1, 4, 4, 96), (1, 8, 8, 72), (1, 8, 1, 40)])
def test_long_codes_equal_the_slow_path(shape, k_mode, B, H, rep, D):
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(600, B, H, D, shape, k_mode)
    assert kc.code_hint & 0x100 and kc.max_code_bits > 7
    q = S.synth_q(B, H * rep, D).to(DEV)
    fast = CompressedAttention(kc, vc).attend(q)
    scores, _ = kc.mat_vec_mul(q)
    dense, sym = kc.get()[0], kc.get_decode_quant_ints()[0]
    was = _lib.set_option("fused_mfma", 0), _lib.set_option("decode_pipelined", 0)
    try:
        slow = CompressedAttention(kc, vc).attend(q)
        slow_scores, _ = kc.mat_vec_mul(q)
        assert torch.equal(kc.get_decode_quant_ints()[0], sym)
    finally:
        _lib.set_option("fused_mfma", was[0])
        _lib.set_option("decode_pipelined", was[1])
    n = kc.compressed_ctx_len
    want = torch.matmul(dense[:n].permute(1, 2, 0, 3).float().repeat_interleave(rep, dim=1), q.float().unsqueeze(-1)).squeeze(-1)
    assert (scores.float() - want).abs().max() <= 2e-3 * want.abs().max()
    assert (scores.float() - slow_scores.float()).abs().max() <= 2e-3 * want.abs().max()
    assert (fast - slow).abs().max() <= 1e-4 * slow.abs().max()
    from kvcomp_amd.compute import dequant
    assert torch.equal(dense[:n], dequant(sym, kc.quant_min_ints, kc.quant_scales, kc.quant_dims).flatten(0, 1))


@pytest.mark.parametrize("rep,D", [(1, 128), (4, 96), (2, 72)])
def test_long_codes_in_v(rep, D):
    """V at a fine bound: per-token groups with codes beyond 7 bits."""
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(600, 2, 8, D, "fine", v_eb=0.03)
    assert vc.max_code_bits > 7 and vc.code_hint & 0x100
    q = S.synth_q(2, 8 * rep, D).to(DEV)
    fast = CompressedAttention(kc, vc).attend(q)
    was = _lib.set_option("fused_mfma", 0)
    try:
        slow = CompressedAttention(kc, vc).attend(q)
    finally:
        _lib.set_option("fused_mfma", was)
    assert (fast - slow).abs().max() <= 1e-4 * slow.abs().max()
