"""Decode attention of caches either side of the line from which a wave takes a group, by the rule that users get, and with streams of
uneven length; equal bit for bit to the two kernels."""
import ctypes as C

import pytest
import torch

from kvcomp_amd import _lib
from kvcomp_amd.attention import CompressedAttention
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
from tests import _synth as S
from tests.test_gpu_joint_attention import _contexts as _some_contexts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TWO_KERNELS, JOINT, WAVES = range(3)


def _contexts(T, B, H, odd=()):
    """odd: tokens of the second head whose every element is its block's largest: all their symbols are rare ones"""
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)
    g = torch.Generator(device=DEV).manual_seed(T)
    k, v = (torch.randn(T, B, H, 128, generator=g, device=DEV).to(torch.float16) for _ in range(2))
    for t in odd:
        k[t, 0, 1] = k[t // 64 * 64:t // 64 * 64 + 64, 0, 1].amax(0)
    ctxs = KVCompCtx(True, B, H, 128, 0.1), KVCompCtx(False, B, H, 128, 0.2)
    for c, x in zip(ctxs, (k, v)):
        c.codebook_smoothing = True
        c.store(x, want_symbols=False)
        assert c.max_code_bits in (6, 7) and c.code_hint & 0x200 and c.pair_bits == 0
    return ctxs


def _route(kc, vc, B, H, rep):
    """KvcAttendRoute of the call"""
    return _lib.lib().kvc_attention_kernels(C.byref(kc.descriptor()), C.byref(vc.descriptor()), *(C.c_int64(n) for n in (B, H, H * rep, 128))) >> 8


def _equal(kc, vc, q, joint):
    outs = []
    for value in (0, joint):
        was = _lib.set_option("attention_joint", value)
        try:
            outs.append(CompressedAttention(kc, vc).attend(q).clone())
        finally:
            _lib.set_option("attention_joint", was)
    return torch.isfinite(outs[0]).all() and torch.equal(*outs)


@pytest.mark.parametrize("groups,T,want", [(6, 777, JOINT), (6, 831, JOINT), (7, 900, WAVES), (8, 1030, WAVES), (9, 1279, WAVES)])
@pytest.mark.parametrize("rep", [1, 4, 8])
def test_either_side_of_the_line(groups, T, want, rep):
    kc, vc = _contexts(T, 8, 32)
    assert vc.compressed_ctx_len // 128 == groups and _route(kc, vc, 8, 32, rep) == want
    assert _equal(kc, vc, S.synth_q(8, 32 * rep, 128).to(DEV), -1)


@pytest.mark.parametrize("rep", [1, 2, 4, 8])
def test_a_token_of_rare_symbols(rep):
    """One stream as long as streams get, or a hint that says so: the cache goes to other kernels, and to this one where it is asked for and
    fits."""
    kc, vc = _contexts(1279, 8, 32, odd=(70, 391))
    assert kc.max_stream_bytes > 1.4 * kc.encoded_data.numel() / (kc.compressed_ctx_len * 8 * 32)
    q = S.synth_q(8, 32 * rep, 128).to(DEV)
    assert _equal(kc, vc, q, -1)
    kc.max_stream_bytes = 112
    assert _route(kc, vc, 8, 32, rep) == (JOINT if rep == 8 else TWO_KERNELS) and _equal(kc, vc, q, -1) and _equal(kc, vc, q, 1)
    small = _contexts(900, 1, 2, odd=(70, 391))
    assert _equal(*small, S.synth_q(1, 2 * rep, 128).to(DEV), 2)


@pytest.mark.parametrize("k_mode,v_mode,B", [("BlockQuant", "VectorQuant", 2), ("BlockQuant", "TokenQuant", 1), ("ChannelQuant", "VectorQuant", 1),
                                             ("ChannelQuant", "TokenQuant", 2)])
@pytest.mark.parametrize("eb_k,eb_v", [(0.2, 0.2), (0.2, 0.25), (0.25, 0.2), (0.3, 0.3)])
def test_layouts_of_both_code_lengths(k_mode, v_mode, B, eb_k, eb_v):
    kc, vc = _some_contexts(330, B, 3, 128, k_mode, v_mode, eb_k, eb_v)
    assert kc.max_code_bits in (6, 7) and vc.max_code_bits in (6, 7)
    q = S.synth_q(B, 6, 128).to(DEV)
    was = _lib.set_option("attention_joint", 2)
    try:
        assert _route(kc, vc, B, 3, 2) == WAVES
    finally:
        _lib.set_option("attention_joint", was)
    assert _equal(kc, vc, q, 2)


@pytest.mark.parametrize("longest", [0, 40, 56])
def test_a_stream_hint_that_is_absent_or_too_short(longest):
    """Tiles with longer streams are decoded one symbol at a time: sums of 128 products one by one in fp32 instead of four at a time, 128
    roundings of 2^-24, then the softmax."""
    kc, vc = _contexts(900, 8, 32)
    q = S.synth_q(8, 32, 128).to(DEV)
    want = CompressedAttention(kc, vc).attend(q).clone()
    kc.max_stream_bytes = vc.max_stream_bytes = longest
    got = CompressedAttention(kc, vc).attend(q)
    assert (got - want).abs().max() <= 1e-5 * want.abs().max()
