"""The kernel whose waves take a 128-token group each (two K tiles, then two V tiles, at a time) against the two kernels it stands
in for: the same symbols, fp16 values, operand splits and order of sums, so the results are equal bit for bit."""
import pytest
import torch

from tests import _synth as S
from tests.test_gpu_joint_attention import _contexts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _attend(kc, vc, q, joint):
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    was = _lib.set_option("attention_joint", joint)
    try:
        return CompressedAttention(kc, vc).attend(q).clone()
    finally:
        _lib.set_option("attention_joint", was)


# T: one group and nothing else, a token more; K a block ahead of V; every number of groups in the last workgroup; both tails
@pytest.mark.parametrize("T", [128, 129, 192, 257, 448, 520, 700, 1000])
@pytest.mark.parametrize("B,H,rep", [(1, 1, 1), (3, 2, 2), (1, 8, 4), (1, 2, 8)])
@pytest.mark.parametrize("skew", [0, 1, 2])
def test_equals_the_two_kernels(T, B, H, rep, skew):
    from kvcomp_amd import _lib
    kc, vc = _contexts(T, B, H, 128)
    assert kc.code_hint & 0x200 and vc.code_hint & 0x200 and kc.max_code_bits in (6, 7) and vc.max_code_bits in (6, 7)
    q = S.synth_q(B, H * rep, 128).to(DEV)
    got = _attend(kc, vc, q, 2)
    was = _lib.set_option("fused_skew", skew)                   # how the two kernels' payloads lie
    try:
        want = _attend(kc, vc, q, 0)
    finally:
        _lib.set_option("fused_skew", was)
    assert torch.isfinite(got).all() and torch.equal(want, got)


@pytest.mark.parametrize("k_mode,v_mode,B", [("BlockQuant", "VectorQuant", 2), ("ChannelQuant", "VectorQuant", 1), ("ChannelQuant", "TokenQuant", 2)])
@pytest.mark.parametrize("eb_k,eb_v", [(0.1, 0.2), (0.2, 0.3), (0.08, 0.12), (0.05, 0.05)])
def test_code_lengths_and_layouts(k_mode, v_mode, B, eb_k, eb_v):
    """(where the codes are not this kernel's, the call goes to the others; its own in test_gpu_waves_default.py)"""
    kc, vc = _contexts(330, B, 3, 128, k_mode, v_mode, eb_k, eb_v)
    q = S.synth_q(B, 6, 128).to(DEV)
    assert torch.equal(_attend(kc, vc, q, 0), _attend(kc, vc, q, 2))


@pytest.mark.parametrize("hint", ["too_small", "absent", "bits"])
def test_wrong_or_missing_size_hints(hint):
    """Tiles that do not fit the LDS areas, or tables that are not what the hint says, are decoded one symbol at a time."""
    kc, vc = _contexts(600, 1, 4, 128)
    q = S.synth_q(1, 8, 128).to(DEV)
    want = _attend(kc, vc, q, 0)
    for c in (kc, vc):
        if hint == "bits":
            c.max_code_bits = 13 - c.max_code_bits
        else:
            c.max_tile_bytes = c.max_stream_bytes = 64 if hint == "too_small" else 0
    got = _attend(kc, vc, q, 2)
    # sums of 128 products one by one in fp32 instead of four at a time: 128 roundings of 2^-24, then the softmax
    assert (got - want).abs().max() <= 1e-5 * want.abs().max()


def test_subnormal_and_infinite_queries():
    kc, vc = _contexts(300, 1, 4, 128)
    q = S.synth_q(1, 4, 128)
    q[0, 0] *= 1e-4
    q[0, 0, 0], q[0, 1, 0] = 3e-7, float("inf")
    two, waves = (_attend(kc, vc, q.to(DEV), joint) for joint in (0, 2))
    assert torch.equal(torch.isnan(two), torch.isnan(waves)) and torch.equal(torch.nan_to_num(two), torch.nan_to_num(waves))
