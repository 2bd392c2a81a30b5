"""Payloads packed, packed and skewed, and in columns: the same symbols, values and order of sums, so results are equal bit for bit."""
import pytest
import torch

from kvcomp_amd import _lib
from tests import _synth as S
from tests.test_gpu_joint_attention import _contexts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _results(kc, vc, q, p):
    from kvcomp_amd.attention import CompressedAttention
    return CompressedAttention(kc, vc).attend(q).clone(), kc.mat_vec_mul(q)[0], vc.mat_vec_mul(p)[0]


# codes of 6 and 7 bits; short ones, two symbols per look-up; products that are not rounded
@pytest.mark.parametrize("eb_k,eb_v,smooth,rounded", [(0.1, 0.2, True, 1), (0.3, 0.5, False, 1), (0.1, 0.3, True, 0)])
@pytest.mark.parametrize("B,H,rep,D,T", [(1, 2, 1, 128, 64), (3, 2, 1, 96, 457), (1, 5, 2, 128, 700), (1, 8, 2, 72, 330), (1, 3, 4, 64, 1000), (2, 3, 4, 96, 257),
                                         (1, 4, 8, 128, 391)])
def test_every_layout_gives_the_same_bits(B, H, rep, D, T, eb_k, eb_v, smooth, rounded):
    kc, vc = _contexts(T, B, H, D, eb_k=eb_k, eb_v=eb_v, smooth=smooth)
    q = S.synth_q(B, H * rep, D).to(DEV)
    p = torch.softmax(torch.randn(B, H * rep, vc.compressed_ctx_len, generator=torch.Generator().manual_seed(1)), dim=-1).to(torch.float16).to(DEV)
    was = [(name, _lib.set_option(name, value)) for name, value in (("attention_joint", 0), ("fused_rounded", rounded))]
    try:
        got = []
        for layout in (0, 1, 2, -1):
            was.append(("fused_skew", _lib.set_option("fused_skew", layout)))
            got.append(_results(kc, vc, q, p) if vc.compressed_ctx_len else (kc.mat_vec_mul(q)[0],))
        # a stream hint that is too short: some tiles do not fit the columns and are decoded one symbol at a time
        _lib.set_option("fused_skew", 2)
        kc.max_stream_bytes = kc.max_stream_bytes * 9 // 10
        few = kc.mat_vec_mul(q)[0]
    finally:
        for name, value in reversed(was):
            _lib.set_option(name, value)
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    want = got[0][1 if vc.compressed_ctx_len else 0].float()
    # fp32 sums of at most 128 products in another order, rounded to fp16 (2^-11 of each result): 1e-3 of the largest covers both
    assert (few.float() - want).abs().max() <= 1e-3 * want.abs().max()


@pytest.mark.parametrize("rep,tiles", [(2, 2560), (8, 2560)])
def test_either_side_of_the_line_for_columns(rep, tiles):
    for T in (tiles // 8 * 64 - 64, tiles // 8 * 64):
        kc, _ = _contexts(T, 1, 8, 64)
        assert kc.max_code_bits in (6, 7) and kc.code_hint & 0x200
        q = S.synth_q(1, 8 * rep, 64).to(DEV)
        got = kc.mat_vec_mul(q)[0]
        was = _lib.set_option("fused_skew", 0)
        try:
            assert torch.equal(kc.mat_vec_mul(q)[0], got)
        finally:
            _lib.set_option("fused_skew", was)
