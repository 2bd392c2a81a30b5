"""The kernel that decodes K and V of a 128-token group in one workgroup against the two kernels it stands in for: the same
symbols, fp16 values, operand splits and order of sums, so the results are equal bit for bit."""
import pytest
import torch

from tests import _synth as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _contexts(T, B, H, D, k_mode="ChannelQuant", v_mode="TokenQuant", eb_k=0.1, eb_v=0.2, smooth=True):
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode(k_mode), QuantMode(v_mode), 64, 128, 64, 128, eb_k, eb_v)
    ctxs = KVCompCtx(True, B, H, D, eb_k), KVCompCtx(False, B, H, D, eb_v)
    for c, x in zip(ctxs, (S.synth_k(T, B, H, D), S.synth_v(T, B, H, D))):
        c.codebook_smoothing = smooth
        c.store(x.to(DEV), want_symbols=False)
    return ctxs


def _both(kc, vc, q):
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    att, outs = CompressedAttention(kc, vc), []
    for joint in (0, 1):
        was = _lib.set_option("attention_joint", joint)
        try:
            outs.append(att.attend(q))
        finally:
            _lib.set_option("attention_joint", was)
    return outs


# T: one group and nothing else, a token more; K a block ahead of V (every number of waves in the K-only workgroups' last
# one); both tails
@pytest.mark.parametrize("T", [128, 129, 192, 193, 257, 448, 1000])
@pytest.mark.parametrize("B,H,rep,D", [(1, 1, 1, 128), (1, 3, 1, 64), (3, 2, 2, 128), (2, 5, 4, 64), (1, 8, 4, 128), (1, 2, 8, 128), (2, 1, 8, 64)])
def test_equals_the_two_kernels(T, B, H, rep, D):
    kc, vc = _contexts(T, B, H, D)
    two, joint = _both(kc, vc, S.synth_q(B, H * rep, D).to(DEV))
    assert torch.isfinite(joint).all() and torch.equal(two, joint)


@pytest.mark.parametrize("eb_k", [0.1, 0.15, 0.2, 0.3, 0.5])          # codes of different lengths: one or two symbols per look-up
@pytest.mark.parametrize("eb_v", [0.1, 0.2, 0.3, 0.5])
@pytest.mark.parametrize("smooth", [True, False])
@pytest.mark.parametrize("k_mode,v_mode", [("ChannelQuant", "TokenQuant"), ("BlockQuant", "VectorQuant")])
def test_code_lengths_and_layouts(eb_k, eb_v, smooth, k_mode, v_mode):
    kc, vc = _contexts(330, 2, 3, 128, k_mode, v_mode, eb_k, eb_v, smooth)
    two, joint = _both(kc, vc, S.synth_q(2, 6, 128).to(DEV))
    assert torch.equal(two, joint)


@pytest.mark.parametrize("hint", ["too_small", "absent", "bits"])
def test_wrong_or_missing_size_hints(hint):
    """Tiles that do not fit the LDS areas, or tables that are not what the hint says, are decoded from global memory."""
    kc, vc = _contexts(600, 1, 4, 128)
    q = S.synth_q(1, 8, 128).to(DEV)
    want = _both(kc, vc, q)[0]
    for c in (kc, vc):
        if hint == "bits":
            c.max_code_bits = 3
        else:
            c.max_tile_bytes = c.max_stream_bytes = 64 if hint == "too_small" else 0
    got = _both(kc, vc, q)[1]
    assert (got - want).abs().max() <= 1e-5 * want.abs().max()


def test_subnormal_and_infinite_queries():
    kc, vc = _contexts(300, 1, 4, 128)
    q = S.synth_q(1, 4, 128)
    q[0, 0] *= 1e-4
    q[0, 0, 0], q[0, 1, 0] = 3e-7, float("inf")
    two, joint = _both(kc, vc, q.to(DEV))
    assert torch.equal(torch.isnan(two), torch.isnan(joint)) and torch.equal(torch.nan_to_num(two), torch.nan_to_num(joint))
