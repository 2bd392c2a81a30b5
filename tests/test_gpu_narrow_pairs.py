"""V decoded two symbols at a time through a table that not every pair of codes fits: tiles that meet a pair beyond it are
decoded again, so whatever width the caller states the results are those of the whole table."""
import pytest
import torch

from tests import _synth as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _contexts(T, B, H, D, eb_v, heavy=False):
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, eb_v)
    ctxs = KVCompCtx(True, B, H, D, 0.1), KVCompCtx(False, B, H, D, eb_v)
    for c, x in zip(ctxs, (S.synth_k(T, B, H, D), S.synth_laplace(T, B, H, D, 5) if heavy else S.synth_v(T, B, H, D))):
        c.codebook_smoothing = True
        c.store(x.to(DEV), want_symbols=False)
    return ctxs


@pytest.mark.parametrize("bits", [2, 3, 5, 6, 7])           # from "nearly every tile twice" to "none"
@pytest.mark.parametrize("B,H,rep,D", [(1, 4, 1, 128), (2, 3, 4, 64), (1, 8, 1, 96), (1, 8, 2, 72), (1, 8, 8, 48)])
@pytest.mark.parametrize("heavy", [True, False])
def test_any_width_gives_the_same(bits, B, H, rep, D, heavy, fused_mode):
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(700, B, H, D, 0.3, heavy)
    assert vc.max_code_bits in (5, 6, 7)
    q, att = S.synth_q(B, H * rep, D).to(DEV), CompressedAttention(kc, vc)
    p = torch.softmax(S.synth_q(B, H * rep, vc.compressed_ctx_len).float() * 3, dim=-1).to(torch.float16).to(DEV)
    was = _lib.set_option("attention_joint", 0)
    try:
        vc.pair_bits = 0
        want, want_mv = att.attend(q), vc.mat_vec_mul(p)[0]
        vc.pair_bits = bits
        got, got_mv = att.attend(q), vc.mat_vec_mul(p)[0]
    finally:
        _lib.set_option("attention_joint", was)
    assert torch.equal(got, want) and torch.equal(got_mv, want_mv)


@pytest.mark.parametrize("heavy", [True, False])
def test_the_first_store_states_the_narrowest_width(heavy):
    _, vc = _contexts(4096, 1, 8, 128, 0.3, heavy)
    lengths = vc.encode_codebook.view(torch.int32)[1::2].cpu()
    counts = torch.bincount(vc.get_decode_quant_ints()[0].flatten().int().cpu(), minlength=256)[:lengths.numel()].double()
    share = torch.zeros(33, dtype=torch.float64).index_add_(0, lengths.clamp(max=32).long(), counts / counts.sum())
    both = torch.outer(share, share)
    total = torch.arange(33)[:, None] + torch.arange(33)[None, :]
    fits = [w for w in range(2, 8) if float(both[total > w].sum()) <= 5e-6]
    assert vc.pair_bits == (fits[0] if fits else 0)
    assert vc.code_hint >> 12 & 7 == vc.pair_bits and vc.code_hint & 0xff == vc.max_code_bits
