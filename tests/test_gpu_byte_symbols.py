"""Codes of 6 or 7 bits of symbols up to 16: table entries with the symbol in one byte, by kernels of their own.  The other
two-byte and the four-byte entries give the same values to the last bit, so every comparison is exact."""
import pytest
import torch

from tests import _synth as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _contexts(T, B, H, D, symbols):
    """K whose blocks span `symbols` levels, most entries on few of them; V of a normal distribution."""
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    eb = 1.0 / (symbols - 1)
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, eb, 0.2)
    g = torch.Generator().manual_seed(symbols)
    p = torch.tensor([2.0 ** -min(1 + abs(i - symbols // 2) / 2, 3 if symbols > 12 else 4) for i in range(symbols)])
    level = torch.multinomial(p, T * B * H * D, replacement=True, generator=g).view(T, B, H, D)
    level[::64], level[1::64] = 0, symbols - 1
    k = (level.float() - 3.0).to(torch.float16)                 # steps of one
    v = S.synth_v(T, B, H, D)
    ctxs = KVCompCtx(True, B, H, D, eb), KVCompCtx(False, B, H, D, 0.2)
    for c, x in zip(ctxs, (k, v)):
        c.codebook_smoothing = True
        c.store(x.to(DEV), want_symbols=False)
    return ctxs


@pytest.mark.parametrize("symbols", [11, 15, 17])       # smoothing gives two more a code: 15 come to symbols 0 .. 16, 17 are too many
@pytest.mark.parametrize("B,H,rep,D", [(1, 2, 1, 128), (2, 3, 2, 64), (1, 4, 4, 96), (1, 8, 8, 72)])
def test_every_entry_form_gives_the_same_bits(symbols, B, H, rep, D):
    from kvcomp_amd import _lib
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(600, B, H, D, symbols)
    assert kc.max_code_bits in (6, 7) and kc.encode_codebook.shape[0] // 8 == symbols + 2 and bool(kc.code_hint & 0x200) == (symbols <= 15)
    q = S.synth_q(B, H * rep, D).to(DEV)
    p = torch.softmax(torch.randn(B, H * rep, vc.compressed_ctx_len, generator=torch.Generator().manual_seed(1)), dim=-1).to(torch.float16).to(DEV)

    def results():
        return CompressedAttention(kc, vc).attend(q).clone(), kc.mat_vec_mul(q)[0], vc.mat_vec_mul(p)[0]
    was_joint = _lib.set_option("attention_joint", 0)
    was = []
    try:
        got = results()
        was.append(("fused_half_table", _lib.set_option("fused_half_table", 0)))
        for a, b in zip(got, results()):
            assert torch.equal(a, b)
        was.append(("fused_skew", _lib.set_option("fused_skew", 1)))
        _lib.set_option("fused_half_table", 1)
        for a, b in zip(got, results()):
            assert torch.equal(a, b)
    finally:
        _lib.set_option("attention_joint", was_joint)
        for name, value in was:
            _lib.set_option(name, value)
    n = kc.compressed_ctx_len
    want = torch.matmul(kc.get()[0][:n].permute(1, 2, 0, 3).float().repeat_interleave(rep, dim=1), q.float().unsqueeze(-1)).squeeze(-1)
    # fp32 sums of at most 128 products, rounded to fp16 (2^-11 of each result): 1e-3 of the largest covers both
    assert (got[1].float() - want).abs().max() <= 1e-3 * want.abs().max()


def test_symbols_beyond_what_the_hint_states_take_the_slow_path():
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(300, 1, 2, 128, 20)
    q = S.synth_q(1, 2, 128).to(DEV)
    want = kc.mat_vec_mul(q)[0]
    hint = type(kc).code_hint
    try:
        type(kc).code_hint = property(lambda c: hint.fget(c) | 0x200)
        got = kc.mat_vec_mul(q)[0]
    finally:
        type(kc).code_hint = hint
    # the slow path's products are added up one by one in fp32: 128 roundings of 2^-24, then fp16's 2^-11
    assert (got.float() - want.float()).abs().max() <= 1e-3 * want.float().abs().max()


@pytest.mark.parametrize("T", [32704, 32768])           # (the line from which columns are taken: test_gpu_payload_layouts.py)
def test_eight_query_heads(T):
    from kvcomp_amd import _lib
    kc, _ = _contexts(T, 1, 8, 64, 11)
    assert kc.code_hint & 0x200 and kc.max_code_bits in (6, 7) and (kc.compressed_ctx_len // 64 * 8 >= 4096) == (T == 32768)
    q = S.synth_q(1, 64, 64).to(DEV)
    got = kc.mat_vec_mul(q)[0]
    was = _lib.set_option("fused_half_table", 0)
    try:
        assert torch.equal(kc.mat_vec_mul(q)[0], got)
    finally:
        _lib.set_option("fused_half_table", was)
