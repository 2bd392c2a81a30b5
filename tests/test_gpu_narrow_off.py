"""V's narrow two-symbol table is turned off for a codebook whose tiles mostly meet pairs beyond it, by the calls themselves and
on the device; what counts as a miss, and that results do not depend on it."""
import pytest
import torch

from tests import _synth as S
from tests.test_gpu_narrow_pairs import _contexts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NARROW = 8 + 512 + 1024 + 1024 + 128                 # KVC_LUT_NARROW_OFFSET: 64 counters, one per 64 bytes


def _words(ctx):
    """(turned off, tiles counted as missed since a call last looked)"""
    words = ctx.decode_lut().view(torch.int32)
    counters = words[NARROW:].view(64, 16)
    assert not counters[:, 1:].any()
    return [int(words[6] < 0), int(counters[:, 0].sum())]


@pytest.fixture(autouse=True)
def the_kernels_that_have_the_table():
    """... whatever the environment presets."""
    from kvcomp_amd import _lib
    was = {name: _lib.set_option(name, value) for name, value in (("attention_joint", 0), ("fused_mfma", -1), ("fused_pair_bits", 8), ("fused_rows", -1))}
    yield
    for name, value in was.items():
        _lib.set_option(name, value)


@pytest.mark.parametrize("by", ["attend", "mat_vec_mul"])
@pytest.mark.parametrize("B,H,rep,D", [(1, 4, 1, 128), (2, 3, 4, 64), (1, 8, 1, 96), (1, 8, 2, 72), (1, 8, 8, 48)])
def test_a_table_that_most_tiles_miss_is_turned_off(by, B, H, rep, D):
    from kvcomp_amd.attention import CompressedAttention
    kc, vc = _contexts(1500, B, H, D, 0.3)
    p = torch.softmax(S.synth_q(B, H * rep, vc.compressed_ctx_len).float() * 3, dim=-1).to(torch.float16).to(DEV)
    q, att = S.synth_q(B, H * rep, D).to(DEV), CompressedAttention(kc, vc)
    call = (lambda: att.attend(q)) if by == "attend" else (lambda: vc.mat_vec_mul(p)[0])
    vc.pair_bits = 0
    want = call()
    assert _words(vc) == [0, 0]
    vc.pair_bits = 2
    for _ in range(3):                                # tried, and off from the second call on
        assert torch.equal(call(), want) and _words(vc) == [1, 0]
    vc._lut_source = None                             # tables of a codebook put in place anew
    vc.pair_bits = 7
    assert _words(vc) == [0, 0] and torch.equal(call(), want)


def _few_misses():
    """Contexts of which twelve of V's 576 tiles (those of the rare values) meet pairs that seven bits do not hold."""
    from kvcomp_amd.ctx import KVCompCtx
    _contexts(128, 1, 24, 128, 0.3)                    # (the configuration)
    g = torch.Generator().manual_seed(3)
    x = torch.where(torch.rand(12 * 128, 1, 24, 128, generator=g) < 0.9, 0.0, 1.0)
    x[:, :, 0, 0], x[:, :, 0, 1], x[:, :, 0, 2] = 0.5, 1.5, 0.0       # every token spans 0 .. 1.5: the step is 0.45
    pair = KVCompCtx(True, 1, 24, 128, 0.1), KVCompCtx(False, 1, 24, 128, 0.3)
    for c, t in zip(pair, (S.synth_k(12 * 128, 1, 24, 128), x.to(torch.float16))):
        c.codebook_smoothing = True
        c.store(t.to(DEV), want_symbols=False)
    return pair


def _misses(v):
    """Tiles of V whose lanes meet a pair of codes of more than seven bits, from the symbols."""
    lengths = v.encode_codebook.view(torch.int32)[1::2].cpu()
    assert lengths.max() <= 7 and 2 * lengths.max() > 8, lengths      # (else the whole pair table is taken)
    bits = lengths[v.get_decode_quant_ints()[0].flatten(2).int().cpu()]          # [rows, 128 tokens, channels]
    beyond = (bits[:, 0::2] + bits[:, 1::2]) > 7
    return int(beyond.reshape(bits.shape[0], 64, -1, 64).any(dim=3).any(dim=1).sum())


def test_a_table_that_few_tiles_miss_stays_on():
    from kvcomp_amd.attention import CompressedAttention, v_partials
    k, v = _few_misses()
    missed = _misses(v)
    assert missed == 12
    q, att = S.synth_q(1, 24, 128).to(DEV), CompressedAttention(k, v)
    p = torch.softmax(S.synth_q(1, 24, v.compressed_ctx_len).float() * 3, dim=-1).to(torch.float16).to(DEV)
    v.pair_bits = 0
    want, want_p = att.attend(q), v_partials(v, v.decode_lut(), p)[0]
    v.pair_bits = 7
    assert torch.equal(v_partials(v, v.decode_lut(), p)[0], want_p) and _words(v) == [0, missed]       # counted
    for _ in range(8):
        assert torch.equal(att.attend(q), want) and _words(v) == [0, 0]           # looked at, kept on


def test_queries_that_are_not_numbers_are_no_misses():
    from kvcomp_amd.attention import CompressedAttention, v_partials
    k, v = _few_misses()
    missed = _misses(v)
    v.pair_bits = 7
    q, att = S.synth_q(1, 24, 128).to(DEV), CompressedAttention(k, v)
    want = att.attend(q)
    bad, p = q.clone(), torch.full((1, 24, v.compressed_ctx_len), float("nan"), dtype=torch.float16, device=DEV)
    bad[0, :, 5] = float("nan")
    assert torch.isnan(att.attend(bad)).all() and _words(v) == [0, 0]
    assert torch.isnan(v_partials(v, v.decode_lut(), p)[0]).all() and _words(v) == [0, 0]
    assert torch.equal(att.attend(q), want) and missed > 0
