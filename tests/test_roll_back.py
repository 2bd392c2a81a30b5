"""What a context falls back to when a queued store turns out to have failed: the last store that is good, looked at or not."""
import struct

import pytest
import torch

from kvcomp_amd import kvcomp_cuda
from kvcomp_amd._lib import KvcompError
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
from tests import _synth as S


def _config(k_mode=QuantMode.ChannelQuant):
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", k_mode, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


@pytest.mark.parametrize("longest,rows_kept", [(7, False), (8, True)])
def test_a_failed_second_store_leaves_a_prompt_that_nobody_has_looked_at(monkeypatch, longest, rows_kept):
    """Through store() with a library that queues nothing: the prompt's codes either rule its failure out (it stays) or do
    not (its rows were kept and return to the tail, and the codebook goes)."""
    from kvcomp_amd import _lib
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.async_store = True
    book = _lib.Codebook(tree_format=5, max_code_bits=longest, payload_bits=8 * 100000)
    sizes = []                                                    # payload bytes of the tiles of each call

    def encode(is_k, *, tokens, block_infos, encoded, **kw):
        n, at = tokens // 64 * 2, 0 if not sizes else sum(sizes)
        if not sizes:                                             # the second call fails and leaves nothing
            for i in range(n):
                block_infos[8 * i:8 * i + 8] = torch.frombuffer(bytearray(struct.pack("<IHH", at + 700 * i, 700, 0)), dtype=torch.uint8)
        sizes.append(700 * n)
    monkeypatch.setattr(kvcomp_cuda, "quant_codebook", lambda x, *a: (x.to(torch.uint8), book))
    monkeypatch.setattr(kvcomp_cuda, "put_codebook", lambda *a: tuple(torch.zeros(24, dtype=torch.uint8) for _ in range(3)))
    monkeypatch.setattr(kvcomp_cuda, "encode_async", encode)
    monkeypatch.setattr(KVCompCtx, "_issue_probe", lambda self: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    x = torch.arange(512 * 128, dtype=torch.float32).remainder(50).reshape(512, 1, 2, 64).to(torch.float16)
    ctx._encoded.reserve(1 << 20, (), torch.uint8, torch.device("cpu"))          # room for both: nothing has to be waited for
    ctx.store(x[:384], want_symbols=False)
    assert ctx.compressed_ctx_len == 384 and len(ctx._unverified) == 1
    ctx.store(x[384:], want_symbols=False)
    assert ctx.ctx_len == 512 and ctx.compressed_ctx_len == 512 and len(ctx._unverified) == 2

    def failed(*a):
        raise KvcompError("a symbol has no code")
    monkeypatch.setattr(kvcomp_cuda, "encode_result", failed)
    with pytest.raises(KvcompError, match="no code"):
        ctx.encoded_data
    assert ctx.ctx_len == 512 and not ctx._unverified and ctx._enc_pending == 0
    if rows_kept:
        assert ctx.compressed_ctx_len == 0 and torch.equal(ctx.buffer, x) and ctx.encoded_data.numel() == 0
        assert ctx.encode_codebook is None and ctx.decode_codebook is None
    else:
        assert ctx.compressed_ctx_len == 384 and torch.equal(ctx.buffer, x[384:]) and ctx.encoded_data.numel() == 12 * 700
        assert ctx.block_infos.numel() == 12 * 8 and ctx.max_tile_bytes == 700
        assert ctx._state[1:5].tolist() == [0, 0, 0, 12] and int(ctx._state[8]) == 12 * 700
        assert ctx.encode_codebook is not None and ctx.max_code_bits == longest


@pytest.mark.gpu
def test_a_second_store_that_fails_right_behind_the_prompt():
    _config(QuantMode.BlockQuant)
    dev, B, H, D = "cuda:0", 1, 2, 128
    flat = torch.zeros(64 * 12, B, H, D, dtype=torch.float16, device=dev)
    flat[::2] = 1.0                                               # two symbols only: 0 and 10
    wide = S.synth_k(64, B, H, D).to(dev)                         # needs the symbols in between
    ctx = KVCompCtx(True, B, H, D, 0.1)
    ctx.store(flat, want_symbols=False)
    good = ctx.encoded_data.clone()
    ctx = KVCompCtx(True, B, H, D, 0.1)
    ctx.async_store = True
    ctx._encoded.reserve(1 << 20, (), torch.uint8, torch.device(dev))    # room for both stores: nothing has to be waited for
    ctx.store(flat, want_symbols=False)                           # queued; codes of one bit cannot fail
    assert len(ctx._unverified) == 1
    ctx._probe = None                                             # as if its outcome were still on the way
    ctx.store(wide, want_symbols=False)
    assert len(ctx._unverified) == 2 and ctx.compressed_ctx_len == 64 * 13
    with pytest.raises(KvcompError, match="no code"):
        ctx.encoded_data
    assert ctx.ctx_len == 64 * 13 and ctx.compressed_ctx_len == 64 * 12 and torch.equal(ctx.buffer, wide)
    assert torch.equal(ctx.get()[0], torch.cat([flat, wide]))
    assert ctx.encoded_data.numel() == good.numel() and torch.equal(ctx.encoded_data, good)


def test_what_is_kept_says_how_long_its_streams_are(monkeypatch):
    """A prompt that nobody has looked at stays when the store behind it fails; the hint that the decoders' LDS is planned by covers its
    longest stream."""
    from kvcomp_amd import _lib
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.async_store = True
    book = _lib.Codebook(tree_format=5, max_code_bits=7, payload_bits=8 * 100000)
    lengths = torch.randint(9, 40, (12, 64), generator=torch.Generator().manual_seed(3))
    lengths[7, 0], lengths[9, 63] = 55, 51
    calls = []

    def encode(is_k, *, tokens, block_infos, thread_infos, encoded, **kw):
        if not calls:                                             # the second call fails and leaves nothing
            ends = lengths.cumsum(1)
            at = torch.cat([torch.zeros(1, dtype=torch.int64), ends[:, -1].cumsum(0)])
            for i in range(12):
                block_infos[8 * i:8 * i + 8] = torch.frombuffer(bytearray(struct.pack("<IHH", int(at[i]), int(ends[i, -1]), 0)), dtype=torch.uint8)
            thread_infos[:12 * 128] = ((ends << 3) + 5).to(torch.int16).view(torch.uint8).flatten()
        calls.append(tokens)
    monkeypatch.setattr(kvcomp_cuda, "quant_codebook", lambda x, *a: (x.to(torch.uint8), book))
    monkeypatch.setattr(kvcomp_cuda, "put_codebook", lambda *a: tuple(torch.zeros(24, dtype=torch.uint8) for _ in range(3)))
    monkeypatch.setattr(kvcomp_cuda, "encode_async", encode)
    monkeypatch.setattr(KVCompCtx, "_issue_probe", lambda self: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ctx._encoded.reserve(1 << 20, (), torch.uint8, torch.device("cpu"))
    x = torch.zeros(512, 1, 2, 64, dtype=torch.float16)
    ctx.store(x[:384], want_symbols=False)
    ctx.store(x[384:], want_symbols=False)
    assert calls == [384, 128]

    def failed(*a):
        raise KvcompError("a symbol has no code")
    monkeypatch.setattr(kvcomp_cuda, "encode_result", failed)
    with pytest.raises(KvcompError, match="no code"):
        ctx.encoded_data
    assert ctx.compressed_ctx_len == 384 and ctx.max_tile_bytes == int(lengths.sum(1).max()) and ctx.max_stream_bytes == 55
