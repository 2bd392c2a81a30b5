"""A first store tells the encoder the room that its code needs.  The encoder chooses between kernels by the mean size that
tiles can have in that room; the quarter that a context's payload buffer keeps for growing made them look larger."""
import pytest
import torch

from kvcomp_amd import _lib, kvcomp_cuda
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode


@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("is_k", [True, False])
def test_the_room_is_what_the_code_needs(monkeypatch, is_k, prepared):
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)
    ctx = KVCompCtx(is_k, 1, 2, 64, 0.1)
    ctx.async_store = True
    book = _lib.Codebook(tree_format=5, max_code_bits=7, payload_bits=8 * 50000 + 3)
    told = []

    def quant_codebook(x, *args):
        args[-1](x.to(torch.uint8))
        return x.to(torch.uint8), book
    monkeypatch.setattr(kvcomp_cuda, "quant_codebook", quant_codebook)
    monkeypatch.setattr(kvcomp_cuda, "codebook_room", lambda device: None)
    monkeypatch.setattr(kvcomp_cuda, "put_codebook", lambda *a: tuple(torch.zeros(24, dtype=torch.uint8) for _ in range(3)))
    monkeypatch.setattr(kvcomp_cuda, "encode_prepare", lambda *a, tokens, **kw: kvcomp_cuda.PreparedEncode(
        None, None, 0, kvcomp_cuda.buffer_sizes(tokens, 128, is_k, 2, 64)))
    monkeypatch.setattr(kvcomp_cuda, "encode_prepared", lambda prepared, table, encoded, outcome, longest, room: told.append((encoded, room)))
    monkeypatch.setattr(kvcomp_cuda, "encode_async", lambda is_k, *, encoded, room, **kw: told.append((encoded, room)))
    monkeypatch.setattr(KVCompCtx, "_issue_probe", lambda self: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    if not prepared:
        ctx.device = torch.device("cpu")
        ctx._device_state()                                       # (as after a store that was taken back)
    ctx.store(torch.ones(1024, 1, 2, 64, dtype=torch.float16), want_symbols=False)
    vectors = ctx.compressed_ctx_len * 128 // (64 if is_k else 128)
    (encoded, room), = told
    assert room == 50000 + vectors + 1 and encoded.numel() >= room * 5 // 4
