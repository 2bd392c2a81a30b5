"""A first store's codebook and encode in one native call: the same context as by the calls from Python, a codebook that is not for it left
to those, and a failure that leaves the context as it was."""
import pytest
import torch

from kvcomp_amd import _lib
from tests.test_gpu_packed_symbols import HELD, _ctx, _data

pytestmark = pytest.mark.gpu


@pytest.fixture
def calls(monkeypatch):
    """What first_encode has returned."""
    host, made = _lib.host(), []

    class Host:
        append_rows = staticmethod(host.append_rows)

        @staticmethod
        def first_encode(*args):
            made.append(host.first_encode(*args))
            return made[-1]
    monkeypatch.setattr(_lib, "host", lambda: Host)
    return made


@pytest.mark.parametrize("is_k,mode,shape,eb,wide,taken", [
    (True, "ChannelQuant", (64, 1, 1, 64), 0.1, False, True), (True, "ChannelQuant", (777, 2, 3, 96), 0.1, True, True), (False, "TokenQuant", (300, 1, 8, 128), 0.2, False, True),
    (True, "BlockQuant", (640, 1, 8, 128), 0.1, True, False)])                  # codes of more than seven bits
def test_the_same_context(monkeypatch, calls, is_k, mode, shape, eb, wide, taken):
    x = _data(*shape, wide, 3)
    got, want = _ctx(is_k, mode, *shape[1:], eb, True), _ctx(is_k, mode, *shape[1:], eb, True)
    got.store(x, want_symbols=False)
    assert len(calls) == 1 and calls[0][:2] == (0, 0) and (calls[0][3] is not None) == taken and (got.max_code_bits <= 7) == taken
    with monkeypatch.context() as p:
        p.setattr(_lib, "hooked", lambda: True)
        want.store(x, want_symbols=False)
    assert len(calls) == 1
    for name in HELD + ("max_code_bits", "pair_bits", "max_tile_bytes", "max_stream_bytes", "waits", "ctx_len", "compressed_ctx_len", "tree_format"):
        a, b = getattr(got, name), getattr(want, name)
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a == b, name
    assert got._encoded.data.numel() == want._encoded.data.numel()


def test_a_refused_encode_leaves_the_context_as_it_was(monkeypatch, calls):
    x = _data(256, 1, 2, 64, False, 1)
    ctx = _ctx(True, "ChannelQuant", 1, 2, 64, 0.1, True)
    prepare = type(ctx)._prepare_encode

    def spoiled(self, *args):
        p = prepare(self, *args)
        p.job.heads = 0
        return p
    with monkeypatch.context() as m:
        m.setattr(type(ctx), "_prepare_encode", spoiled)
        with pytest.raises(_lib.KvcompError):
            ctx.store(x, want_symbols=False)
    assert calls[-1][0] == 0 and calls[-1][1] != 0 and ctx.compressed_ctx_len == 0 and ctx.encode_codebook is None
    ctx.store(x, want_symbols=False)
    want = _ctx(True, "ChannelQuant", 1, 2, 64, 0.1, True)
    want.store(x, want_symbols=False)
    assert all(torch.equal(getattr(ctx, name), getattr(want, name)) for name in HELD)
