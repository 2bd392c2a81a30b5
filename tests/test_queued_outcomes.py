"""What a context learns of its queued stores where something else goes wrong or differs: a later call that the library refuses,
streams other than the one its buffers came from, buffers that grow meanwhile."""
import struct
import time
import types

import pytest
import torch

from kvcomp_amd import _lib, kvcomp_cuda
from kvcomp_amd._lib import KvcompError
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode, _Growable, _Outcome

DEV = "cuda:0"


def _config():
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


def _ordinary_words():
    """An _Outcome in ordinary memory: the test writes what a kernel would."""
    outcome = object.__new__(_Outcome)
    outcome.words = torch.zeros(16, dtype=torch.int32)
    outcome._seen, outcome.number, outcome.stream = outcome.words.numpy(), 0, 0
    return outcome


@pytest.fixture
def queued(monkeypatch):
    """A context with one queued store of 384 tokens through a library that queues nothing, and the list of what its encodes
    were told; an encode fails while `refuse` is not empty."""
    _config()
    ctx, told, refuse = KVCompCtx(True, 1, 2, 64, 0.1), [], []
    ctx.async_store, ctx._outcome = True, _ordinary_words()
    book = _lib.Codebook(tree_format=5, max_code_bits=7, payload_bits=8 * 100000)

    def encode(is_k, *, tokens, block_infos, outcome, **kw):
        if refuse:
            raise KvcompError("the library refuses the call")
        for i in range(tokens // 64 * 2):
            block_infos[8 * i:8 * i + 8] = torch.frombuffer(bytearray(struct.pack("<IHH", 700 * i, 700, 0)), dtype=torch.uint8)
        told.append(outcome)
    monkeypatch.setattr(kvcomp_cuda, "quant_codebook", lambda x, *a: (x.to(torch.uint8), book))
    monkeypatch.setattr(kvcomp_cuda, "put_codebook", lambda *a: tuple(torch.zeros(24, dtype=torch.uint8) for _ in range(3)))
    monkeypatch.setattr(kvcomp_cuda, "encode_async", encode)
    monkeypatch.setattr(KVCompCtx, "_ask_outcome", lambda self: self._outcome)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 11)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(synchronize=lambda: None))
    x = torch.arange(512 * 128, dtype=torch.float32).remainder(50).reshape(512, 1, 2, 64).to(torch.float16)
    ctx._encoded.reserve(1 << 20, (), torch.uint8, torch.device("cpu"))
    ctx.store(x[:384], want_symbols=False)
    assert len(ctx._unverified) == 1 and ctx._probe is not None
    return ctx, told, refuse, x


def _arrives(outcome, number, used, largest):
    outcome.words[2], outcome.words[3], outcome.words[8], outcome.words[9] = largest, 40, used, number


@pytest.mark.parametrize("arrives", ["before", "behind"])
def test_a_refused_encode_does_not_hide_the_outcome_of_an_earlier_one(queued, arrives):
    ctx, told, refuse, x = queued
    if arrives == "before":
        _arrives(ctx._outcome, told[0][1], 12 * 700, 700)
        ctx._probe, probe = None, ctx._probe                      # (store() would take note of it at once)
    refuse.append(True)
    with pytest.raises(KvcompError, match="refuses"):
        ctx.store(x[384:], want_symbols=False)
    if arrives == "before":
        ctx._probe = probe
    else:
        assert not ctx._outcome.query() and ctx._outcome.stream == 11
        _arrives(ctx._outcome, told[0][1], 12 * 700, 700)
    assert ctx._outcome.query()
    ctx.poll_stores()
    assert not ctx._unverified and ctx._enc_pending == 0 and ctx._encoded.used == 12 * 700 and ctx.max_tile_bytes == 700
    seen = ctx._outcome._seen
    ctx._outcome = ctx._probe = None
    assert not any(words is seen for words, _ in _Outcome._late)  # nothing is still to come
    refuse.clear()
    ctx._outcome = _ordinary_words()
    ctx.store(x[384:], want_symbols=False)                        # the refused store, again
    assert ctx.ctx_len == 512 and len(ctx._unverified) == 1 and told[1][1] == ctx._outcome.number != told[0][1]


def test_a_refused_encode_whose_last_kernel_ran_all_the_same():
    outcome = _ordinary_words()
    first = outcome.ask(11)[1]
    second = outcome.ask(11)[1]
    outcome.words[9] = second
    outcome.refused(first, 11)
    assert outcome.query() and outcome.number == second


def _store_all(is_k, parts, refuse_behind=()):
    B, H, D = parts[0].shape[1:]
    ctx = KVCompCtx(is_k, B, H, D, 0.1)
    ctx.codebook_smoothing = ctx.async_store = True
    for i, x in enumerate(parts):
        ctx.store(x, want_symbols=False)
        if i in refuse_behind:
            ctx.quant_scale_rel = 0.0
            probe, ctx._probe = ctx._probe, None                  # as if nothing of the queued stores had arrived when store() looked
            with pytest.raises(KvcompError, match="error bound"):
                ctx.store(x, want_symbols=False)
            ctx.quant_scale_rel, ctx._probe = 0.1, probe
    return ctx


@pytest.mark.gpu
@pytest.mark.parametrize("is_k", [True, False])
def test_stores_around_a_refused_one(is_k):
    from tests import _synth as S
    _config()
    x = (S.synth_k if is_k else S.synth_v)(1280, 2, 4, 128).to(DEV)
    parts = [x[:512], x[512:640], x[640:1024], x[1024:]]
    want, got = _store_all(is_k, parts), _store_all(is_k, parts, (0, 1, 2))
    got.poll_stores()                                             # nobody waits: what has arrived is found
    torch.cuda.synchronize()
    for _ in parts:
        got.poll_stores()
    assert not got._unverified and got._enc_pending == 0
    assert got.ctx_len == want.ctx_len == 1280 and got.compressed_ctx_len == want.compressed_ctx_len
    for name in ("encoded_data", "block_infos", "thread_infos", "quant_min_ints", "quant_scales", "buffer"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name


def _busy(stream, seconds):
    """Keep a stream busy for about that long, with a kernel that counts clock ticks."""
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with torch.cuda.stream(stream):
        torch.cuda._sleep(1000)
        start.record()
        torch.cuda._sleep(5000000)
        end.record()
        end.synchronize()
        torch.cuda._sleep(int(5000000 * seconds * 1e3 / start.elapsed_time(end)))
        end.record()
    return end


def _ticks(stream, seconds):
    """What _sleep takes for about that long."""
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    with torch.cuda.stream(stream):
        torch.cuda._sleep(1000)
        start.record()
        torch.cuda._sleep(5000000)
        end.record()
        end.synchronize()
    return int(5000000 * seconds * 1e3 / start.elapsed_time(end))


@pytest.mark.gpu
def test_a_number_that_never_comes_is_waited_for_on_its_own_stream_alone():
    from tests import _synth as S
    _config()
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    x = S.synth_k(512, 1, 2, 64).to(DEV)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        ctx = _store_all(True, [x])
    outcome = ctx._outcome
    outcome.synchronize()
    words = [w & 0xffffffff for w in outcome.words.tolist()]
    assert outcome.query() and words[10] | words[11] << 32 == side.cuda_stream == outcome.stream and words[12] == torch.cuda.current_device()
    there = outcome.number
    end = _busy(other, 6.0)
    began = time.monotonic()
    outcome.number = there + 1                                    # as if a call had been told so
    outcome.synchronize()
    waited = time.monotonic() - began
    assert not outcome.query() and not end.query() and 1.9 < waited < 4.0
    outcome.number = there
    end.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("ask", ["poll", "sizes"])
@pytest.mark.parametrize("is_k", [True, False])
def test_a_store_without_words_of_its_own_is_waited_for_on_its_stream(is_k, ask):
    """The words are the first stream's, the last store is the second's, and still behind a long kernel there when the default
    stream, which is ordered behind nothing, asks for what has become of it."""
    from tests import _synth as S
    _config()
    x = (S.synth_k if is_k else S.synth_v)(1280, 2, 4, 128).to(DEV)
    parts = [x[:512], x[512:640], x[640:1024], x[1024:]]
    want = _store_all(is_k, parts)
    expect = {name: getattr(want, name).clone() for name in ("encoded_data", "block_infos", "thread_infos", "quant_min_ints", "quant_scales", "buffer")}
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    ticks, end = _ticks(first, 0.2), torch.cuda.Event()
    with torch.cuda.stream(first):
        got = _store_all(is_k, parts[:2])
        torch.cuda._sleep(ticks)
        got.store(parts[2], want_symbols=False)
        outcome = got._outcome
    second.wait_stream(first)
    with torch.cuda.stream(second):
        torch.cuda._sleep(ticks)
        end.record()
        got.store(parts[3], want_symbols=False)
        assert not outcome.query() and len(got._unverified) > got._probe[1]
    outcome.synchronize()
    if ask == "poll":
        got.poll_stores()
        assert len(got._unverified) == 1 and not end.query()
    assert got.encoded_data.numel() == expect["encoded_data"].numel() and end.query() and not got._unverified
    for name, value in expect.items():
        assert torch.equal(getattr(got, name), value), name


@pytest.mark.gpu
@pytest.mark.parametrize("is_k", [True, False])
def test_stores_on_a_stream_are_learnt_of_on_another(is_k):
    """Queued behind a long kernel on a stream of their own; asked for on the default stream, which is ordered behind nothing."""
    from tests import _synth as S
    _config()
    x = (S.synth_k if is_k else S.synth_v)(1280, 2, 4, 128).to(DEV)
    parts = [x[:512], x[512:640], x[640:1024], x[1024:]]
    want = _store_all(is_k, parts)
    expect = {name: getattr(want, name).clone() for name in ("encoded_data", "block_infos", "thread_infos", "quant_min_ints", "quant_scales", "buffer")}
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        got = _store_all(is_k, parts[:2])
        _busy(first, 0.2)
        got.store(parts[2], want_symbols=False)
        outcome = got._outcome
        assert not outcome.query() and got._probe[0] is outcome and got._probe[2] == first.cuda_stream
    second.wait_stream(first)
    with torch.cuda.stream(second):                               # the words are another stream's: this store has none to write to
        got.store(parts[3], want_symbols=False)
        assert got._outcome is outcome and got._probe[1] == len(got._unverified) - 1
    with pytest.MonkeyPatch.context() as m:
        m.setattr(kvcomp_cuda, "encode_result", None)             # what the words say is enough for the first three
        outcome.synchronize()
        got.poll_stores()
    assert len(got._unverified) == 1
    second.synchronize()
    assert got.ctx_len == 1280
    for name, value in expect.items():
        assert torch.equal(getattr(got, name), value), name
    assert not got._unverified


@pytest.mark.gpu
@pytest.mark.parametrize("is_k", [True, False])
def test_a_first_store_that_is_learnt_of_has_its_codebook_in_place(monkeypatch, is_k):
    """What a first store's outcome says on one stream goes for the codebook and the decode tables on any other."""
    from tests import _synth as S
    _config()
    x = (S.synth_k if is_k else S.synth_v)(640, 2, 4, 128).to(DEV)
    room = kvcomp_cuda.codebook_room
    monkeypatch.setattr(kvcomp_cuda, "codebook_room", lambda device: room(device).fill_(0xee))     # (not what an earlier one has left there)
    want = _store_all(is_k, [x])
    names = ("encode_codebook", "decode_codebook", "_lut", "encoded_data", "block_infos", "thread_infos")
    expect = {name: getattr(want, name).clone() for name in names}
    restored = want.get_only_compressed()[0]
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    for i in range(10):
        with torch.cuda.stream(first):
            got = _store_all(is_k, [x])
        with torch.cuda.stream(second):                               # ordered behind nothing
            if got._unverified:
                got._outcome.synchronize()
            copies = [getattr(got, name).clone() for name in names]
            again = got.get_only_compressed()[0]
        second.synchronize()
        for name, value in zip(names, copies):
            assert torch.equal(value, expect[name]), (name, i)
        assert torch.equal(again, restored), i
        torch.cuda.synchronize()


class _FromAnotherStream:
    """Stands for a tensor in device memory that came from another stream; notes the streams it is kept for."""
    is_cuda = True

    def __init__(self, data):
        self._data, self.kept_for = data, []

    def __getattr__(self, name):
        return getattr(self._data, name)

    def __getitem__(self, at):
        return self._data[at]

    def record_stream(self, stream):
        self.kept_for.append(stream)


@pytest.mark.parametrize("grow", [lambda g: g.reserve(400, (), torch.uint8, None, 32), lambda g: g.append(torch.zeros(400, dtype=torch.uint8)), lambda g: g.trim()])
def test_a_buffer_that_is_replaced_is_kept_for_the_stream_that_uses_it(monkeypatch, grow):
    """Queued encodes may still write to it, and the copy into the new one reads it."""
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: "the current stream")
    g = _Growable()
    g.append(torch.arange(200, dtype=torch.uint8))
    g.used = 8
    old = g.data = _FromAnotherStream(g.data)
    grow(g)
    assert g.data is not old and old.kept_for == ["the current stream"] and torch.equal(g.data[:8], torch.arange(8, dtype=torch.uint8))


def test_other_memory_that_is_replaced_is_kept_for_the_stream_that_uses_it(monkeypatch):
    from kvcomp_amd.cache import _DenseHistory
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: "the current stream")
    h = _DenseHistory()
    h.append(torch.ones(1, 2, 200, 8, dtype=torch.float16))
    old = h.data = _FromAnotherStream(h.data)
    h.append(torch.ones(1, 2, 1000, 8, dtype=torch.float16))
    assert old.kept_for == ["the current stream"] and bool((h.view() == 1).all())
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.store(torch.ones(20, 1, 2, 64, dtype=torch.float16))
    old = ctx._tail = _FromAnotherStream(ctx._tail)
    ctx._tail_append(torch.ones(200, 1, 2, 64, dtype=torch.float16))
    assert old.kept_for == ["the current stream"] and bool((ctx.buffer == 1).all())


@pytest.mark.gpu
@pytest.mark.parametrize("is_k", [True, False])
def test_a_context_of_one_stream_grows_on_another_with_stores_outstanding(is_k):
    """The payload buffer comes from the default stream; queued encodes write to it on a busy side stream while it is
    replaced.  Nothing that the default stream allocates then may lie where they write."""
    from tests import _synth as S
    _config()
    x = (S.synth_k if is_k else S.synth_v)(1280, 2, 4, 128).to(DEV)
    parts = [x[:512], x[512:640], x[640:768], x[768:896], x[896:1152], x[1152:]]
    want = _store_all(is_k, parts)
    expect = {name: getattr(want, name).clone() for name in ("encoded_data", "block_infos", "thread_infos", "quant_min_ints", "quant_scales", "buffer")}
    got = _store_all(is_k, parts[:1])                             # on the default stream
    got.encoded_data
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.default_stream())
    growing, addresses, sizes = got._encoded, [got._encoded.data.data_ptr()], [got._encoded.data.numel()]
    with torch.cuda.stream(side):
        end = _busy(side, 1.0)
        for part in parts[1:]:
            got.store(part, want_symbols=False)
            if growing.data.data_ptr() != addresses[-1]:
                addresses.append(growing.data.data_ptr())
                sizes.append(growing.data.numel())
        assert len(addresses) > 2 and not end.query() and len(got._unverified) > 2 and got.waits == 2     # (the codebook, encoded_data)
    other = [torch.full((n,), 0xA5, dtype=torch.uint8, device=DEV) for n in sizes]
    assert not {t.data_ptr() for t in other} & set(addresses)
    side.synchronize()
    assert all(bool((t == 0xA5).all()) for t in other)
    for name, value in expect.items():
        assert torch.equal(getattr(got, name), value), name


@pytest.mark.gpu
def test_words_that_another_stream_will_write_to_are_not_used_again():
    """A store on a second stream while nobody follows the first one's outcome any more (as behind stores that were taken back)."""
    from tests import _synth as S
    _config()
    x = S.synth_k(1024, 2, 4, 128).to(DEV)
    want = _store_all(True, [x[:512], x[512:640], x[640:]]).encoded_data.clone()
    torch.cuda.synchronize()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(first):
        ctx = _store_all(True, [x[:512]])
        _busy(first, 0.2)
        ctx.store(x[512:640], want_symbols=False)
    words, ctx._probe = ctx._outcome, None
    assert not words.query()
    second.wait_stream(first)
    with torch.cuda.stream(second):
        ctx.store(x[640:], want_symbols=False)
    assert ctx._outcome is not words and ctx._probe[0] is ctx._outcome and ctx._probe[1] == len(ctx._unverified) == 2
    words.synchronize()
    ctx._outcome.synchronize()
    ctx.poll_stores()
    assert words.query() and not ctx._unverified and torch.equal(ctx.encoded_data, want)
