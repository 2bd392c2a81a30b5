"""A context's decode tables are built where its codebook is put in place, so that nobody ordered behind the store can meet
tables that another stream has yet to build."""
import pytest
import torch

from kvcomp_amd import _lib, kvcomp_cuda
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
from tests import _synth as S


def _config():
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


@pytest.fixture
def built(monkeypatch):
    """Tables built so far, as (codebook, table)."""
    made = []

    def build(codebook, tree_format):
        made.append((codebook, torch.zeros(4)))
        return made[-1][1]
    monkeypatch.setattr(kvcomp_cuda, "build_lut", build)
    return made


def test_the_first_store_brings_the_tables(monkeypatch, built):
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.device = torch.device("cpu")
    book = _lib.Codebook(tree_format=3, max_code_bits=3)
    enc, dec, lut = (torch.zeros(24, dtype=torch.uint8) for _ in range(3))
    monkeypatch.setattr(kvcomp_cuda, "quant_codebook", lambda *a: (a[0].to(torch.uint8), book))
    monkeypatch.setattr(kvcomp_cuda, "put_codebook", lambda *a: (enc, dec, lut))
    monkeypatch.setattr(KVCompCtx, "_encode_direct", lambda self, T, **kw: None)
    ctx._first_chunk(torch.zeros(1, 64, 1, 2, 64, dtype=torch.float16))
    assert ctx.decode_lut() is lut and ctx.decode_codebook is dec and not built


def test_a_codebook_put_in_place_later_brings_them_too(monkeypatch, built):
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)

    class Codebook(torch.Tensor):
        is_cuda = property(lambda self: True)

        def to(self, device):
            return self
    ctx._set_codebook(torch.zeros(24, dtype=torch.uint8), torch.zeros(24, dtype=torch.uint8).as_subclass(Codebook))
    assert len(built) == 1 and built[0][0] is ctx.decode_codebook and ctx.decode_lut() is built[0][1] and len(built) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("symbols", [2, 23, 100, 250])             # 250: the tables do not fit one launch's arguments
def test_the_launch_that_brings_a_codebook_builds_its_tables(symbols):
    _config()
    book = _lib.Codebook()
    g = torch.Generator().manual_seed(symbols)
    x = torch.randint(0, symbols, (4, 64, 1, 2, 64), generator=g).to(torch.float16)
    x[:, 0], x[:, 1] = 0.0, float(symbols - 1)                      # the step of every block is (symbols - 1) * eb = 1
    x = x.to("cuda:0")
    mins, scales = torch.empty(4, dtype=torch.int8, device="cuda:0"), torch.empty(4, dtype=torch.float16, device="cuda:0")
    sym, book = kvcomp_cuda.quant_codebook(x, kvcomp_cuda.MASK_K_BLOCK, 1.0 / (symbols - 1), mins, scales, 0)
    enc, dec, lut = kvcomp_cuda.put_codebook(book, torch.device("cuda:0"))
    assert bytes(enc.cpu().tolist()) == bytes(book.encode_table)[:book.encode_bytes]
    assert bytes(dec.cpu().tolist()) == bytes(book.decode_tree)[:book.decode_bytes]
    want = kvcomp_cuda.build_lut(dec, book.tree_format)
    # (entries beyond 1 << index bits, and list places beyond their counts, are never written or read)
    words, ref = lut.view(torch.int32).cpu(), want.view(torch.int32).cpu()
    bits, fast = int(ref[0]), 8 + 512 + 1024
    assert torch.equal(words[:8], ref[:8]) and torch.equal(words[520:520 + (1 << bits)], ref[520:520 + (1 << bits)])
    assert torch.equal(words[fast:fast + (1 << bits)], ref[fast:fast + (1 << bits)])


def test_tables_of_an_assigned_codebook_are_waited_for_and_never_shared_out_of_a_recording(monkeypatch, built):
    _config()
    ctx, waits = KVCompCtx(True, 1, 2, 64, 0.1), []
    ctx.decode_codebook = torch.zeros(24, dtype=torch.uint8)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: type("S", (), {"synchronize": lambda self: waits.append(1)})())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert ctx.decode_lut() is built[0][1] and not waits
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert ctx.decode_lut() is built[1][1] and len(waits) == 1
    assert ctx.decode_lut() is built[1][1] and len(waits) == 1


def test_nothing_is_asked_of_an_event_while_a_stream_is_recorded(monkeypatch):
    _config()

    class Event:
        asked = 0

        def query(self):
            self.asked += 1
            return False
    ctx, event = KVCompCtx(True, 1, 2, 64, 0.1), Event()
    ctx._probe = event, 1, None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    ctx.poll_stores()
    ctx.descriptor()
    assert event.asked == 0
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ctx.poll_stores()
    assert event.asked == 1


def _stored(T=700):
    _config()
    pair = KVCompCtx(True, 1, 4, 128, 0.1), KVCompCtx(False, 1, 4, 128, 0.2)
    for c, x in zip(pair, (S.synth_k(T, 1, 4, 128), S.synth_v(T, 1, 4, 128))):
        c.codebook_smoothing = c.async_store = True
        c.store(x.to("cuda:0"), want_symbols=False)
    return pair


@pytest.mark.gpu
def test_readers_on_other_streams_behind_the_store():
    from kvcomp_amd.attention import CompressedAttention
    k, v = _stored()
    q = S.synth_q(1, 4, 128).to("cuda:0")
    stored, sides = torch.cuda.Event(), [torch.cuda.Stream() for _ in range(2)]
    stored.record()
    got = []
    for side in sides:                      # two streams that wait for the stores and not for each other
        side.wait_event(stored)
        with torch.cuda.stream(side):
            got.append((CompressedAttention(k, v).attend(q), k.mat_vec_mul(q)[0], v.get()[0]))
    torch.cuda.synchronize()
    want = CompressedAttention(k, v).attend(q), k.mat_vec_mul(q)[0], v.get()[0]
    for g in got:
        assert all(torch.equal(a, b) for a, b in zip(g, want))


@pytest.mark.gpu
def test_eager_calls_before_the_replay_of_a_first_call_that_was_recorded():
    from kvcomp_amd.attention import CompressedAttention
    k, v = _stored()
    q = S.synth_q(1, 4, 128).to("cuda:0")
    att, out = CompressedAttention(k, v), torch.empty(1, 4, 128, device="cuda:0")
    assert k._probe is not None and v._probe is not None      # nobody has looked at the stores yet, and the recording must not
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        att.attend(q, out=out)
    want = CompressedAttention(k, v).attend(q)      # nothing has been replayed yet
    assert torch.isfinite(want).all()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(CompressedAttention(k, v).attend(q), want)
