"""One-token appends through the native module do what the Python code beside them does, over the forms that either may meet."""
import threading
import time

import pytest
import torch

from kvcomp_amd import _lib
from kvcomp_amd.compute import append_dense
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _NotTaken:
    append_dense = append_rows = staticmethod(lambda *args: 0)


class _Own(torch.Tensor):
    pass


def _note_answers(monkeypatch):
    """What the native functions answer from now on."""
    module, answers = _lib.host(), []

    def noting(function):
        def call(*args):
            answers.append(function(*args))
            return answers[-1]
        return call
    noted = type("Noted", (), {name: staticmethod(noting(getattr(module, name))) for name in ("append_dense", "append_rows")})
    monkeypatch.setattr(_lib, "host", lambda: noted)
    return answers


def _randn(*shape, dtype=torch.float16):
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


B, H, T, D = 2, 3, 5, 16
FORMS = {
    "plain": lambda k, v, c, s: (k, v, c, s),
    "angles of every sequence": lambda k, v, c, s: (k, v, c.repeat(B, 1, 1), s.repeat(B, 1, 1)),
    "no angles": lambda k, v, c, s: (k, v, None, None),
    "tokens first": lambda k, v, c, s: (k.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3), v, c, s),
    "slices": lambda k, v, c, s: (torch.cat([k, k], 2)[:, :, 1:1 + T], v, torch.cat([c, c], 1)[:, 2:2 + T], s),
    "elements apart": lambda k, v, c, s: (torch.cat([k, k], 3)[..., ::2], v, c, s),
    "angles apart": lambda k, v, c, s: (k, v, torch.cat([c, c], 2)[..., ::2], s),
    "other type": lambda k, v, c, s: (k.float(), v, c, s),
    "other angles": lambda k, v, c, s: (k, v, c.float(), s.float()),
    "fewer angles": lambda k, v, c, s: (k, v, c[:, :T - 1], s[:, :T - 1]),
    "values of another shape": lambda k, v, c, s: (k, v[:, :, :T - 1], c, s),
    "a gradient": lambda k, v, c, s: (k.clone().requires_grad_(), v, c, s),
    "a gradient of the angles": lambda k, v, c, s: (k, v, c.clone().requires_grad_(), s),
    "a class of its own": lambda k, v, c, s: (k.as_subclass(_Own), v, c, s),
    "a parameter": lambda k, v, c, s: (torch.nn.Parameter(k, requires_grad=False), v, c, s),
    "host memory": lambda k, v, c, s: (k.cpu(), v.cpu(), c.cpu(), s.cpu()),
    "no tokens": lambda k, v, c, s: (k[:, :, :0], v[:, :, :0], c[:, :0], s[:, :0]),
    "rows of 15": lambda k, v, c, s: (k[..., :15], v[..., :15], c[..., :15], s[..., :15]),
}
TAKEN = {"plain", "angles of every sequence", "no angles", "tokens first", "slices", "a parameter", "no tokens"}      # by the native function


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("grad", [True, False])
def test_append_dense(monkeypatch, form, grad):
    args = FORMS[form](_randn(B, H, T, D), _randn(B, H, T, D) + 1, _randn(1, T, D), _randn(1, T, D))
    wide = args[0].shape[3]
    caches = [torch.zeros(B, H, 12, wide, dtype=torch.float16, device=DEV) for _ in range(4)]
    answers = _note_answers(monkeypatch)
    with torch.set_grad_enabled(grad):
        native = append_dense(*args, *caches[:2], 4)
        monkeypatch.setattr(_lib, "host", lambda: _NotTaken)
        assert append_dense(*args, *caches[2:], 4) is native
    taken = form in TAKEN or (not grad and form.startswith("a gradient"))
    assert answers == ([] if form == "host memory" else [int(taken)]) and native >= taken
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3]) and (not native or bool(args[0].numel()) == bool(caches[0].any()))


def test_append_dense_to_other_caches(monkeypatch):
    args = (_randn(B, H, T, D), _randn(B, H, T, D), None, None)
    room = torch.zeros(B, H, 12, D, dtype=torch.float16, device=DEV)
    noted = _note_answers(monkeypatch)
    for caches in ((room, room[:, :, :10]), (room[:1], room[:1]), (room.permute(0, 2, 1, 3), room), (room.float(), room), (room, room.cpu())):
        answers = [append_dense(*args, *caches, 4)]
        with monkeypatch.context() as m:
            m.setattr(_lib, "host", lambda: _NotTaken)
            answers.append(append_dense(*args, *caches, 4))
        assert answers == [False, False] and noted.pop() == 0 and not noted
    with pytest.raises(_lib.KvcompError):
        append_dense(*args, room, room.clone(), 8)                 # five tokens behind eight of twelve
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert append_dense(*args, room, room.clone(), 4)
    side.synchronize()
    assert len(noted) == 2 and noted[0] < 0 and noted[1] == 1
    assert torch.equal(room[:, :, 4:4 + T], args[0])


@pytest.mark.parametrize("D,form", [(D, f) for D in (64, 8) for f in ("plain", "permuted", "offset", "gradient", "own")])
def test_rows_behind_a_tail(monkeypatch, D, form):
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode("ChannelQuant"), QuantMode("TokenQuant"), 64, 128, 64, 128, 0.1, 0.2)
    heads = 2
    rows = {"plain": lambda x: x, "permuted": lambda x: x.permute(2, 1, 0, 3).contiguous().permute(2, 1, 0, 3),
            "offset": lambda x: torch.empty(x.numel() + 3, dtype=x.dtype, device=DEV)[3:].view(x.shape).copy_(x),
            "gradient": lambda x: x.clone().requires_grad_(), "own": lambda x: x.as_subclass(_Own)}[form]
    held, counts = [], (1, 3, 1, 2)
    for native in (True, False):
        with monkeypatch.context() as m:
            answers = _note_answers(m)
            if not native:
                m.setattr(_lib, "host", lambda: _NotTaken)
            ctx = KVCompCtx(True, 1, heads, D, 0.1)
            with torch.no_grad():
                for n in counts:
                    ctx.store(rows(_randn(n, 1, heads, D)))
            held.append((ctx.buffer, ctx.ctx_len, ctx._tail._version))
            taken = {"plain": [1] * 4, "permuted": [int(n == 1) for n in counts]}.get(form, [0] * 4)     # (one token is in order either way)
            assert answers == (taken if native else [])
    assert torch.equal(held[0][0], held[1][0]) and held[0][1:2] == held[1][1:2] and held[0][0].shape[0] == 7
    assert held[0][2] == held[1][2]


def _sleep_for(seconds):
    """Keep the current stream busy for about that long, with a kernel that counts clock ticks."""
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000000)
    start.record()
    torch.cuda._sleep(10000000)
    end.record()
    end.synchronize()
    torch.cuda._sleep(int(10000000 * seconds * 1e3 / start.elapsed_time(end)))


@pytest.mark.parametrize("which", ["append_rows", "append_dense"])
def test_other_threads_run_on_while_an_append_waits_for_its_queue(which):
    """Appends behind a kernel of half a second fill their queue (2700 of them do); the launch that waits for room then does so
    without the interpreter's lock."""
    tail, rows = torch.zeros(64, 1, 1, 64, dtype=torch.float16, device=DEV), _randn(1, 1, 1, 64)
    call = {"append_rows": lambda: _lib.host().append_rows(tail, 0, rows, 128),
            "append_dense": lambda: _lib.host().append_dense(rows, rows, None, None, tail.view(1, 1, 64, 64), tail.view(1, 1, 64, 64), 0)}[which]
    assert call() == 1
    gaps, stop = [], threading.Event()

    def other():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.0005)
            gaps.append(time.perf_counter() - last)
            last += gaps[-1]

    thread = threading.Thread(target=other)
    _sleep_for(0.5)
    begun, longest = time.perf_counter(), 0.0
    thread.start()
    while time.perf_counter() - begun < 0.4:
        before = time.perf_counter()
        call()
        longest = max(longest, time.perf_counter() - before)
    stop.set()
    thread.join()
    torch.cuda.synchronize()
    assert longest > 0.1, "no append has waited"
    assert max(gaps) < longest / 2
