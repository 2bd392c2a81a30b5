"""Where a kernel takes the place of PyTorch's copies: what PyTorch would have recorded (gradients, tangents, traces) still is,
by its own operations, and a write that it cannot see moves the tensor's version on."""
import pytest
import torch

from kvcomp_amd import _lib, compute, kvcomp_cuda
from kvcomp_amd.cache import KVCompCachePytorchQuant
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
from tests import _synth as S

DEV = "cuda:0"


class _OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)

    def get_device(self):
        return 0


@pytest.fixture
def calls(monkeypatch):
    """Names of the library's functions that are called (all succeed and do nothing), on tensors that claim to lie on a GPU."""
    made = []

    class Library:
        def __getattr__(self, name):
            return lambda *a: made.append(name) or 0
    monkeypatch.setattr(_lib, "lib", lambda: Library())
    monkeypatch.setattr(_lib, "device_guard", lambda t: _lib._HERE_GUARD)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    return made


def _tensor(*shape):
    return torch.zeros(*shape, dtype=torch.float16).as_subclass(_OnGpu)


@pytest.mark.parametrize("which", ["k", "v", "cos", "sin", "k_cache", "v_cache"])
def test_rows_that_require_gradients_are_left_to_pytorch(calls, which):
    t = {"k": _tensor(1, 2, 3, 64), "v": _tensor(1, 2, 3, 64), "cos": _tensor(1, 3, 64), "sin": _tensor(1, 3, 64),
         "k_cache": _tensor(1, 2, 8, 64), "v_cache": _tensor(1, 2, 8, 64)}
    t[which].requires_grad_()
    assert not compute.append_dense(*t.values(), 0) and not calls
    with torch.no_grad():
        assert compute.append_dense(*t.values(), 0) and calls == ["kvc_append_dense"]


def test_tangents_and_traces_are_left_to_pytorch():
    x = torch.zeros(3)
    assert not _lib.recorded(x, None)
    with torch.autograd.forward_ad.dual_level():
        assert _lib.recorded(x)
    seen = []
    torch.jit.trace(lambda t: (seen.append(_lib.recorded(t)), t + 1)[1], x, check_trace=False)
    assert seen == [True] and not _lib.recorded(x)


def test_writes_over_what_views_hold_move_the_version(calls):
    cache = _tensor(1, 2, 8, 64)
    at = cache._version
    compute.quant_in_place(cache[:, :, 2:4], 2, 0.1, QuantMode.ChannelQuant)
    assert calls == ["kvc_quant_in_place"] and cache._version > at


@pytest.mark.gpu
def test_a_tail_that_was_written_over_since_is_refused_by_backward():
    _quantized()
    x = S.synth_k(400, 1, 2, 64).to(DEV)
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.store(x[:70])                                              # 6 tokens stay behind the first block
    q = torch.ones(ctx.buffer.shape, dtype=torch.float16, device=DEV, requires_grad=True)
    loss = (ctx.buffer * q).float().sum()                          # saves the view
    tail = ctx._tail
    ctx.store(x[70:170])                                           # one more block leaves, and the tail starts again
    assert ctx._tail is tail and ctx.buffer.shape[0] == 42
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def _quantized():
    KVCompCacheConfigStatic.extract_cache = None
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


@pytest.mark.gpu
def test_gradients_reach_the_keys_and_values_of_an_update():
    KVCompCacheConfigStatic.extract_cache = None
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", None, None, None, None, None, None, None, None, enable_quant=False)
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn(1, 2, 6, 64, generator=g).to(torch.float16).to(DEV).requires_grad_() for _ in range(2))
    cos, sin = (torch.rand(1, 6, 64, generator=g).to(torch.float16).to(DEV).requires_grad_() for _ in range(2))
    cache = KVCompCachePytorchQuant(1, 2, 64, 1)
    keys, values = cache.update(k, v, 0, {"cos": cos, "sin": sin})
    wk, wv = (torch.randn(1, 2, 6, 64, generator=g).to(torch.float16).to(DEV) for _ in range(2))
    got = torch.autograd.grad((keys * wk).sum() + (values * wv).sum(), (k, v, cos, sin))
    rotated = compute.apply_rotary_pos_emb_single(k, cos, sin)
    want = torch.autograd.grad((rotated * wk).sum() + (v * wv).sum(), (k, v, cos, sin))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_a_view_that_was_quantized_since_is_refused_by_backward():
    _quantized()
    x = S.synth_k(200, 1, 2, 64).permute(1, 2, 0, 3).contiguous().to(DEV)
    one, zero = torch.ones(1, 200, 64, dtype=torch.float16, device=DEV), torch.zeros(1, 200, 64, dtype=torch.float16, device=DEV)
    cache = KVCompCachePytorchQuant(1, 2, 64, 1)
    keys, _ = cache.update(x[:, :, :60], x[:, :, :60], 0, {"cos": one[:, :60], "sin": zero[:, :60]})
    q = torch.ones(60, 64, dtype=torch.float16, device=DEV, requires_grad=True)
    loss = (keys * q).float().sum()                                # saves the view
    cache.update(x[:, :, 60:], x[:, :, 60:], 0, {"cos": one[:, 60:], "sin": zero[:, 60:]})     # in the room the first made
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


@pytest.mark.gpu
def test_gradients_reach_the_tokens_of_a_tail():
    _quantized()
    x = S.synth_k(240, 1, 2, 64).to(DEV)
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    with torch.no_grad():
        ctx.store(x[:200])
    new = x[200:230].clone().requires_grad_()
    ctx.store(new)
    dense, _ = ctx.get()
    w = torch.randn(dense.shape, generator=torch.Generator().manual_seed(1)).to(torch.float16).to(DEV)
    (dense * w).sum().backward()
    assert torch.equal(new.grad, w[200:]) and torch.equal(dense[200:], new)
    with torch.no_grad():
        assert torch.equal(ctx.get()[0], dense)
