"""Tensors in host memory: what works on them in PyTorch keeps working, and none of their addresses reaches a kernel.  The
library is replaced by one that fails the test when it is called, so no GPU is needed (and none is given a host address)."""
import pytest
import torch

from kvcomp_amd import _lib, attention, compute, kvcomp_cuda
from kvcomp_amd.cache import KVCompCachePytorchQuant
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode


class _NoLibrary:
    def __getattr__(self, name):
        if name == "kvc_attention_workspace_bytes":             # host arithmetic
            return lambda *a: 1 << 16
        raise AssertionError("%s was called with a tensor in host memory" % name)


@pytest.fixture(autouse=True)
def no_kernels(monkeypatch):
    monkeypatch.setattr(_lib, "lib", lambda: _NoLibrary())
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


def _context(is_k, tokens=0):
    ctx = KVCompCtx(is_k, 1, 2, 64, 0.1)
    if tokens:
        ctx.store(torch.zeros(tokens, 1, 2, 64, dtype=torch.float16))
    return ctx


def test_guard_and_stream_refuse_host_tensors():
    t = torch.zeros(4)
    with pytest.raises(ValueError, match="cuda device"):
        _lib.device_guard(t)
    with pytest.raises(ValueError, match="cuda device"):
        _lib.stream_of(t)


def test_tokens_that_stay_in_a_host_tail_come_back():
    x = torch.arange(60 * 128, dtype=torch.float32).reshape(60, 1, 2, 64).to(torch.float16)
    ctx = _context(True)
    for part in (x[:40], x[40:41], x[41:]):
        ctx.store(part)
    assert torch.equal(ctx.buffer, x) and torch.equal(ctx.get()[0], x)


def test_queries_in_host_memory_are_refused():
    k, v, q = _context(True, 40), _context(False, 40), torch.zeros(1, 2, 64, dtype=torch.float16)
    with pytest.raises(ValueError, match="cuda device"):
        attention.CompressedAttention(k, v).attend(q)


def test_queries_on_another_device_than_the_cache_are_refused():
    k, v = _context(True, 40), _context(False, 40)
    with pytest.raises(_lib.KvcompError, match="queries on meta"):
        attention.CompressedAttention(k, v).attend(torch.zeros(1, 2, 64, dtype=torch.float16, device="meta"))


def test_products_of_host_operands_are_refused():
    k, v = _context(True), _context(False)
    for ctx in (k, v):
        ctx.device, ctx.compressed_ctx_len, ctx.tree_format = torch.device("cpu"), 128, 3
        groups = 128 // ctx.block_size * ctx._groups_per_block
        for g, n, dtype in ((ctx._min_ints, groups, torch.int8), (ctx._scales, groups, torch.float16), (ctx._encoded, 64, torch.uint8),
                            (ctx._block_infos, 64, torch.uint8), (ctx._thread_infos, 64, torch.uint8)):
            g.append(torch.zeros(n, dtype=dtype))
        ctx.decode_codebook = ctx._lut_source = torch.zeros(6, dtype=torch.uint8)
        ctx._lut = torch.zeros(16, dtype=torch.uint8)
    q, p = torch.zeros(1, 2, 64, dtype=torch.float16), torch.zeros(1, 2, 128, dtype=torch.float16)
    for call in (lambda: k.mat_vec_mul(q), lambda: v.mat_vec_mul(p), lambda: attention.k_scores(k, k._lut, q),
                 lambda: attention.v_partials(v, v._lut, p)):
        with pytest.raises((ValueError, _lib.KvcompError), match="device"):
            call()
    with pytest.raises(_lib.KvcompError, match="device"):
        compute.dequant(torch.zeros(1, 64, 1, 2, 64, dtype=torch.uint8), k.quant_min_ints, k.quant_scales, k.quant_dims)


def test_blocks_in_host_memory_are_refused_by_the_simulated_quantizer():
    with pytest.raises(_lib.KvcompError, match="device float16"):
        compute.quant_in_place(torch.zeros(1, 2, 64, 64, dtype=torch.float16), 64, 0.1, QuantMode.ChannelQuant)


@pytest.mark.parametrize("which", ["k", "cos", "sin"])
def test_rows_and_angles_elsewhere_than_the_caches_are_left_to_pytorch(which):
    class Elsewhere(torch.Tensor):                               # claims to lie on a GPU
        is_cuda = property(lambda self: True)
        device = property(lambda self: torch.device("cuda", self.get_device()))

        def get_device(self):
            return 1 if which in self.at else 0

    def at(name, *shape):
        t = torch.zeros(*shape, dtype=torch.float16).as_subclass(Elsewhere)
        t.at = name
        return t
    k, v = at("k", 1, 2, 3, 64), at("v", 1, 2, 3, 64)
    cos, sin = at("cos", 1, 3, 64), at("sin", 1, 3, 64)
    assert not compute.append_dense(k, v, cos, sin, at("cache", 1, 2, 8, 64), at("cache", 1, 2, 8, 64), 0)


def test_the_dense_cache_works_on_host_tensors_until_a_block_is_quantized():
    cache = KVCompCachePytorchQuant(1, 2, 64, 1)
    x = torch.arange(2 * 20 * 64, dtype=torch.float32).reshape(1, 2, 20, 64).to(torch.float16)
    one, zero = torch.ones(1, 20, 64, dtype=torch.float16), torch.zeros(1, 20, 64, dtype=torch.float16)
    k, v = cache.update(x, x, 0, {"cos": one, "sin": zero})
    assert torch.equal(k, x) and torch.equal(v, x)


def test_angles_in_fp32_keep_the_keys_in_fp32():
    cache = KVCompCachePytorchQuant(1, 2, 64, 1)
    k = torch.randn(1, 2, 3, 64, generator=torch.Generator().manual_seed(1)).to(torch.float16)
    cos, sin = (torch.rand(1, 3, 64, generator=torch.Generator().manual_seed(s)) for s in (2, 3))
    keys, values = cache.update(k, k, 0, {"cos": cos, "sin": sin})
    assert keys.dtype is torch.float32 and torch.equal(keys, compute.apply_rotary_pos_emb_single(k, cos, sin)) and values.dtype is torch.float16
