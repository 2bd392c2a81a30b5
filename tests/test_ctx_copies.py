"""Contexts can be copied like any object that holds tensors: a copy has memory of its own, and nothing in it refers to the
original's."""
import copy
import pickle

import pytest
import torch

from kvcomp_amd.cache import KVCompCache
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode


def _config():
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode.TokenQuant, 64, 128, 64, 128, 0.1, 0.2)


# a context's arrays and the descriptor's fields for them, which are what the kernels get
ARRAYS = {"_encoded": "d_encoded", "_block_infos": "d_block_infos", "_thread_infos": "d_thread_infos", "_min_ints": "d_quant_min_ints",
          "_scales": "d_quant_scales_f16"}


def _filled():
    """A context with a block of 64 tokens, 128 groups."""
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    for name in ARRAYS:
        getattr(ctx, name).append(torch.arange(128, dtype=torch.uint8))
    ctx.decode_codebook = ctx._lut_source = torch.zeros(6, dtype=torch.uint8)
    ctx._lut = torch.zeros(4)
    ctx.compressed_ctx_len = ctx.ctx_len = 64
    return ctx


@pytest.mark.parametrize("how", [copy.deepcopy, lambda x: pickle.loads(pickle.dumps(x))])
def test_a_copy_refers_to_its_own_memory(how):
    ctx = _filled()
    got = how(ctx)
    for name, field in ARRAYS.items():
        mine, theirs = getattr(got, name), getattr(ctx, name)
        assert torch.equal(mine.view, theirs.view) and getattr(got.descriptor(), field) == mine.data.data_ptr() != getattr(ctx.descriptor(), field)
    assert got.descriptor().d_luts == got._lut.data_ptr() != ctx.descriptor().d_luts
    assert got._descriptor is not ctx._descriptor
    assert got._lut_source is got.decode_codebook            # the copy's tables still belong to its codebook


@pytest.mark.parametrize("how", [copy.deepcopy, lambda x: pickle.loads(pickle.dumps(x))])
def test_a_queued_store_is_waited_for(how, monkeypatch):
    """A context whose store has not been looked at yet holds an event and pinned words, which no copy can have."""
    from kvcomp_amd import kvcomp_cuda
    from kvcomp_amd.ctx import _QueuedStore

    class Event:                                              # like torch.cuda.Event: cannot be pickled
        def __reduce__(self):
            raise TypeError("cannot pickle 'Event' object")
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    for g in (ctx._encoded, ctx._block_infos, ctx._thread_infos, ctx._min_ints, ctx._scales):
        g.append(torch.arange(40, dtype=torch.uint8))
    ctx._state = torch.zeros(16, dtype=torch.int32)
    ctx._state[8] = 33
    ctx._verified = ctx._bookkeeping() + (0,)
    ctx._unverified = [_QueuedStore(64, None, ctx._bookkeeping(), 40, False, True, True)]
    ctx._enc_pending, ctx._encoded.used = 40, 0
    ctx._host_words, ctx._probe = torch.zeros(16, dtype=torch.int32), (Event(), 0, None)
    monkeypatch.setattr(kvcomp_cuda, "encode_result", lambda *a: (33, 20, 9, 1))
    got = how(ctx)
    for c in (got, ctx):
        assert c._encoded.used == 33 and c._enc_pending == 0 and not c._unverified and c.max_tile_bytes == 20
    assert got._probe is None and got._host_words is None


def test_every_call_has_a_descriptor_of_its_own():
    """Two threads may attend over one context: the library reads what a call was given without the GIL."""
    _config()
    ctx = KVCompCtx(True, 1, 2, 64, 0.1)
    ctx.store(torch.zeros(20, 1, 2, 64, dtype=torch.float16))
    first = ctx.descriptor()
    ctx.store(torch.zeros(5, 1, 2, 64, dtype=torch.float16))
    second = ctx.descriptor()
    assert (first.tail_tokens, second.tail_tokens) == (20, 25) and first.d_tail_f16 == second.d_tail_f16 == ctx._tail.data_ptr()


def test_moved_data_is_seen():
    ctx = _filled()
    for name, field in ARRAYS.items():
        before, array = getattr(ctx.descriptor(), field), getattr(ctx, name)
        array.data = array.data.clone()
        assert getattr(ctx.descriptor(), field) == array.data.data_ptr() != before


def test_dense_caches_can_be_copied():
    _config()
    copy.deepcopy(KVCompCache(1, 2, 64, 2))


@pytest.mark.gpu
def test_attention_over_a_copy_outlives_the_original():
    from kvcomp_amd.attention import CompressedAttention
    from tests import _synth as S
    _config()
    pair = KVCompCtx(True, 1, 4, 128, 0.1), KVCompCtx(False, 1, 4, 128, 0.2)
    for c, x in zip(pair, (S.synth_k(300, 1, 4, 128), S.synth_v(300, 1, 4, 128))):
        c.store(x.to("cuda:0"))
    q = S.synth_q(1, 4, 128).to("cuda:0")
    want = CompressedAttention(*pair).attend(q)
    twin = copy.deepcopy(pair)
    for c in pair:
        for g in (c._encoded, c._block_infos, c._thread_infos, c._min_ints, c._scales):
            g.data.zero_()
    assert torch.equal(CompressedAttention(*twin).attend(q), want)


@pytest.mark.gpu
@pytest.mark.parametrize("how", [copy.deepcopy, lambda x: pickle.loads(pickle.dumps(x))])
def test_contexts_as_the_model_caches_hold_them_can_be_copied_right_after_a_store(how):
    from kvcomp_amd.attention import CompressedAttention
    from tests import _synth as S
    _config()
    pair = KVCompCtx(True, 1, 4, 128, 0.1), KVCompCtx(False, 1, 4, 128, 0.2)
    for c, x in zip(pair, (S.synth_k(300, 1, 4, 128), S.synth_v(300, 1, 4, 128))):
        c.codebook_smoothing = c.async_store = True
        c.store(x.to("cuda:0"), want_symbols=False)
        assert c._probe is not None
    twin = how(pair)
    q = S.synth_q(1, 4, 128).to("cuda:0")
    want = CompressedAttention(*pair).attend(q)
    for c, x in zip(twin, (S.synth_k(1, 1, 4, 128, 5), S.synth_v(1, 1, 4, 128, 5))):
        assert torch.equal(c.encoded_data, pair[0 if c.is_k else 1].encoded_data)
        c.store(x.to("cuda:0"), want_symbols=False)               # the copy goes on by itself
    assert pair[0].ctx_len == 300 and twin[0].ctx_len == 301
    assert torch.equal(CompressedAttention(*pair).attend(q), want)


@pytest.mark.gpu
def test_two_threads_attend_over_one_pair_of_contexts():
    import threading
    from kvcomp_amd.attention import CompressedAttention
    from tests import _synth as S
    _config()
    pair = KVCompCtx(True, 2, 4, 128, 0.1), KVCompCtx(False, 2, 4, 128, 0.2)
    for c, x in zip(pair, (S.synth_k(900, 2, 4, 128), S.synth_v(900, 2, 4, 128))):
        c.store(x.to("cuda:0"))
    queries = [S.synth_q(2, 4 * rep, 128, seed).to("cuda:0") for seed, rep in ((1, 1), (2, 4))]
    want = [CompressedAttention(*pair).attend(q) for q in queries]
    torch.cuda.synchronize()
    wrong = []

    def run(q, w):
        att = CompressedAttention(*pair)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(60):
                if not torch.equal(att.attend(q), w):
                    wrong.append(q.shape)
    threads = [threading.Thread(target=run, args=a) for a in zip(queries, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
