"""An encode in two halves (kvc_encode_prepare, kvc_encode_queue) writes what kvc_encode_async writes, whichever way of encoding
the option asks for when each half is queued, and leaves its outcome in pinned words."""
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd import _lib
from kvcomp_amd.ctx import _Growable, _Outcome

DEV = "cuda:0"


def test_a_growing_buffer_takes_rows_along_that_may_be_filled():
    g = _Growable()
    g.reserve(40, (), torch.uint8, torch.device("cpu"))
    g.data[:40] = torch.arange(40, dtype=torch.uint8)
    g.used = 8
    g.reserve(100, (), torch.uint8, None, 32)
    assert g.data.numel() >= 8 + 32 + 100 and torch.equal(g.data[:40], torch.arange(40, dtype=torch.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("first,second", [(1, 1), (1, 0), (0, 1), (0, 0), (2, 3)])
@pytest.mark.parametrize("is_k,T,B,H,D", [(True, 64, 1, 1, 8), (True, 192, 1, 3, 72), (False, 128, 1, 1, 64), (False, 1024, 2, 32, 128),
                                          (True, 4096, 4, 32, 32)])
def test_prepared_encodes_write_the_same(is_k, T, B, H, D, first, second):
    g = torch.Generator().manual_seed(T)
    sym = torch.randint(0, 11, (T, B, H, D), generator=g, dtype=torch.uint8).to(DEV)
    _, enc, _ = m.build_codebook_from_counts(m.symbol_counts([sym]), m.TREE_I8)
    enc = enc.to(DEV)
    sizes = m.buffer_sizes(T, B * H * D, is_k, H, D)

    def buffers():
        return (torch.full((sizes[0],), 7, dtype=torch.uint8, device=DEV), torch.zeros(sizes[1], dtype=torch.uint8, device=DEV),
                torch.zeros(sym.numel(), dtype=torch.uint8, device=DEV), torch.full((16,), 9, dtype=torch.int32, device=DEV))
    geometry = dict(batch=B, head_num=H, head_dim=D, tokens=T)
    bi, ti, payload, state = buffers()
    state[:9] = 0
    m.encode_async(is_k, symbols=sym, encode_tables=enc, table_bytes=enc.numel(), block_infos=bi, thread_infos=ti, encoded=payload,
                   stream_bytes=state[8:9], result=state[:8], **geometry)
    bi2, ti2, payload2, state2 = buffers()
    outcome, option = _Outcome(), _lib.set_option("encode_one_pass", first)
    try:
        prepared = m.encode_prepare(is_k, symbols=sym, block_infos=bi2, thread_infos=ti2, state=state2, **geometry)
        _lib.set_option("encode_one_pass", second)
        m.encode_prepared(prepared, enc, payload2, outcome.ask(_lib.stream_of(sym)))
    finally:
        _lib.set_option("encode_one_pass", option)
    outcome.synchronize()
    assert outcome.query()
    assert torch.equal(bi, bi2) and torch.equal(ti, ti2) and torch.equal(payload, payload2)
    for at in (0, 1, 2, 3, 4, 5, 8):                              # (word 6 counts looks)
        assert int(state[at]) == int(state2[at]) == int(outcome.words[at])


@pytest.mark.gpu
def test_words_that_a_kernel_may_still_write_to_outlive_their_context():
    late = _Outcome()
    late.ask(0)                                                   # as if its encode had been queued
    number, seen = late.number, late._seen
    del late
    assert any(n == number for _, n in _Outcome._late)
    _Outcome()
    assert any(n == number for _, n in _Outcome._late)
    seen[9] = number                                              # the encode's last store
    _Outcome()
    assert not any(n == number for _, n in _Outcome._late)
