"""First-store encoders whose runs of tiles are more than the waves that the chip holds: each workgroup draws several runs, and a run's
images wait until the next run's first tile is counted.  They write what the general one-pass kernel writes, byte for byte: with
two and more rounds of the waves, a last run that is not whole, tiles whose images do not fit beside each other, a buffer that is
one byte too small, and waves that give up waiting."""
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd import _lib

from .test_gpu_packed_symbols import _both, _data

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [1, 2, 3, 4, 5, 6, 7, 7]


def _symbols(T, B, H, D, is_k, rare_tiles):
    """Geometric symbols (two bits each); in some tiles uniform ones (4.4 bits)."""
    g = torch.Generator(device=DEV).manual_seed(T + D)
    u = torch.rand((T, B * H * D), generator=g, device=DEV)
    few = torch.floor(-torch.log2(u.clamp_(min=1e-6))).clamp_(max=7)
    rows, cols = (64, D) if is_k else (128, 64)
    rare = (torch.rand((T // rows, B * H * D // cols), generator=g, device=DEV) < rare_tiles).repeat_interleave(rows, 0).repeat_interleave(cols, 1)
    return torch.where(rare, torch.floor(u * 8), few).to(torch.uint8).reshape(T, B, H, D)


def _table():
    code, entries = 0, []
    for i, l in enumerate(LENGTHS):
        code = code << (l - LENGTHS[i - 1]) if i else 0
        entries += [code, l]
        code += 1
    return torch.tensor(entries, dtype=torch.int32).view(torch.uint8).to(DEV)


def _encode(is_k, sym, cap, longest):
    T, B, H, D = sym.shape
    sizes = m.buffer_sizes(T, B * H * D, is_k, H, D)
    bi, ti = torch.zeros(sizes[0], dtype=torch.uint8, device=DEV), torch.zeros(sizes[1], dtype=torch.uint8, device=DEV)
    out, state = torch.zeros(cap, dtype=torch.uint8, device=DEV), torch.zeros(16, dtype=torch.int32, device=DEV)
    p = m.encode_prepare(is_k, batch=B, head_num=H, head_dim=D, tokens=T, symbols=sym, block_infos=bi, thread_infos=ti, state=state)
    m.encode_prepared(p, _table(), out, None, longest)
    torch.cuda.synchronize()
    return bi, ti, out, state


def _room(is_k, sym):
    counts = torch.bincount(sym.flatten(), minlength=8)
    return int((counts * torch.tensor(LENGTHS, device=DEV)).sum()) // 8 + sym.numel() // (sym.shape[3] if is_k else 128) + 1


# tiles a little beyond one round of 4096 waves' runs, beyond two and beyond three
CASES = [(True, 64 * 129, 1, 64, 64), (True, 64 * 257, 1, 65, 64), (True, 64 * 131, 1, 67, 96), (True, 64 * 131, 1, 67, 72), (True, 64 * 385, 1, 65, 128),
         (False, 128 * 129, 1, 130, 64), (False, 128 * 253, 1, 199, 64), (False, 128 * 131, 1, 67, 128),
         # three whole rounds, and a rest that runs of three would fill, which do not divide a group
         (False, 128 * 300, 1, 197, 64)]


@pytest.mark.parametrize("rare_tiles", [0.0, 0.2])
@pytest.mark.parametrize("is_k,T,B,H,D", CASES)
def test_writes_what_the_general_kernel_writes(is_k, T, B, H, D, rare_tiles):
    sym = _symbols(T, B, H, D, is_k, rare_tiles)
    cap = _room(is_k, sym)
    want, got = _encode(is_k, sym, cap, 0), _encode(is_k, sym, cap, 7)
    assert int(want[3][1]) == int(got[3][1]) == 0 and torch.equal(want[3][:6], got[3][:6]) and int(want[3][8]) == int(got[3][8])
    assert all(torch.equal(a, b) for a, b in zip(want[:3], got[:3]))


@pytest.mark.parametrize("is_k,T,B,H,D", [CASES[1], CASES[6]])
def test_a_buffer_that_is_too_small_is_told(is_k, T, B, H, D):
    sym = _symbols(T, B, H, D, is_k, 0.0)
    used = int(_encode(is_k, sym, _room(is_k, sym), 7)[3][0])
    assert int(_encode(is_k, sym, used, 7)[3][1]) == 0
    want, got = _encode(is_k, sym, used - 1, 0), _encode(is_k, sym, used - 1, 7)
    assert int(got[3][1]) == int(want[3][1]) != 0


@pytest.mark.parametrize("polls", [-1, 0, 1])
@pytest.mark.parametrize("is_k,T,B,H,D", [CASES[1], CASES[6]])
def test_waves_that_give_up_waiting(is_k, T, B, H, D, polls):
    """Every wave ends, and the call is encoded again in two passes."""
    sym = _symbols(T, B, H, D, is_k, 0.0)
    cap = _room(is_k, sym)
    want = _encode(is_k, sym, cap, 0)
    default = _lib.set_option("encode_lookback_polls", polls)
    try:
        got = _encode(is_k, sym, cap, 7)
    finally:
        _lib.set_option("encode_lookback_polls", default)
    assert int(got[3][1]) == 0 and all(torch.equal(a, b) for a, b in zip(want[:3], got[:3]))


@pytest.mark.parametrize("polls", [None, ("encode_lookback_polls", -1)])
@pytest.mark.parametrize("is_k,mode,T,B,H,D,eb,wide", [(True, "ChannelQuant", 64 * 400, 1, 64, 64, 0.1, False), (True, "ChannelQuant", 64 * 131, 2, 64, 96, 0.1, True),
                                                       (True, "BlockQuant", 64 * 260, 1, 64, 128, 0.08, True), (False, "TokenQuant", 128 * 261, 1, 65, 128, 0.2, False),
                                                       (False, "TokenQuant", 128 * 131, 2, 67, 96, 0.1, True)])
def test_first_stores_of_several_rounds(is_k, mode, T, B, H, D, eb, wide, polls):
    _both(is_k, mode, _data(T, B, H, D, wide, 3), eb, polls=polls)


def test_the_budget_of_waiting_is_a_runs():
    """What is reported is the most that a wave has asked in vain for a run of its tiles, not for the five or six that it takes in this call:
    50 to 170 here, added up over the runs 180 to 330.  The least of a few calls, which other work on the machine does not raise."""
    sym = _symbols(128 * 650, 1, 129, 64, False, 0.0)
    cap = _room(False, sym)
    assert min(int(_encode(False, sym, cap, 7)[3][6]) for _ in range(8)) < 140
