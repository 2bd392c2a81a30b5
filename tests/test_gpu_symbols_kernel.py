"""The one-pass encoder from symbols whose codes are known to be short writes what the general one writes: every vector length it
takes, alphabets on both sides of the pair table, runs of one, two and four tiles, tiles whose images do not fit beside each
other, symbols without a code, buffers that are too small, and the path of a wave that gives up."""
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _symbols(T, B, H, D, alphabet, rare_tiles, is_k, seed=1):
    """Geometric symbols; in `rare_tiles` of the tiles uniform ones (long codes, large tiles)."""
    g = torch.Generator().manual_seed(seed)
    shape = (T, B * H * D)
    few = torch.empty(shape).geometric_(0.6, generator=g).sub_(1).clamp_(max=alphabet - 1)
    if rare_tiles:
        rows, cols = (64, D) if is_k else (128, 64)
        rare = torch.rand(T // rows, B * H * D // cols, generator=g) < rare_tiles
        rare = rare.repeat_interleave(rows, 0).repeat_interleave(cols, 1)
        few = torch.where(rare, torch.randint(0, alphabet, shape, generator=g).float(), few)
    return few.to(torch.uint8).reshape(T, B, H, D).to(DEV)


def _table(alphabet, longest):
    """Codes of 1, 2, 3 ... bits, the rest of equal length `longest`; a prefix code."""
    lengths = []
    left = 1 << longest
    for s in range(alphabet):
        rest = alphabet - s - 1
        l = 1
        while l < longest and left - (1 << (longest - l)) < rest:
            l += 1
        lengths.append(l)
        left -= 1 << (longest - l)
    assert left >= 0
    code, entries = 0, []
    for i, l in enumerate(lengths):
        code = code << (l - lengths[i - 1]) if i else 0
        entries += [code, l]
        code += 1
    return torch.tensor(entries, dtype=torch.int32).view(torch.uint8).to(DEV), max(lengths)


def _encode(is_k, sym, table, cap, longest, base=0):
    T, B, H, D = sym.shape
    sizes = m.buffer_sizes(T, B * H * D, is_k, H, D)
    bi, ti = torch.zeros(sizes[0], dtype=torch.uint8, device=DEV), torch.zeros(sizes[1], dtype=torch.uint8, device=DEV)
    out, state = torch.zeros(cap + base, dtype=torch.uint8, device=DEV)[base:], torch.zeros(16, dtype=torch.int32, device=DEV)
    p = m.encode_prepare(is_k, batch=B, head_num=H, head_dim=D, tokens=T, symbols=sym, block_infos=bi, thread_infos=ti, state=state)
    m.encode_prepared(p, table, out, None, longest)
    torch.cuda.synchronize()
    return bi, ti, out, state


CASES = [(True, 64, 1, 1, 128, 13, 7), (True, 128, 1, 5, 96, 16, 8), (True, 192, 1, 3, 64, 17, 8), (False, 128, 1, 1, 64, 2, 1),
         (False, 384, 1, 3, 128, 23, 8), (True, 64 * 33, 8, 32, 64, 13, 7), (True, 64 * 43, 6, 32, 96, 11, 6), (True, 64 * 33, 8, 32, 128, 16, 8),
         (False, 128 * 17, 4, 32, 256 // 2, 8, 7), (False, 128 * 65, 8, 32, 64, 7, 6), (False, 128 * 33, 8, 32, 128, 8, 5), (False, 128 * 33, 8, 32, 128, 20, 8),
         (False, 128 * 129, 1, 65, 64, 7, 5), (False, 128 * 253, 1, 65, 64, 7, 5),
         (True, 64 * 127, 1, 65, 64, 7, 5), (True, 64 * 127, 1, 65, 96, 9, 6), (True, 64 * 129, 1, 66, 96, 9, 6),
         (True, 64, 1, 1, 72, 13, 7), (True, 192, 1, 3, 72, 17, 8), (True, 64 * 43, 6, 32, 72, 11, 6), (True, 64 * 129, 1, 66, 72, 23, 8)]   # last tiles without all their neighbours


@pytest.mark.parametrize("rare_tiles", [0.0, 0.15])
@pytest.mark.parametrize("is_k,T,B,H,D,alphabet,longest", CASES)
def test_writes_what_the_general_kernel_writes(is_k, T, B, H, D, alphabet, longest, rare_tiles):
    sym = _symbols(T, B, H, D, alphabet, rare_tiles, is_k)
    table, longest = _table(alphabet, longest)
    counts = torch.bincount(sym.flatten().long(), minlength=alphabet)[:alphabet].cpu()
    bits = int((counts * table.cpu().view(torch.int32)[1::2]).sum())
    cap = bits // 8 + sym.numel() // (D if is_k else 128) + 1
    for base in (0, 3):
        want = _encode(is_k, sym, table, cap, 0, base)
        got = _encode(is_k, sym, table, cap, longest, base)
        assert int(want[3][1]) == int(got[3][1]) == 0 and torch.equal(want[3][:6], got[3][:6]) and int(want[3][8]) == int(got[3][8])
        assert all(torch.equal(a, b) for a, b in zip(want[:3], got[:3]))


@pytest.mark.parametrize("is_k,T,B,H,D,alphabet,longest", [CASES[0], CASES[5], CASES[6], CASES[9]])
def test_errors_and_a_wave_that_gives_up(is_k, T, B, H, D, alphabet, longest):
    sym = _symbols(T, B, H, D, alphabet, 0.1, is_k)
    table, longest = _table(alphabet, longest)
    good = _encode(is_k, sym, table, sym.numel(), longest)
    old = _lib.set_option("encode_lookback_polls", -1)
    try:
        again = _encode(is_k, sym, table, sym.numel(), longest)
    finally:
        _lib.set_option("encode_lookback_polls", old)
    assert all(torch.equal(a, b) for a, b in zip(good[:3], again[:3])) and int(again[3][1]) == 0
    short = _encode(is_k, sym, table, int(good[3][0]) - 1, longest)
    assert int(short[3][1]) == 4 and int(short[3][8]) == 0
    assert torch.equal(short[2][:int(good[3][0]) - 8192 if int(good[3][0]) > 8192 else 0], good[2][:max(int(good[3][0]) - 8192, 0)])
    for symbol in (alphabet, 16, 255):
        bad = sym.clone()
        bad.view(-1)[bad.numel() // 2] = symbol
        assert int(_encode(is_k, bad, table, sym.numel(), longest)[3][1]) == 2
    unaligned = torch.empty(sym.numel() + 4, dtype=torch.uint8, device=DEV)[4:].view(sym.shape).copy_(sym)
    assert all(torch.equal(a, b) for a, b in zip(good[:3], _encode(is_k, unaligned, table, sym.numel(), longest)[:3]))
