"""The last workgroup of a quantizer hands the symbol counts to the host: whole counts, whichever workgroup is last, of one workgroup and
of more than a launch has, of symbols on both sides of the counters held in LDS, and call after call from streams that take turns."""
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _counted(x, mask, eb, packed):
    groups = m._lib.lib().kvc_quant_groups(*x.shape, mask)
    mins, scales = torch.empty(groups, dtype=torch.int8, device=DEV), torch.empty(groups, dtype=torch.float16, device=DEV)
    sym, book = (m.quant_codebook_packed if packed else m.quant_codebook)(x, mask, eb, mins, scales, 0, lambda s: None)
    return sym, book


def _check(sym, book):
    counts = torch.bincount(sym.flatten().long(), minlength=256).cpu()
    fmt = book.tree_format
    _, enc, _ = m.build_codebook_from_counts(counts, fmt)
    assert bytes(book.encode_table)[:book.encode_bytes] == enc.numpy().tobytes()
    lengths = enc.view(torch.int32).view(-1, 2)[:, 1].long()
    assert book.payload_bits == int((counts[:lengths.numel()] * lengths).sum())


# (NB, BS, B, H, D): one workgroup; a few; more than the 1536 that a counting launch has at most
@pytest.mark.parametrize("eb", [0.2, 0.012])
@pytest.mark.parametrize("mask,shape", [("MASK_CHANNEL", (1, 64, 1, 1, 64)), ("MASK_CHANNEL", (5, 64, 1, 3, 96)), ("MASK_CHANNEL", (200, 64, 2, 32, 128)),
                                        ("MASK_K_BLOCK", (1, 64, 1, 1, 64)), ("MASK_K_BLOCK", (130, 64, 1, 4, 128)),
                                        ("MASK_V_TOKEN", (1, 128, 1, 4, 128)), ("MASK_V_TOKEN", (60, 128, 1, 8, 128)), ("MASK_V_TOKEN", (14, 128, 4, 32, 128)),
                                        ("MASK_V_TOKEN", (1, 128, 9, 32, 128)), ("MASK_V_TOKEN", (1, 128, 1, 2, 20))])
def test_counts_are_whole_call_after_call(mask, shape, eb):
    mask, g = getattr(m, mask), torch.Generator(device=DEV).manual_seed(3)
    streams, held = [torch.cuda.Stream(), torch.cuda.Stream()], []
    xs = [torch.randn(*shape, generator=g, device=DEV).to(torch.float16) * (i + 1) for i in range(2)]
    torch.cuda.synchronize()
    for i in range(6):
        with torch.cuda.stream(streams[i % 2]):
            held.append(_counted(xs[i % 2], mask, eb, False))
    torch.cuda.synchronize()
    for sym, book in held:
        _check(sym, book)
    if eb == 0.2 and m.packed_symbols_supported(mask != m.MASK_V_TOKEN, mask, xs[0], eb):
        _, book = _counted(xs[0], mask, eb, True)
        assert book.payload_bits == held[0][1].payload_bits and bytes(book.encode_table) == bytes(held[0][1].encode_table)
