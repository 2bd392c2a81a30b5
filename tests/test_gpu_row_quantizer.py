"""Per-token rows at the edges of how many waves share a row: quantizer with and without counts, against the
oracle."""
import numpy as np
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd.compute import quant
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("R", [512, 4096, 4104, 8192, 8200, 16384, 16392, 32768, 32776, 65536])
def test_rows_on_both_sides_of_every_split(R):
    D = 8
    x = torch.randn(2, 64, 1, R // D, D, generator=torch.Generator().manual_seed(R)).to(torch.float16)
    x[0, 3, 0, -1, -1], x[1, 5, 0, 0, 0] = 40.0, -50.0             # the row's extremes in its last and first elements
    x[1, 7] = x[1, 7] * 0.25 + 60.0                                # quotients beyond the packed arithmetic
    o = O.quant(x.numpy(), m.MASK_V_TOKEN, 0.1)
    dev = x.to(DEV)
    sym, mins, scales = quant(dev, [2, 3, 4], 0.1)
    assert np.array_equal(sym.cpu().numpy(), o[3])
    assert np.array_equal(mins.cpu().numpy().ravel(), np.asarray(o[4]).ravel())
    assert np.array_equal(scales.cpu().numpy().view(np.uint16).ravel(), np.asarray(o[2]).view(np.uint16).ravel())
    mins2, scales2 = torch.empty_like(mins), torch.empty_like(scales)
    counted, book = m.quant_codebook(dev, m.MASK_V_TOKEN, 0.1, mins2, scales2, 0)
    assert torch.equal(counted, sym) and torch.equal(mins2, mins) and torch.equal(scales2, scales)
    counts = m.symbol_counts([sym])
    entries = torch.frombuffer(bytearray(bytes(book.encode_table)[:book.encode_bytes]), dtype=torch.int32)
    assert int((entries[1::2].long() * counts[:entries.numel() // 2]).sum()) == book.payload_bits
