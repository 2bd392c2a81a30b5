"""A tile's payload is written in whole 16-byte pieces of the destination and single bytes at its ends: wherever the payload buffer starts,
the bytes are those of an aligned one and nothing beside them is touched -- from symbols (both kernels) and straight from fp16."""
import ctypes as C

import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
T, B, H = 256, 1, 4


def _encode(is_k, D, x, sym, table, offset, fused):
    sizes = m.buffer_sizes(T, B * H * D, is_k, H, D)
    infos, state = [torch.empty(n, dtype=torch.uint8, device=DEV) for n in sizes[:2]], torch.zeros(16, dtype=torch.int32, device=DEV)
    room = T * B * H * D
    buffer = torch.full((room + 64,), 0xA5, dtype=torch.uint8, device=DEV)
    start = (-buffer.data_ptr()) % 16 + offset
    mins, scales = torch.empty(65536, dtype=torch.int8, device=DEV), torch.empty(65536, dtype=torch.float16, device=DEV)
    job = _lib.EncodeJob(is_k=int(is_k), tokens=T, batch=B, heads=H, head_dim=D, d_encode_tables=table.data_ptr(), encode_table_bytes=table.numel(),
                         d_block_infos=infos[0].data_ptr(), d_thread_infos=infos[1].data_ptr(), d_encoded=buffer.data_ptr() + start, encoded_cap=room,
                         d_result=state.data_ptr(), d_stream_bytes=state.data_ptr() + 32)
    if fused:
        job.d_x_f16, job.quant_mask, job.eb, job.d_min_i8, job.d_scale_f16 = x.data_ptr(), m.MASK_CHANNEL if is_k else m.MASK_V_TOKEN, 0.1, mins.data_ptr(), scales.data_ptr()
    else:
        job.d_sym = sym.data_ptr()
    m.check(_lib.lib().kvc_encode_async(C.byref(job), torch.cuda.current_stream().cuda_stream))
    n = m.encode_result(state[:8], room)[0]
    assert bool((buffer[:start] == 0xA5).all()) and bool((buffer[start + n:] == 0xA5).all())
    return [buffer[start:start + n]] + infos


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("is_k,D", [(True, 128), (True, 72), (True, 40), (False, 128), (False, 64)])
def test_wherever_the_payload_starts(is_k, D, fused):
    x = torch.randn(T // (64 if is_k else 128), 64 if is_k else 128, B, H, D, generator=torch.Generator(device=DEV).manual_seed(D), device=DEV).to(torch.float16)
    mask = m.MASK_CHANNEL if is_k else m.MASK_V_TOKEN
    groups = _lib.lib().kvc_quant_groups(*x.shape, mask)
    sym, book = m.quant_codebook(x, mask, 0.1, torch.empty(groups, dtype=torch.int8, device=DEV), torch.empty(groups, dtype=torch.float16, device=DEV), 13)
    table = torch.frombuffer(bytearray(bytes(book.encode_table)[:book.encode_bytes]), dtype=torch.uint8).to(DEV)
    want = _encode(is_k, D, x, sym, table, 0, fused)
    for offset in list(range(1, 16)) + [17]:
        assert all(torch.equal(g, w) for g, w in zip(_encode(is_k, D, x, sym, table, offset, fused), want))
