"""First stores whose symbols go from the quantizer to the encoder two to a byte write what stores with a byte per symbol write: every
vector length, code lengths on both sides of eight bits, runs of one to four tiles, groups that leave the quantizer's packed
arithmetic, and data whose symbols half a byte does not hold.  The oracle's streams are what the byte path is held to elsewhere."""
import pytest
import torch

import kvcomp_amd.kvcomp_cuda as m
from kvcomp_amd import _lib
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HELD = ("encoded_data", "block_infos", "thread_infos", "quant_min_ints", "quant_scales", "encode_codebook", "decode_codebook", "buffer")


def _ctx(is_k, mode, B, H, D, eb, smoothed=True):
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode(mode if is_k else "ChannelQuant"), QuantMode("TokenQuant" if is_k else mode),
                                                       64, 128, 64, 128, eb, eb)
    ctx = KVCompCtx(is_k, B, H, D, eb)
    ctx.codebook_smoothing, ctx.async_store = smoothed, True
    return ctx


def _data(T, B, H, D, wide, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(T, B, H, D, generator=g, device=DEV)
    if wide:
        x = torch.where(torch.rand(x.shape, generator=g, device=DEV) < 0.02, x * 50, x)
    return x.to(torch.float16)


@pytest.fixture
def packed(monkeypatch):
    """Counts the first stores that took the packed path."""
    calls, original = [], m.quant_codebook_packed

    def quantize(*args):
        calls.append(original(*args))
        return calls[-1]
    monkeypatch.setattr(m, "quant_codebook_packed", quantize)
    return calls


def _both(is_k, mode, x, eb, smoothed=True, polls=None):
    got, want = _ctx(is_k, mode, *x.shape[1:], eb, smoothed), _ctx(is_k, mode, *x.shape[1:], eb, smoothed)
    old = None if polls is None else _lib.set_option(*polls)
    try:
        got.store(x, want_symbols=False)
        held = [getattr(got, name) for name in HELD]
    finally:
        if polls is not None:
            _lib.set_option(polls[0], old)
    want.store(x)
    assert all(torch.equal(a, getattr(want, name)) for a, name in zip(held, HELD))
    assert got.max_tile_bytes == want.max_tile_bytes and got.max_stream_bytes == want.max_stream_bytes and got.max_code_bits == want.max_code_bits
    return got


CASES = [(True, "ChannelQuant", 128, 1, 1, 128, 0.1, False), (True, "ChannelQuant", 192, 1, 3, 96, 0.1, False), (True, "ChannelQuant", 64 * 9, 2, 3, 72, 0.2, True),
         (True, "ChannelQuant", 64 * 10, 2, 5, 64, 1 / 13, False), (True, "ChannelQuant", 64 * 34, 8, 32, 128, 0.1, False), (True, "ChannelQuant", 64 * 34, 6, 32, 96, 0.1, True),
         (True, "ChannelQuant", 64 * 66, 3, 24, 72, 0.1, False), (True, "ChannelQuant", 64 * 66, 3, 24, 64, 0.08, False),
         (True, "BlockQuant", 192, 1, 3, 128, 0.1, False), (True, "BlockQuant", 64 * 34, 5, 32, 128, 0.1, True), (True, "BlockQuant", 64 * 70, 2, 32, 96, 0.1, False),
         (True, "BlockQuant", 64 * 12, 2, 3, 72, 0.2, True), (True, "BlockQuant", 64 * 100, 2, 24, 64, 0.08, True),
         (False, "TokenQuant", 256, 1, 8, 64, 0.2, False), (False, "TokenQuant", 256, 1, 4, 128, 0.1, True), (False, "TokenQuant", 128 * 34, 8, 32, 128, 0.2, False),
         (False, "TokenQuant", 128 * 34, 4, 32, 96, 0.3, True), (False, "TokenQuant", 128 * 20, 8, 24, 72, 0.1, True), (False, "TokenQuant", 128 * 66, 1, 65, 64, 0.2, False),
         (False, "TokenQuant", 128 * 130, 1, 65, 64, 0.2, False), (False, "TokenQuant", 128 * 131, 2, 40, 64, 0.1, True), (False, "TokenQuant", 128 * 4, 16, 32, 128, 0.08, False),
         # more tiles than waves: runs of three and of four, with a last one that is not whole
         (True, "ChannelQuant", 64 * 131, 2, 40, 64, 0.2, False), (True, "BlockQuant", 64 * 101, 2, 65, 64, 0.3, True), (True, "ChannelQuant", 64 * 131, 2, 64, 72, 0.2, True),
         (True, "ChannelQuant", 64 * 132, 2, 64, 96, 0.3, False), (False, "TokenQuant", 128 * 99, 2, 67, 64, 0.2, True), (False, "TokenQuant", 128 * 88, 2, 65, 96, 0.3, False)]


@pytest.mark.parametrize("smoothed", [True, False])
@pytest.mark.parametrize("is_k,mode,T,B,H,D,eb,wide", CASES)
def test_writes_what_a_byte_per_symbol_gives(packed, is_k, mode, T, B, H, D, eb, wide, smoothed):
    ctx = _both(is_k, mode, _data(T, B, H, D, wide, T + D), eb, smoothed)
    assert len(packed) == 1 and packed[0][0].numel() == ctx.compressed_ctx_len * B * H * D // 2


@pytest.mark.parametrize("polls", [("encode_lookback_polls", -1), ("encode_one_pass", 0)])
@pytest.mark.parametrize("is_k,mode,T,B,H,D,eb,wide", [CASES[2], CASES[4], CASES[9], CASES[17]])
def test_a_wave_that_gives_up_and_two_passes(packed, is_k, mode, T, B, H, D, eb, wide, polls):
    _both(is_k, mode, _data(min(T, 64 * 24), B, H, D, wide, 5), eb, polls=polls)
    assert len(packed) == 1


@pytest.mark.parametrize("is_k,mode", [(True, "ChannelQuant"), (True, "BlockQuant"), (False, "TokenQuant")])
def test_groups_beyond_the_packed_arithmetic_and_larger_symbols(packed, is_k, mode):
    x = _data(512, 2, 4, 128, False, 9)
    far = x.clone()
    far[:, :, 1] = far[:, :, 1] * 0.25 + 60.0                      # quotients beyond +-512 in some channels, zero scales in others
    far[:, :, 2, :5] = 3.0
    if mode != "ChannelQuant":
        far = x * 0.25 + 60.0
    _both(is_k, mode, far, 0.1)
    assert len(packed) == 1 and packed[0][1].encode_bytes <= 16 * 8
    tiny = (torch.randint(0, 22, x.shape, generator=torch.Generator().manual_seed(1)).float() * 2.0 ** -24).to(torch.float16).to(DEV)
    ctx = _both(is_k, mode, tiny, 0.078)                           # a range of 21 smallest numbers, a scale of two: or of one
    ctx = _both(is_k, mode, torch.where(tiny.float() * 2 ** 24 > 18, tiny * 0, tiny), 0.08)
    assert len(packed) == 3 and packed[2][1].encode_bytes > 16 * 8 and ctx.encode_codebook.numel() > 16 * 8


@pytest.mark.parametrize("is_k,mode,shape,eb", [(True, "ChannelQuant", (256, 1, 2, 128), 0.05), (True, "ChannelQuant", (256, 1, 4, 40), 0.1),
                                                (False, "VectorQuant", (384, 1, 4, 128), 0.2), (False, "TokenQuant", (384, 1, 2, 128), 0.2)])
def test_other_layouts_keep_a_byte_per_symbol(packed, is_k, mode, shape, eb):
    _both(is_k, mode, _data(*shape, False, 2), eb)
    assert not packed


def test_unaligned_input_keeps_a_byte_per_symbol(packed):
    x = _data(256, 1, 4, 128, False, 3)
    shifted = torch.empty(x.numel() + 4, dtype=torch.float16, device=DEV)[4:].view(x.shape).copy_(x)
    _both(True, "ChannelQuant", shifted, 0.1)
    assert not packed


@pytest.mark.parametrize("name,room,taken", [("kvc_encode_prepare", 16384, True), ("kvc_encode_prepare", 16383, False),
                                             ("kvc_encode_prepare_packed", 16384, False), ("kvc_encode_prepare_packed", 20480, True)])
def test_scratch_that_a_preparation_asks_for(name, room, taken):
    import ctypes as C
    T, B, H, D = 128, 1, 2, 128
    sizes = m.buffer_sizes(T, B * H * D, True, H, D)
    sym, scratch = torch.zeros(T * B * H * D, dtype=torch.uint8, device=DEV), torch.empty(20480, dtype=torch.uint8, device=DEV)
    infos, state = [torch.empty(n, dtype=torch.uint8, device=DEV) for n in sizes[:2]], torch.zeros(16, dtype=torch.int32, device=DEV)
    job = _lib.EncodeJob(is_k=1, d_sym=sym.data_ptr(), tokens=T, batch=B, heads=H, head_dim=D, d_block_infos=infos[0].data_ptr(),
                         d_thread_infos=infos[1].data_ptr(), d_result=state.data_ptr(), d_stream_bytes=state.data_ptr() + 32)
    done = C.c_int(0)
    rc = getattr(_lib.lib(), name)(C.byref(job), scratch.data_ptr(), room, C.byref(done), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (rc == 0) == taken


@pytest.mark.parametrize("mode", ["ChannelQuant", "BlockQuant", "TokenQuant"])
@pytest.mark.parametrize("bits", [0x7e00, 0x7e05, 0xfe0b, 0x7fff])
@pytest.mark.parametrize("tiny", [False, True])
def test_not_a_number_gives_the_same_symbol_in_every_pass(packed, mode, bits, tiny):
    """What a NaN's symbol is depends on which arithmetic its group takes: that of the group, whatever the groups beside it take."""
    is_k = mode != "TokenQuant"
    x = _data(256, 1, 4, 128, False, 12)
    x[70:90, :, 1, 6] = torch.tensor(bits, dtype=torch.int32, device=DEV).to(torch.int16).view(torch.float16)
    if is_k:
        x[:128, :, 1, 8:10] = 3.0                                     # no range, a scale of zero
    if tiny:                                                          # more symbols than half a byte holds
        x[128:192, :, 2, 4] = torch.arange(64, device=DEV).remainder(19).float().mul(2.0 ** -24).to(torch.float16)[:, None]
    _both(is_k, mode, x, 0.08)
    assert len(packed) == 1


@pytest.mark.parametrize("is_k,mode", [(True, "ChannelQuant"), (False, "TokenQuant")])
@pytest.mark.parametrize("eb,smoothed,taken", [(1 / 13, True, 1), (0.0769230769, False, 1), (0.0769230769, True, 0)])
def test_codes_for_seventeen_symbols_keep_a_byte_per_symbol(packed, is_k, mode, eb, smoothed, taken):
    """An error bound that is 1/13 as an fp32 number and a little less in double precision: smoothing starts from ceil(1 / eb)."""
    ctx = _both(is_k, mode, _data(256, 1, 4, 128, False, 4), eb, smoothed)
    assert len(packed) == taken and (ctx.encode_codebook.numel() > 16 * 8) == (not taken)
