"""A context's first store (kvc_quant_codebook, kvc_put_bytes and the encode behind them) against the oracle's quantizer
and the host builder over the same symbols, at the sizes that take different kernels: rows of a wave, of a workgroup and
beyond, per-channel and block groups, groups that leave the packed arithmetic, alphabets beyond the 64 counted in LDS."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import _synth as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _store(is_k, mode, x, eb, asynchronous):
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode(mode if is_k else "ChannelQuant"), QuantMode("TokenQuant" if is_k else mode),
                                                       64, 128, 64, 128, eb, eb)
    T, B, H, D = x.shape
    ctx = KVCompCtx(is_k, B, H, D, eb)
    ctx.async_store = asynchronous
    sym = ctx.store(x.to(DEV))
    return ctx, sym


@pytest.mark.parametrize("asynchronous", [False, True])
@pytest.mark.parametrize("is_k,mode,T,B,H,D,eb", [
    (True, "ChannelQuant", 192, 1, 2, 72, 0.1), (True, "ChannelQuant", 128, 2, 4, 128, 0.012), (True, "BlockQuant", 192, 2, 3, 40, 0.1),
    (True, "BlockQuant", 128, 1, 4, 128, 0.012), (False, "TokenQuant", 256, 1, 4, 64, 0.2), (False, "TokenQuant", 256, 1, 36, 128, 0.012),
    (False, "TokenQuant", 256, 4, 32, 128, 0.2), (False, "TokenQuant", 256, 5, 32, 128, 0.2), (False, "TokenQuant", 256, 9, 32, 128, 0.2),
    (False, "TokenQuant", 256, 17, 32, 128, 0.2), (False, "VectorQuant", 256, 2, 4, 128, 0.2)])
def test_first_store_equals_oracle_and_host_builder(is_k, mode, T, B, H, D, eb, asynchronous):
    import kvcomp_amd.kvcomp_cuda as m
    from kvcomp_amd.compute import dims_to_mask
    x = (S.synth_k if is_k else S.synth_v)(T, B, H, D)
    ctx, sym = _store(is_k, mode, x, eb, asynchronous)
    n = ctx.compressed_ctx_len
    assert n > 0 and sym is not None and sym.numel() == n * B * H * D
    o = O.quant(S.np16(S.blocked(x[:n], ctx.block_size)), dims_to_mask(ctx.quant_dims), eb)
    assert np.array_equal(sym.cpu().numpy(), o[3])
    assert np.array_equal(ctx.quant_min_ints.cpu().numpy().ravel(), np.asarray(o[4]).ravel())
    assert np.array_equal(ctx.quant_scales.cpu().numpy().view(np.uint16).ravel(), np.asarray(o[2]).view(np.uint16).ravel())
    counts = torch.from_numpy(np.bincount(o[3].ravel(), minlength=256))
    enc, dec, fmt = ctx._host_codebook(counts)
    assert ctx.tree_format == fmt and torch.equal(ctx.encode_codebook.cpu(), enc) and torch.equal(ctx.decode_codebook.cpu(), dec)
    assert ctx.max_code_bits == int(enc.view(torch.int32)[1::2].max())
    assert torch.equal(ctx.get_decode_quant_ints()[0], sym)
    # what was reserved for the payload bounds it to a byte per lane stream (and the quarter a growing buffer keeps)
    bound = int((counts * enc.view(torch.int32)[1::2].to(torch.int64).new_tensor(
        np.pad(enc.numpy().view(np.int32)[1::2], (0, 256 - enc.numel() // 8)))).sum()) // 8 + ctx.thread_infos.numel() // 2 + 1
    assert ctx.encoded_data.numel() <= bound and ctx._encoded.data.numel() <= bound + max(bound // 4, 16)
    assert torch.equal(ctx.get()[0][n:].cpu(), x[n:])
    assert m.symbol_counts([sym]).equal(counts)


def test_first_store_far_from_zero_counts_what_it_writes():
    """Groups whose quotients leave the packed arithmetic's range are quantized, and counted, one element at a time."""
    x = (torch.rand(128, 1, 4, 128, generator=torch.Generator().manual_seed(3)) * 0.5 + 60.0).to(torch.float16)
    for is_k, mode in ((True, "ChannelQuant"), (True, "BlockQuant"), (False, "TokenQuant")):
        ctx, sym = _store(is_k, mode, torch.cat([x, x]), 0.1, False)
        counts = torch.bincount(sym.flatten().long(), minlength=256).cpu()
        assert torch.equal(ctx.encode_codebook.cpu(), ctx._host_codebook(counts)[0])
        assert torch.equal(ctx.get_decode_quant_ints()[0], sym)


def test_put_bytes_beyond_one_launch():
    import ctypes as C
    from kvcomp_amd import _lib
    data = np.random.default_rng(1).integers(0, 256, 9001, dtype=np.uint8)
    for n in (1, 3839, 3840, 3841, 9001):
        out = torch.zeros(9010, dtype=torch.uint8, device=DEV)
        _lib.check(_lib.lib().kvc_put_bytes(C.c_void_p(out.data_ptr()), data[:n].tobytes(), n, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert np.array_equal(out.cpu().numpy()[:n], data[:n]) and int(out[n:].max()) == 0


@pytest.mark.parametrize("is_k,mask", [(True, "MASK_K_BLOCK"), (False, "MASK_V_TOKEN")])
def test_one_call_and_its_halves_give_the_same_code(is_k, mask):
    import kvcomp_amd.kvcomp_cuda as m
    T, B, H, D = 256, 2, 3, 128
    blocked = S.blocked((S.synth_k if is_k else S.synth_v)(T, B, H, D), 64 if is_k else 128).to(DEV)
    results = []
    for meanwhile in (None, lambda sym: None):
        groups = m._lib.lib().kvc_quant_groups(*blocked.shape, getattr(m, mask))
        mins, scales = torch.empty(groups, dtype=torch.int8, device=DEV), torch.empty(groups, dtype=torch.float16, device=DEV)
        sym, book = m.quant_codebook(blocked, getattr(m, mask), 0.1, mins, scales, 13, meanwhile)
        results.append((sym, mins, scales, bytes(book)))
    assert all(torch.equal(a, b) for a, b in zip(results[0][:3], results[1][:3])) and results[0][3] == results[1][3]
