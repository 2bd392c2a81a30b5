"""Head sizes of which a tile of 64 V channels can touch three and more heads (8, 16, 24, 40), beside the ones next to them that
stay at two: V's products, attention and the restored values, for every layout of V's groups."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests import _synth as S
from tests.test_gpu_codec import _dev, _make_stream, kc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(params=[1, 0], ids=["rounded", "unrounded"])
def rounded(request):
    from kvcomp_amd import _lib
    was = _lib.set_option("fused_rounded", request.param)
    yield request.param
    _lib.set_option("fused_rounded", was)


SHAPES = [(8, 2, 8), (16, 1, 4), (24, 1, 8), (24, 2, 4), (40, 1, 8), (40, 3, 8), (32, 2, 3), (48, 1, 4), (56, 1, 8)]      # D, B, H


@pytest.mark.parametrize("D,B,H", SHAPES)
@pytest.mark.parametrize("rep", [1, 2, 4, 8])
@pytest.mark.parametrize("mask", [O.MASK_V_TOKEN, O.MASK_SIM_TOKEN, O.MASK_VECTOR])
@pytest.mark.parametrize("eb", [0.2, 0.03])                        # codes within a look-up's index, and longer ones
def test_products_equal_the_oracles(D, B, H, rep, mask, eb, rounded):
    T = 256
    s = _make_stream(S.synth_v(T, B, H, D), False, eb, mask, 128)
    p = S.synth_p(B, H * rep, T)
    ref = O.fused_v(s["sym"].reshape(T, B, H, D), s["mn"], s["scale"], mask, 128, S.np16(p))
    part = torch.full((T // 128, B, H * rep, D), float("nan"), dtype=torch.float16, device=DEV)
    kc().v_decode_and_mat_vec_mul_cuda_export(_dev(s["dec"]), _dev(s["bi"]), _dev(s["ti"]), _dev(s["payload"]), _dev(s["mn"].ravel()),
                                              _dev(s["scale"].ravel().view(np.uint16), torch.float16), p.to(DEV), part, H, D)
    got = part.float().sum(dim=0).cpu().numpy().astype(np.float64)
    assert np.abs(got - ref).max() <= 1e-3 * np.abs(ref).max()     # (fp16 partial sums: 2^-11 of each)


@pytest.mark.parametrize("D,B,H", SHAPES)
@pytest.mark.parametrize("rep", [1, 4])
@pytest.mark.parametrize("v_mode", ["TokenQuant", "VectorQuant"])
def test_attention_and_restored_values(D, B, H, rep, v_mode, rounded):
    from kvcomp_amd.attention import CompressedAttention
    from kvcomp_amd.compute import dequant
    from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode
    KVCompCacheConfigStatic.config = KVCompCacheConfig("t", QuantMode.ChannelQuant, QuantMode(v_mode), 64, 128, 64, 128, 0.1, 0.2)
    T = 555
    pair = KVCompCtx(True, B, H, D, 0.1), KVCompCtx(False, B, H, D, 0.2)
    dense, exact = [], []
    for c, x in zip(pair, (S.synth_k(T, B, H, D), S.synth_v(T, B, H, D))):
        c.codebook_smoothing = True
        c.store(x.to(DEV), want_symbols=False)
        sym = c.get_decode_quant_ints()[0]
        dense.append(torch.cat([dequant(sym, c.quant_min_ints, c.quant_scales, c.quant_dims).flatten(0, 1), c.buffer]))
        assert torch.equal(c.get()[0].view(torch.int16), dense[-1].view(torch.int16))
        values = (sym.double() + c.quant_min_ints.double()) * c.quant_scales.double()      # what is not rounded to fp16
        exact.append(torch.cat([values.flatten(0, 1), c.buffer.double()]))
    q = S.synth_q(B, H * rep, D)
    k, v = (t.double().cpu().repeat_interleave(rep, dim=2) for t in (dense if rounded else exact))
    w = torch.softmax(torch.einsum("tbhd,bhd->bht", k, q.double()) / D ** 0.5, dim=-1)
    want = torch.einsum("tbhd,bht->bhd", v, w)
    got = CompressedAttention(*pair).attend(q.to(DEV)).double().cpu()
    # fp32 scores of up to some hundred (K's outliers), whose absolute error of about 2^-17 the softmax makes a relative one
    assert (got - want).abs().max() <= 1e-4 * want.abs().max()
