"""kvc_append_quantized writes what kvc_append_dense and kvc_quant_in_place write one after the other, bit for bit."""
import pytest
import torch

from tests import _synth as S
from tests.test_gpu_cache import _rope

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one and two pieces of a block per thread, head sizes whose pairs do not divide the workgroup, blocks behind other tokens,
# nothing quantized on one side, groups that leave the packed arithmetic
@pytest.mark.parametrize("B,H,T,D,kn,vn,at", [(2, 3, 200, 128, 128, 128, 0), (1, 5, 197, 96, 192, 0, 7), (2, 2, 64, 64, 64, 0, 0), (1, 2, 131, 16, 64, 128, 1),
                                              (1, 1, 260, 112, 0, 256, 0), (1, 40, 130, 128, 64, 128, 3), (1, 260, 128, 32, 128, 128, 0)])
@pytest.mark.parametrize("v_mode,angles,offset", [("TokenQuant", "shared", 0.0), ("VectorQuant", "per entry", 0.0), ("TokenQuant", "none", 40.0)])
def test_equals_the_two_steps(B, H, T, D, kn, vn, at, v_mode, angles, offset):
    from kvcomp_amd.compute import QuantMode, append_dense, append_quantized, quant_in_place
    k = (S.synth_k(T, B, H, D).permute(1, 2, 0, 3) + offset).to(torch.float16).to(DEV)                   # rows of a token adjacent
    v = (S.synth_v(T, B, H, D).permute(1, 2, 0, 3) + offset).to(torch.float16).contiguous().to(DEV)
    cos, sin = (t.to(DEV) for t in _rope(T, D))
    if angles == "none":
        cos = sin = None
    elif angles == "per entry":
        cos, sin = cos.repeat(B, 1, 1), sin.flip(1).repeat(B, 1, 1)
    caches = [torch.full((B, H, at + T + 5, D), 7.0, dtype=torch.float16, device=DEV) for _ in range(4)]
    mode = QuantMode(v_mode)
    assert append_quantized(k, v, cos, sin, caches[0], caches[1], at, (kn, 64, 0.1, QuantMode.ChannelQuant), (vn, 64, 0.2, mode))
    assert append_dense(k, v, cos, sin, caches[2], caches[3], at)
    quant_in_place(caches[2][:, :, at:at + kn], 64, 0.1, QuantMode.ChannelQuant)
    quant_in_place(caches[3][:, :, at:at + vn], 64, 0.2, mode)
    assert torch.equal(caches[0].view(torch.int16), caches[2].view(torch.int16))
    assert torch.equal(caches[1].view(torch.int16), caches[3].view(torch.int16))


def test_what_it_does_not_take_is_left_alone():
    from kvcomp_amd.compute import QuantMode, append_quantized
    C, T, V, B = QuantMode.ChannelQuant, QuantMode.TokenQuant, QuantMode.VectorQuant, QuantMode.BlockQuant
    for D, heads, k_plan, v_plan in ((72, 2, (64, 64, .1, C), (64, 64, .2, T)), (64, 2, (64, 64, .1, B), (64, 64, .2, T)),
                                     (64, 2, (128, 128, .1, C), (128, 128, .2, V)), (128, 520, (64, 64, .1, C), (64, 64, .2, T))):
        x = torch.randn(1, heads, 130, D, dtype=torch.float16, device=DEV)
        cache = torch.full_like(x, 3.0)
        assert not append_quantized(x, x, None, None, cache, cache, 0, k_plan, v_plan) and (cache == 3).all()


@pytest.mark.parametrize("angles", [False, True])
@pytest.mark.parametrize("D", [128, 96, 16])
def test_special_values(D, angles):
    """Channels whose minima and maxima are joined from parts: constant ones, zeros of both signs, infinities, NaN in one part,
    in several and everywhere, the largest and the smallest values.  The same bits as the two steps (of a NaN, that it is one)."""
    from kvcomp_amd.compute import QuantMode, append_dense, append_quantized, quant_in_place
    B, H, T = 2, 3, 140
    g = torch.Generator().manual_seed(D)
    k, v = (torch.randn(B, H, T, D, generator=g).to(torch.float16) for _ in range(2))
    inf, nan = float("inf"), float("nan")
    for x in (k, v):
        x[..., 0] = 0.375
        x[..., 1] = 0.0
        x[..., 2] = torch.where(torch.arange(T) % 3 == 0, -0.0, 0.0).to(torch.float16)
        x[0, :, 17, 3], x[0, :, 90, 4] = inf, -inf
        x[1, 0, 5, 5], x[1, 0, 40, 5], x[1, 0, 41, 5] = inf, -inf, nan
        x[:, 1, 0, 6], x[:, 1, 63, 7], x[:, 1, 64:128, 8] = nan, nan, nan
        x[:, 2, 2:64:4, 9] = nan
        x[..., 10] = torch.where(torch.arange(T) % 2 == 0, 65504.0, -65504.0).to(torch.float16)
        x[..., 11] = 6e-8 * (torch.arange(T) % 5).to(torch.float16)
        x[0, 0, 70], x[1, 2, 71], x[1, 2, 72] = nan, inf, 1.5       # whole vectors
    k, v = k.to(DEV), v.to(DEV)
    cos, sin = (t.to(DEV) for t in _rope(T, D)) if angles else (None, None)
    caches = [torch.full((B, H, T + 3, D), 7.0, dtype=torch.float16, device=DEV) for _ in range(4)]
    for v_mode in (QuantMode.TokenQuant, QuantMode.VectorQuant):
        assert append_quantized(k, v, cos, sin, caches[0], caches[1], 0, (128, 64, 0.1, QuantMode.ChannelQuant), (128, 64, 0.2, v_mode))
        assert append_dense(k, v, cos, sin, caches[2], caches[3], 0)
        quant_in_place(caches[2][:, :, :128], 64, 0.1, QuantMode.ChannelQuant)
        quant_in_place(caches[3][:, :, :128], 64, 0.2, v_mode)
        for one, two in ((caches[0], caches[2]), (caches[1], caches[3])):
            assert bool(((one.view(torch.int16) == two.view(torch.int16)) | (one.isnan() & two.isnan())).all())
        if not angles:                                            # (a rotation carries a NaN to the channel's partner)
            assert bool(torch.isfinite(caches[0][0, 1, :128, D - 1]).all())
