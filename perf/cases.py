"""Performance cases: what programs have this framework do, through its public entry points.

A case is a plain dict.  Its "op" says which of the framework's uses it stands for:

  attend    decode attention of one layer over its compressed cache (CompressedAttention.attend): the call a model makes
            per layer and generated token
  store     compressing a prompt into a fresh K and V context (KVCompCtx.store, set up as the model caches set theirs up):
            the call a model makes per layer and prompt
  restore   the dense fp16 history back from a compressed cache (KVCompCtx.get of K and V): what the caches whose update()
            returns dense tensors do, and what chunked prefill needs
  matvec    the two fused decode + matrix-vector products of the operator module (KVCompCtx.mat_vec_mul of K and V)
  generate  a short generation: prompt stored, then per token and layer an append to K and V and decode attention, with
            blocks recompressed as they leave the uncompressed tails
  simulate  the simulated-quantization cache (KVCompCache with its default backend): prompt, then single tokens

T is the number of tokens held (attend, store, restore, matvec) or the prompt (generate, simulate); H counts KV heads and
rep query heads per KV head.  Shapes and error bounds are those of this repository's benchmark configurations, with odd
lengths beside the round ones; the data have the same distributions (channels of K with outliers and Gaussian V, or
heavy-tailed Laplace), generated on the GPU.
"""
import math

import torch

from kvcomp_amd.attention import CompressedAttention
from kvcomp_amd.cache import KVCompCache
from kvcomp_amd.ctx import KVCompCacheConfig, KVCompCacheConfigStatic, KVCompCtx, QuantMode

DEVICE = "cuda:0"
K_BLOCK, V_BLOCK = 64, 128           # tokens per compressed block, and of the recent window that stays uncompressed


def _case(name, op, B, H, rep, D, T, dist="gauss", eb_k=0.1, eb_v=0.2, k_mode="ChannelQuant", v_mode="TokenQuant", layers=1,
          steps=0):
    return {"name": name, "op": op, "B": B, "H": H, "rep": rep, "D": D, "T": T, "dist": dist, "eb_k": eb_k, "eb_v": eb_v,
            "k_mode": k_mode, "v_mode": v_mode, "layers": layers, "steps": steps}


def listed():
    return [
        # one chat turn with grouped queries, context of an odd length: a call is launches and host time
        _case("attend_chat", "attend", 1, 8, 4, 128, 1000),
        # one sequence, a layer of 32 heads
        _case("attend_single", "attend", 1, 32, 1, 128, 4096),
        # a serving batch in the middle of generation: both tails hold tokens
        _case("attend_batch", "attend", 8, 32, 1, 128, 4177),
        # a batch with grouped queries
        _case("attend_grouped", "attend", 16, 8, 4, 128, 8192),
        # long context, heavy-tailed data, heads that V's tiles straddle: the largest cache of one layer
        _case("attend_long", "attend", 4, 32, 1, 96, 32768, dist="laplace", eb_v=0.3),
        # a short prompt: the latency of a first store with its codebook
        _case("store_chat", "store", 1, 8, 1, 128, 777),
        # a serving batch's prompts
        _case("store_batch", "store", 8, 32, 1, 128, 4096),
        # the long-context prompt
        _case("store_long", "store", 4, 32, 1, 96, 32768, dist="laplace", eb_v=0.3),
        # the history of a batch in the middle of generation handed back dense
        _case("restore_batch", "restore", 8, 32, 1, 128, 4177),
        # the operator module's matrix-vector products on a cache of its own layouts (one K scale per block)
        _case("matvec_block", "matvec", 1, 32, 1, 128, 8192, k_mode="BlockQuant"),
        # a short generation of two layers
        _case("generate_two_layers", "generate", 4, 8, 4, 128, 1500, layers=2, steps=96),
        # the cache that evaluations run
        _case("simulate_prompt", "simulate", 4, 32, 1, 128, 2048, steps=32),
    ]


#: op -> (fewest tokens, most tokens, most elements of one tensor, largest batch)
_RANGES = {
    "attend": (200, 32768, 4 * 32 * 96 * 32768, 16),
    "store": (200, 32768, 4 * 32 * 96 * 32768, 16),
    "restore": (200, 32768, 8 * 32 * 128 * 4177, 16),
    "matvec": (256, 32768, 8 * 32 * 128 * 4096, 8),
    "generate": (150, 4096, 4 * 8 * 128 * 3000, 8),
    "simulate": (150, 4096, 4 * 32 * 128 * 2048, 8),
}


def draw(rng):
    op = rng.choice(["attend", "attend", "attend", "store", "store", "restore", "matvec", "generate", "simulate"])
    lo, hi, most, batches = _RANGES[op]
    H, rep = rng.choice([(32, 1), (8, 4), (16, 2), (8, 8), (8, 1), (24, 1)])
    D = rng.choice([128, 128, 96, 64, 72])
    T = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    B = max(1, min(int(round(math.exp(rng.uniform(0.0, math.log(batches))))), most // (H * D * T)))
    T = max(lo, min(T, most // (B * H * D)))
    dist = rng.choice(["gauss", "gauss", "laplace"])
    case = {"op": op, "B": B, "H": H, "rep": 1 if op in ("store", "restore", "simulate") else rep, "D": D, "T": T, "dist": dist,
            "eb_k": rng.choice([0.05, 0.1, 0.1, 0.2]), "eb_v": rng.choice([0.2, 0.3]) if dist == "gauss" else 0.3,
            "k_mode": rng.choice(["ChannelQuant", "ChannelQuant", "ChannelQuant", "BlockQuant"]), "v_mode": "TokenQuant",
            "layers": 1, "steps": 0}
    if op == "generate":
        case["layers"], case["steps"] = rng.randint(1, 2), rng.randint(20, 96)
    elif op == "simulate":
        case["steps"] = rng.randint(1, 32)
    elif op != "store" and rng.random() < 0.125:
        case["v_mode"] = "VectorQuant"
    return case


def _keys_values(case, gen, tokens):
    """K and V [tokens, B, H, D] fp16 of the case's distribution."""
    B, H, D = case["B"], case["H"], case["D"]

    def laplace():
        u = torch.rand(tokens, B, H, D, generator=gen, device=DEVICE) - 0.5
        x = -torch.sign(u) * torch.log1p(-2.0 * u.abs_().clamp_(max=0.4999999))
        rare = torch.rand(tokens, B, H, D, generator=gen, device=DEVICE) < 0.02
        return torch.where(rare, x * 50.0, x).to(torch.float16)

    if case["dist"] == "laplace":
        return laplace(), laplace()
    channel = torch.exp(0.5 * torch.randn(H, D, generator=gen, device=DEVICE))
    outliers = torch.rand(H, D, generator=gen, device=DEVICE).argsort(dim=1)[:, :4]
    channel.scatter_(1, outliers, channel.gather(1, outliers) * 20.0)
    k = torch.randn(tokens, B, H, D, generator=gen, device=DEVICE).mul_(channel).to(torch.float16)
    return k, torch.randn(tokens, B, H, D, generator=gen, device=DEVICE).to(torch.float16)


def _contexts(case):
    """A K and a V context as the framework's model caches set theirs up."""
    pair = (KVCompCtx(True, case["B"], case["H"], case["D"], case["eb_k"]), KVCompCtx(False, case["B"], case["H"], case["D"], case["eb_v"]))
    for ctx in pair:
        ctx.codebook_smoothing = True
        ctx.async_store = True
    return pair


def _stored(case, k, v):
    kctx, vctx = _contexts(case)
    kctx.store(k, want_symbols=False)
    vctx.store(v, want_symbols=False)
    return kctx, vctx


def _rope(T, D):
    angle = torch.outer(torch.arange(T, dtype=torch.float32, device=DEVICE),
                        1.0 / (10000 ** (torch.arange(0, D, 2, dtype=torch.float32, device=DEVICE) / D)))
    angle = torch.cat([angle, angle], dim=-1)
    return angle.cos()[None].to(torch.float16), angle.sin()[None].to(torch.float16)


def prepare(case, seed):
    KVCompCacheConfigStatic.extract_cache = None
    KVCompCacheConfigStatic.config = KVCompCacheConfig("cases", QuantMode(case["k_mode"]), QuantMode(case["v_mode"]), K_BLOCK, V_BLOCK,
                                                       K_BLOCK, V_BLOCK, case["eb_k"], case["eb_v"])
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    op, B, H, D, T = case["op"], case["B"], case["H"], case["D"], case["T"]
    Hq = H * case["rep"]
    state = {"case": case}
    if op in ("store", "generate"):      # where the program keeps its sequences' streams: room for a byte per symbol, as the encoder asks
        room = (T + case["steps"]) * B * H * D
        state["pool"] = [torch.zeros(room, dtype=torch.uint8, device=DEVICE) for _ in range(2 * case["layers"])]
    if op in ("generate", "simulate"):
        total = T + case["steps"]
        state["kv"] = [_keys_values(case, gen, total) for _ in range(case["layers"])]
        state["q"] = torch.randn(case["steps"], case["layers"], B, Hq, D, generator=gen, device=DEVICE).to(torch.float16)
        if op == "simulate":       # the layout a model's attention layer holds: [B, H, T, D], keys not yet rotated
            state["kv"] = [(k.permute(1, 2, 0, 3).contiguous(), v.permute(1, 2, 0, 3).contiguous()) for k, v in state["kv"]]
            state["rope"] = _rope(total, D)
        return state
    k, v = _keys_values(case, gen, T)
    if op == "store":
        state["kv"] = (k, v)
        return state
    state["ctx"] = kctx, vctx = _stored(case, k, v)
    if op == "attend":
        state["attention"] = CompressedAttention(kctx, vctx)
        state["q"] = torch.randn(B, Hq, D, generator=gen, device=DEVICE).to(torch.float16)
    elif op == "matvec":
        state["q"] = torch.randn(B, Hq, D, generator=gen, device=DEVICE).to(torch.float16)
        state["p"] = torch.softmax(2.5 * torch.randn(B, Hq, vctx.compressed_ctx_len, generator=gen, device=DEVICE), dim=-1).to(torch.float16)
    return state


def _streams(ctx, pool):
    """Everything a context holds: its stream, put into the program's pool (its length depends on the data), the stream's
    tables and parameters, and the uncompressed tail."""
    stream = ctx.encoded_data
    if stream is not None:
        pool[:stream.numel()].copy_(stream)
    return [pool, ctx.block_infos, ctx.thread_infos, ctx.quant_min_ints, ctx.quant_scales, ctx.encode_codebook,
            ctx.decode_codebook, ctx.buffer]


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "attend":
        return state["attention"].attend(state["q"])
    if op == "store":
        kctx, vctx = _stored(case, *state["kv"])
        return _streams(kctx, state["pool"][0]) + _streams(vctx, state["pool"][1])
    if op == "restore":
        kctx, vctx = state["ctx"]
        return kctx.get()[0], vctx.get()[0]
    if op == "matvec":
        kctx, vctx = state["ctx"]
        return kctx.mat_vec_mul(state["q"])[0], vctx.mat_vec_mul(state["p"])[0]
    T, steps = case["T"], case["steps"]
    if op == "generate":
        layers = []
        for k, v in state["kv"]:
            kctx, vctx = _stored(case, k[:T], v[:T])
            layers.append((k, v, kctx, vctx, CompressedAttention(kctx, vctx)))
        out = torch.empty(state["q"].shape, dtype=torch.float32, device=DEVICE)
        for i in range(steps):
            for j, (k, v, kctx, vctx, attention) in enumerate(layers):
                kctx.store(k[T + i:T + i + 1], want_symbols=False)
                vctx.store(v[T + i:T + i + 1], want_symbols=False)
                attention.attend(state["q"][i, j], out=out[i, j])
        streams = [_streams(ctx, pool) for ctx, pool in zip((c for layer in layers for c in layer[2:4]), state["pool"])]
        return [out] + [t for s in streams for t in s]
    cache = KVCompCache(case["B"], case["H"], case["D"], case["layers"])
    cos, sin = state["rope"]
    (k, v), = state["kv"]
    got = cache.update(k[:, :, :T], v[:, :, :T], 0, {"cos": cos[:, :T], "sin": sin[:, :T]})
    for i in range(T, T + steps):
        got = cache.update(k[:, :, i:i + 1], v[:, :, i:i + 1], 0, {"cos": cos[:, i:i + 1], "sin": sin[:, i:i + 1]})
    return got


# ---- the work a pass cannot do without ------------------------------------------------------------------------------

def _bits_per_symbol(case, is_k):
    """Entropy of a quantized symbol: quantizing with a step of eb times a group's range leaves the data's differential entropy
    less log2(step).  A group's range in standard deviations is the expected one of its size."""
    B, H, D = case["B"], case["H"], case["D"]
    eb = case["eb_k"] if is_k else case["eb_v"]
    if is_k:
        group = K_BLOCK if case["k_mode"] == "ChannelQuant" else K_BLOCK * B * H * D
    else:
        group = D if case["v_mode"] == "VectorQuant" else B * H * D
    if case["dist"] == "laplace" and group == K_BLOCK:
        # a fourth of these groups hold none of the rare wide entries, the others one or two: their mean, as measured
        bits = 3.56 - 0.8 * math.log2(eb / 0.1)
    elif case["dist"] == "laplace":
        # 2 % of the entries are 50 times wider: of a group's n entries the widest is near 50 ln(0.02 n)
        spread = 2.0 * 50.0 * (math.log(max(0.02 * group, 1.0)) + 0.6)
        bits = 0.98 * math.log2(max(2.0 * math.e / (eb * spread), 1.0)) + 0.02 * math.log2(max(100.0 * math.e / (eb * spread), 1.0))
    else:
        spread = 2.0 * math.sqrt(2.0 * math.log(group)) * 0.87
        if is_k and case["k_mode"] == "BlockQuant":
            spread *= 20.0 * 3.0       # one scale for all channels: set by the outlier channels
        bits = math.log2(max(4.133 / (eb * spread), 1.0))
    return max(bits, 1.0)


def _held(case, tokens, is_k):
    """(compressed tokens, bytes of the compressed stream, bytes of the fp16 tail) of a context with `tokens` tokens."""
    B, H, D = case["B"], case["H"], case["D"]
    block = K_BLOCK if is_k else V_BLOCK
    done = tokens // block * block
    row = B * H * D
    tiles = (done // 64) * B * H if is_k else (done // 128) * (row // 64)
    if is_k:
        groups = done // 64 * (row if case["k_mode"] == "ChannelQuant" else 1)
    else:
        groups = done * (B * H if case["v_mode"] == "VectorQuant" else 1)
    stream = done * row * _bits_per_symbol(case, is_k) / 8 + tiles * (8 + 128) + groups * 3
    return done, stream, (tokens - done) * row * 2


def work(case):
    op, T = case["op"], case["T"]
    B, H, D, rep = case["B"], case["H"], case["D"], case["rep"]
    row, query = B * H * D, B * H * rep * D
    (kc, ks, kt), (vc, vs, vt) = _held(case, T, True), _held(case, T, False)
    if op == "attend":
        return {"bytes": ks + kt + vs + vt + query * 6, "flops": 4.0 * query * T}
    if op == "store":
        return {"bytes": 2 * T * row * 2 + ks + kt + vs + vt, "flops": 0}
    if op == "restore":
        return {"bytes": ks + kt + vs + vt + 2 * T * row * 2, "flops": 0}
    if op == "matvec":
        return {"bytes": ks + vs + query * 4 + B * H * rep * (kc + vc) * 2, "flops": 2.0 * query * (kc + vc)}
    total = T + case["steps"]
    if op == "generate":
        n = 2 * total * row * 2 + sum(_held(case, total, True)[1:]) + sum(_held(case, total, False)[1:])
        flops = 0.0
        for i in range(case["steps"]):
            n += sum(_held(case, T + i + 1, True)[1:]) + sum(_held(case, T + i + 1, False)[1:]) + query * 6
            flops += 4.0 * query * (T + i + 1)
        return {"bytes": case["layers"] * n, "flops": case["layers"] * flops}
    return {"bytes": 2 * 2 * total * row * 2 + 2 * total * D * 2, "flops": 0}


def tolerance(case):
    if case["op"] in ("store", "restore", "simulate"):
        return "exact"                      # symbols, streams and fp16 values are defined bit for bit
    if case["op"] == "matvec":
        return {"rel": 1e-3}                # fp16 results, V's as fp16 partial sums that are added up
    # fp32 sums and a softmax of fp32 scores, which turns their absolute error into a relative one; streams are whole bytes
    return {"rel": 5e-5}
