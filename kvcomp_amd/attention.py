"""Decode attention straight from a compressed KV cache.

The reference stops at two separate kernels (models/cache/kvcomp_encode.py:209-280): raw q.K scores and
per-128-token partial p.V sums that PyTorch adds up; nothing chains them, applies 1/sqrt(d) or softmax, or
handles grouped-query heads (kvcomp_encode.py:328-368 is unreachable code).  This module is that missing
operator: for one layer it owns a K context and a V context (kvcomp_amd.ctx.KVCompCtx) and computes

    out[b, hq] = softmax(q[b, hq] . K[b, hq // rep] / sqrt(d)) . V[b, hq // rep]

over the compressed tokens and the uncompressed tail, with the decoded symbols never written to HBM.
"""
import ctypes as C
import math
from typing import Optional

import torch

from . import _lib, kvcomp_cuda
from ._lib import KvcompError, check
from .compute import dims_to_mask
from .ctx import KVCompCtx
from .kvcomp_cuda import build_lut  # noqa: F401


def _ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(0)


def _stream(t):
    return C.c_void_p(_lib.stream_of(t))


def k_scores(ctx: KVCompCtx, lut: torch.Tensor, q: torch.Tensor, out: Optional[torch.Tensor] = None,
             timed: bool = False):
    """fp32 scores [B, Hq, ctx_c] = q . dequant(K) for the compressed part of a K context."""
    B, Hq, D = q.shape
    if out is None:
        out = torch.empty(B, Hq, ctx.compressed_ctx_len, dtype=torch.float32, device=q.device)
    ms = C.c_float(0.0)
    with _lib.device_guard(q):
        check(_lib.lib().kvc_k_scores_lut(
            _ptr(lut), 0, _ptr(ctx.block_infos), ctx.block_infos.numel(), _ptr(ctx.thread_infos), ctx.thread_infos.numel(),
            _ptr(ctx.encoded_data), ctx.encoded_data.numel(), _ptr(ctx.quant_min_ints), _ptr(ctx.quant_scales),
            dims_to_mask(ctx.quant_dims), _ptr(q), _ptr(out), 1 if out.dtype == torch.float32 else 0, ctx.max_tile_bytes,
            ctx.max_stream_bytes, ctx.code_hint,
            ctx.compressed_ctx_len, B, ctx.head_num, Hq, D, C.byref(ms) if timed else None, _stream(q)))
    return out, float(ms.value)


def v_partials(ctx: KVCompCtx, lut: torch.Tensor, p: torch.Tensor, out: Optional[torch.Tensor] = None,
               timed: bool = False):
    """fp32 partial sums [ctx_c / 128, B, Hq, D] of p . dequant(V) for the compressed part of a V context."""
    B, Hq, T = p.shape
    if out is None:
        out = torch.empty(T // kvcomp_cuda.V_VEC_LEN, B, Hq, ctx.head_dim, dtype=torch.float32, device=p.device)
    ms = C.c_float(0.0)
    with _lib.device_guard(p):
        check(_lib.lib().kvc_v_partials_lut(
            _ptr(lut), 0, _ptr(ctx.block_infos), ctx.block_infos.numel(), _ptr(ctx.thread_infos), ctx.thread_infos.numel(),
            _ptr(ctx.encoded_data), ctx.encoded_data.numel(), _ptr(ctx.quant_min_ints), _ptr(ctx.quant_scales),
            dims_to_mask(ctx.quant_dims), _ptr(p), _ptr(out), 1 if out.dtype == torch.float32 else 0, ctx.max_tile_bytes,
            ctx.max_stream_bytes, ctx.code_hint,
            T, B, ctx.head_num, Hq, ctx.head_dim, C.byref(ms) if timed else None, _stream(p)))
    return out, float(ms.value)


class CompressedAttention:
    """Decode attention of one layer over (compressed K, compressed V, uncompressed tails)."""

    def __init__(self, k_ctx: KVCompCtx, v_ctx: KVCompCtx):
        assert k_ctx.is_k and not v_ctx.is_k
        self.k, self.v = k_ctx, v_ctx
        self._workspace = None
        self._workspace_key = None

    def _luts(self):
        return self.k.decode_lut(), self.v.decode_lut()

    @staticmethod
    def _bracket(prof, key):
        if prof is None:
            return None
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        prof[key].append((a, b))
        a.record()
        return b

    @staticmethod
    def _bracket_end(ev):
        if ev is not None:
            ev.record()

    def _desc(self, ctx: KVCompCtx, lut) -> "_lib.CompressedDesc":
        return ctx.descriptor()

    def attend(self, q: torch.Tensor, scale: Optional[float] = None, out: Optional[torch.Tensor] = None,
               kernel_ms: Optional[list] = None) -> torch.Tensor:
        """q fp16 [B, Hq, D] -> fp32 [B, Hq, D] over every stored token, as one library call
        (kvc_attention_decode): scores, softmax and the weighted sum of values never pass through PyTorch.
        `kernel_ms`, if a list, receives (fused K kernel ms, fused V kernel ms) -- which makes the call wait."""
        B, Hq, D = q.shape
        k, v = self.k, self.v
        assert q.dtype is torch.float16 and v.ctx_len == k.ctx_len
        device = q.device
        if not device == k.device == v.device:
            raise KvcompError("queries on %s, keys on %s, values on %s" % (device, k.device, v.device))
        if scale is None:
            scale = 1.0 / math.sqrt(D)
        L = _lib.lib()
        # (what the workspace has to hold grows with the tokens: asked for in steps of 1024)
        index = q.get_device()
        key = ((k.ctx_len + 1023) // 1024, B, Hq, D, index)
        if key != self._workspace_key:
            need = int(L.kvc_attention_workspace_bytes(key[0] * 1024, key[0] * 1024, B, Hq, D))
            if self._workspace is None or self._workspace.numel() < need or self._workspace.device != device:
                _lib.let_go(self._workspace)
                self._workspace = torch.empty(need + need // 4, dtype=torch.uint8, device=device)
            self._workspace_key = key
        if out is None:
            out = torch.empty(B, Hq, D, dtype=torch.float32, device=device)
        kd, vd = k.descriptor(), v.descriptor()
        q = q.contiguous()
        ms = (C.c_float * 2)() if kernel_ms is not None else None
        workspace = self._workspace
        if index >= 0 and torch._C._cuda_getDevice() == index:
            rc = L.kvc_attention_decode(kd, vd, q.data_ptr(), scale, workspace.data_ptr(), workspace.numel(), out.data_ptr(),
                                        B, k.head_num, Hq, D, None, ms, torch._C._cuda_getCurrentRawStream(index))
        else:
            with _lib.device_guard(q):
                rc = L.kvc_attention_decode(kd, vd, q.data_ptr(), scale, workspace.data_ptr(), workspace.numel(), out.data_ptr(),
                                            B, k.head_num, Hq, D, None, ms, _lib.stream_of(q))
        if rc:
            check(rc)
        if kernel_ms is not None:
            kernel_ms[:] = [float(ms[0]), float(ms[1])]
        return out

    def attend_stepwise(self, q: torch.Tensor, scale: Optional[float] = None, prof: Optional[dict] = None) -> torch.Tensor:
        """The same result assembled from the reference-shaped pieces (fused K scores, PyTorch softmax, fused
        p.V partials, PyTorch reduction).  q fp16 [B, Hq, D] -> fp32 [B, Hq, D].  Covers every stored token: the compressed part through the
        fused kernels, the fp16 tails (K and V compress on different block sizes, so their tails differ)
        through dense matvecs.  `prof`, if given, collects (start, end) event pairs recorded on the launch
        stream around the two fused kernels under the keys "k" and "v"."""
        B, Hq, D = q.shape
        rep = Hq // self.k.head_num
        scale = scale if scale is not None else 1.0 / math.sqrt(D)
        k_lut, v_lut = self._luts()
        T = self.k.ctx_len
        assert self.v.ctx_len == T
        kc, vc = self.k.compressed_ctx_len, self.v.compressed_ctx_len
        parts = []
        if kc:
            ev = self._bracket(prof, "k")
            parts.append(k_scores(self.k, k_lut, q)[0])
            self._bracket_end(ev)
        if kc != T:
            tail = self.k.buffer.float().repeat_interleave(rep, dim=2)                  # [t, B, Hq, D]
            parts.append(torch.einsum("tbhd,bhd->bht", tail, q.float()))
        scores = parts[0] if len(parts) == 1 else torch.cat(parts, dim=-1)
        p = torch.softmax(scores * scale, dim=-1)
        out = torch.zeros(B, Hq, D, dtype=torch.float32, device=q.device)
        if vc:
            p16 = p[:, :, :vc].to(torch.float16).contiguous()
            ev = self._bracket(prof, "v")
            part, _ = v_partials(self.v, v_lut, p16)
            self._bracket_end(ev)
            out += part.sum(dim=0)
        if vc != T:
            tail = self.v.buffer.float().repeat_interleave(rep, dim=2)
            out += torch.einsum("tbhd,bht->bhd", tail, p[:, :, vc:])
        return out
