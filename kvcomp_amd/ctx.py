"""Compressed KV-cache context: the object layout and methods of the reference's KVCompCtx
(models/cache/kvcomp_encode.py:15-326), with every device step running through libkvcomp_hip.

Same attribute names (encoded_data, block_infos, thread_infos, quant_min_ints, quant_scales, encode_codebook,
decode_codebook, buffer, ctx_len, compressed_ctx_len, shape) and the same method contracts (store, get,
get_only_compressed, get_decode_quant_ints, mat_vec_mul, build_codebook, get_cr).  Differences:

  * the quantizer is one HIP launch instead of ~8 fp16 PyTorch kernels (bit-identical symbols);
  * encoder scratch is kept per device and only grows (the reference re-allocates and zero-fills four
    buffers on every store, kvcomp_encode.py:88-95), and the accumulated stream lives in amortised
    growable buffers instead of being re-concatenated on every store (kvcomp_encode.py:129-133);
  * batch > 1 and per-channel K (QuantMode.ChannelQuant) are accepted.
"""
import ast
import collections
import contextlib
import ctypes as C
import itertools
import math
import struct
from typing import Dict, List, NamedTuple, Optional, Tuple

import torch

from . import _lib, kvcomp_cuda
from ._lib import KvcompError
from .compute import (QUANT_MODE_MAP, QuantMode, blocks_to_compress, cut_tensor_ctx_len_0, dequant, dims_to_mask,  # noqa: F401
                      expected_groups, mask_keepdim_shape, quant, safe_cat)


class ExtractCacheConfig:
    """utils/config.py:3-19"""

    def __init__(self, collect_round: int):
        self.collect_round = collect_round
        self.key_caches = {}
        self.value_caches = {}

    def size(self):
        total = 0
        for caches in (self.key_caches, self.value_caches):
            for per_round in caches.values():
                for t in per_round.values():
                    total += t.numel() * 16
        return total


class KVCompCacheConfig:
    """utils/config.py:21-140: the eleven configuration fields, printable and parseable."""

    _FIELDS = ("enable_quant", "model_name", "enable_pre_rope", "k_quant_mode", "v_quant_mode", "k_block_size",
               "v_block_size", "k_recent_size", "v_recent_size", "k_quant_scale_rel", "v_quant_scale_rel")

    def __init__(self, model_name, k_quant_mode, v_quant_mode, k_block_size, v_block_size, k_recent_size,
                 v_recent_size, k_quant_scale_rel, v_quant_scale_rel, enable_quant=True, enable_pre_rope=False):
        self.enable_quant = enable_quant
        self.model_name = model_name
        self.enable_pre_rope = enable_pre_rope
        self.k_quant_mode = k_quant_mode
        self.v_quant_mode = v_quant_mode
        self.k_block_size = k_block_size
        self.v_block_size = v_block_size
        self.k_recent_size = k_recent_size
        self.v_recent_size = v_recent_size
        self.k_quant_scale_rel = k_quant_scale_rel
        self.v_quant_scale_rel = v_quant_scale_rel

    def __str__(self):
        d = {"enable_quant": self.enable_quant, "enable_pre_rope": self.enable_pre_rope, "model_name": self.model_name}
        if self.enable_quant:
            d.update(k_quant_mode=self.k_quant_mode.value, v_quant_mode=self.v_quant_mode.value,
                     k_block_size=self.k_block_size, v_block_size=self.v_block_size,
                     k_recent_size=self.k_recent_size, v_recent_size=self.v_recent_size,
                     k_quant_scale_rel=self.k_quant_scale_rel, v_quant_scale_rel=self.v_quant_scale_rel)
        return str(d)

    __repr__ = __str__

    @staticmethod
    def from_str(text: str):
        d = ast.literal_eval(text)       # the reference uses eval (utils/config.py:71); literals are all it needs
        if d["enable_quant"]:
            kw = dict(k_quant_mode=QuantMode(d["k_quant_mode"]), v_quant_mode=QuantMode(d["v_quant_mode"]),
                      k_block_size=d["k_block_size"], v_block_size=d["v_block_size"],
                      k_recent_size=d["k_recent_size"], v_recent_size=d["v_recent_size"],
                      k_quant_scale_rel=d["k_quant_scale_rel"], v_quant_scale_rel=d["v_quant_scale_rel"])
        else:
            kw = dict(k_quant_mode=None, v_quant_mode=None, k_block_size=None, v_block_size=None, k_recent_size=None,
                      v_recent_size=None, k_quant_scale_rel=None, v_quant_scale_rel=None)
        return KVCompCacheConfig(model_name=d["model_name"], enable_quant=d["enable_quant"],
                                 enable_pre_rope=d["enable_pre_rope"], **kw)

    def _key(self):
        return tuple(getattr(self, f) for f in self._FIELDS)

    def __eq__(self, other):
        return isinstance(other, KVCompCacheConfig) and self._key() == other._key()

    def __hash__(self):
        return hash(self._key())


class KVCompCacheConfigStatic:
    """Process-wide configuration slot (models/cache/kvcomp_quant.py:10-12)."""
    config: Optional[KVCompCacheConfig] = None
    extract_cache: Optional[ExtractCacheConfig] = None


class _Growable:
    """Device buffer that grows geometrically (by a quarter) along dim 0; `.view` is the filled prefix."""

    def __init__(self):
        self.data: Optional[torch.Tensor] = None
        self.used = 0
        self.row = 1              # elements per row of `data`

    def _hold(self, data: torch.Tensor):
        _lib.let_go(self.data)                                 # (copied from on this stream, and written to by queued encodes)
        self.data, self.row = data, math.prod(data.shape[1:])

    def append(self, t: torch.Tensor):
        n = t.shape[0]
        # room for a quarter more than is needed: re-allocation stays rare while decoding appends small pieces, and a
        # context never holds much more than its stream
        if self.data is None:
            cap = n + max(n // 4, 16)
            self._hold(torch.empty((cap,) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device))
        elif self.used + n > self.data.shape[0]:
            cap = self.used + n + max((self.used + n) // 4, 16)
            grown = torch.empty((cap,) + tuple(self.data.shape[1:]), dtype=self.data.dtype, device=self.data.device)
            grown[:self.used] = self.data[:self.used]
            self._hold(grown)
        self.data[self.used:self.used + n] = t
        self.used += n

    def reserve(self, n: int, tail_shape, dtype, device, pending: int = 0):
        """Make room for n more rows behind the filled part (which is kept, with `pending` rows behind it); returns the view
        of the rows behind the filled part."""
        kept = self.used + pending
        if self.data is None:
            self._hold(torch.empty((n + max(n // 4, 16),) + tuple(tail_shape), dtype=dtype, device=device))
        elif kept + n > self.data.shape[0]:
            cap = kept + n + max((kept + n) // 4, 16)
            grown = torch.empty((cap,) + tuple(self.data.shape[1:]), dtype=self.data.dtype, device=self.data.device)
            grown[:kept] = self.data[:kept]
            self._hold(grown)
        return self.data[self.used:self.used + n]

    def trim(self):
        """Give back what was reserved beyond a quarter of the filled part (after a worst-case reservation)."""
        cap = self.used + max(self.used // 4, 16)
        if self.data is not None and self.data.shape[0] > cap:
            kept = torch.empty((cap,) + tuple(self.data.shape[1:]), dtype=self.data.dtype, device=self.data.device)
            kept[:self.used] = self.data[:self.used]
            self._hold(kept)

    @property
    def view(self) -> Optional[torch.Tensor]:
        return None if self.data is None else self.data[:self.used]


class _Outcome:
    """Pinned host words that a context's queued encodes leave their result in: written by an encode's last kernel and closed
    with the number of the call (word 9); words 10 - 12 say which stream and device that is to come from.  Used like an event; looking costs no call into the runtime, where a copy and an
    event behind every encode cost ten microseconds of host time and a launch."""
    _numbers = itertools.count(1)
    _late: collections.deque = collections.deque()       # words whose context is gone while a kernel may still write to them
    __slots__ = ("words", "_seen", "number", "stream")

    def __init__(self):
        for _ in range(len(_Outcome._late)):
            try:
                late = _Outcome._late.popleft()
            except IndexError:
                break
            if int(late[0][9]) != late[1]:
                _Outcome._late.append(late)
        self.number = self.stream = 0
        self.words = torch.empty(16, dtype=torch.int32, pin_memory=True)
        self._seen = self.words.numpy()
        self._seen[9:13] = 0

    def ask(self, stream: int) -> Tuple[int, int]:
        """What the next encode on `stream` is to be told; if the library refuses it, refused() has to follow."""
        self.number, self.stream = (next(_Outcome._numbers) & 0x7fffffff) or 1, stream
        return self.words.data_ptr(), self.number

    def refused(self, number: int, stream: int):
        """The encode that was told the latest number has failed, and nothing of it is queued any more: whoever waits for an
        earlier one goes on waiting for its `number` on `stream`.  (A call can fail behind its launches, for an error that
        something else had left; its number is there then, and its words are the newer ones.)"""
        if not self.query():
            self.number, self.stream = number, stream

    def query(self) -> bool:
        return int(self._seen[9]) == self.number

    def synchronize(self):
        """Until the number is there; if its stream runs dry without it, query() says so."""
        _lib.check(_lib.lib().kvc_wait_outcome(self.words.data_ptr(), self.number))

    def __del__(self):
        if getattr(self, "_seen", None) is not None and not self.query():
            self._late.append((self._seen, self.number))


class _QueuedStore(NamedTuple):
    """An encode that was queued and has not been seen to succeed."""
    tokens: int
    rows: Optional[torch.Tensor]     # its tokens' fp16 rows, if they were kept
    books: tuple                     # the bookkeeping as it stood right after the store
    worst: int                       # the store's share of _enc_pending
    lost: bool                       # its tokens are gone if it has to be taken back: counted in ctx_len, rows not kept
    certain: bool                    # nothing about it can fail, whatever a later store does
    codebook: bool                   # it brought the codebook, which goes with it
    done: Optional["torch.cuda.Event"] = None        # behind it on its stream, if it had no outcome's words to write to


class _NativeFirst:
    """What _first_chunk hands the quantizer's second half: the codebook and the encode with it in one native call
    (first_encode of kvcomp_host_module.cpp)."""
    __slots__ = ("prepared", "place", "vectors", "outcome", "before", "told", "failed", "most", "payload")

    def __init__(self, prepared, place, vectors, outcome, stream):
        self.prepared, self.place, self.vectors, self.outcome = prepared, place, vectors, outcome
        self.failed, self.most, self.payload = 0, 0, None
        self.before = outcome.number, outcome.stream
        self.told = outcome.ask(stream)

    def __call__(self, counted, smoothed, book, stream):
        p = self.prepared
        rc, self.failed, self.most, self.payload = _lib.host().first_encode(
            counted, smoothed, C.addressof(book), C.addressof(p.job), p.scratch.data_ptr(), p.done, self.place, _lib.lib().kvc_lut_bytes(),
            self.vectors, *self.told, stream)
        return rc

    def refused(self):
        self.outcome.refused(*self.before)


# the seventeen 8-byte fields of kvc_compressed_desc, in order
_DESC = struct.Struct("=17q")


class KVCompCtx:
    """One compressed K or V stream of one layer (models/cache/kvcomp_encode.py:15-326)."""

    # encoder scratch shared by every context on a device (kvcomp_encode.py:17-21); grown, never shrunk
    buffer_ctx_len: Dict[torch.device, int] = dict()
    block_infos_buffer: Dict[torch.device, torch.Tensor] = dict()
    thread_infos_buffer: Dict[torch.device, torch.Tensor] = dict()
    idx_offset_buffer: Dict[torch.device, torch.Tensor] = dict()
    pre_alloc_compressed_data_buffer: Dict[torch.device, torch.Tensor] = dict()

    def __init__(self, is_k: bool, batch_size: int, head_num: int, head_dim: int, quant_scale_rel: float,
                 encode_codebook_path: str = None, decode_codebook_path: str = None):
        cfg = KVCompCacheConfigStatic.config
        assert cfg is not None, "KVCompCacheConfigStatic.config is None"
        assert cfg.k_quant_mode in (QuantMode.BlockQuant, QuantMode.ChannelQuant), \
            "k_quant_mode must be BlockQuant or ChannelQuant for the kernel implementation"
        assert cfg.v_quant_mode in (QuantMode.TokenQuant, QuantMode.VectorQuant), \
            "v_quant_mode must be TokenQuant or VectorQuant for the kernel implementation"
        assert head_dim <= kvcomp_cuda.K_VEC_LEN and head_dim % 8 == 0, "head_dim must be a multiple of 8, at most K_VEC_LEN"
        self.is_k = is_k
        self.batch_size = batch_size
        self.head_num = head_num
        self.head_dim = head_dim
        self.quant_scale_rel = quant_scale_rel
        self.ctx_len = 0
        self.compressed_ctx_len = 0
        self.device: Optional[torch.device] = None
        self.quant_dims = QUANT_MODE_MAP[cfg.k_quant_mode] if is_k else QUANT_MODE_MAP[cfg.v_quant_mode]
        self.block_size = cfg.k_block_size if is_k else cfg.v_block_size
        self.recent_size = cfg.k_recent_size if is_k else cfg.v_recent_size
        if is_k:
            assert (batch_size * head_num * head_dim) % head_dim == 0
            assert self.block_size == kvcomp_cuda.K_VEC_PER_BLK, "for K, block size must equal VEC_PER_BLK"
        else:
            assert (batch_size * head_num * head_dim) % kvcomp_cuda.V_VEC_PER_BLK == 0, "hidden size must be divisible by VEC_PER_BLK"
            assert self.block_size % kvcomp_cuda.V_VEC_LEN == 0, "block size must be divisible by VEC_LEN"
        self._row_bytes = 2 * batch_size * head_num * head_dim
        self._mask = dims_to_mask(self.quant_dims)
        self._groups_per_block = expected_groups(self.block_size, self.block_size, batch_size, head_num, head_dim, self.quant_dims)
        self._lut: Optional[torch.Tensor] = None       # decode tables of _lut_source, see decode_lut
        self._lut_source: Optional[torch.Tensor] = None
        self._encoded = _Growable()
        self._block_infos = _Growable()
        self._thread_infos = _Growable()
        self._min_ints = _Growable()
        self._scales = _Growable()
        self._tail: Optional[torch.Tensor] = None      # [capacity, B, H, D]; the first _tail_len tokens are the tail
        self._tail_len = 0
        self.max_code_bits = 0           # longest code of the codebook (0 = unknown)
        self.pair_bits = 0             # index width that next to all pairs of symbols fit (kvc_codebook::pair_bits, 0 = none known)
        self.max_tile_bytes = 0            # largest tile payload seen so far (sizes the fused decoders' LDS staging)
        self.max_stream_bytes = 0          # longest lane stream seen so far (sizes the fused decoders' LDS rows)
        self.encode_codebook: Optional[torch.Tensor] = None
        self.decode_codebook: Optional[torch.Tensor] = None
        # node layout of decode_codebook: the reference's 3-byte nodes (include/huffman.h:18-22) while the code fits them
        # (at most 128 nodes, symbols up to 127), else 5-byte nodes; every decoder of this context is told which
        self.tree_format = kvcomp_cuda.TREE_I8
        # what encodes that nobody waited for have left on the device: words 0 - 7 are kvc_encode_async's result words,
        # word 8 counts the payload bytes in _encoded; _enc_pending bounds the bytes the host has not learnt of yet
        self._state: Optional[torch.Tensor] = None
        self._enc_pending = 0
        # Stores that were queued and not yet seen to succeed, oldest first; _verified is the bookkeeping behind the last
        # store that is known to be good.  _probe = (event, stores covered, stream) while the device words are on their way to
        # the host: an encode's own _outcome, or a copy to _host_words (pinned).  Reading them later costs no wait.
        self._unverified: List[_QueuedStore] = []
        self._verified = None
        self._probe = None
        self._host_words: Optional[torch.Tensor] = None
        self._outcome: Optional[_Outcome] = None
        self._trim_after_sync = False
        self.waits = 0                     # how often this context has waited for the device to learn sizes

    def __getstate__(self):
        # (copies and pickles: queued stores are waited for, since a copy cannot share the event and the pinned words that
        # will say what became of them)
        self._sync_sizes()
        return {**self.__dict__, "_probe": None, "_host_words": None, "_outcome": None}

    def _device_state(self) -> torch.Tensor:
        if self._state is None:
            self._state = torch.zeros(16, dtype=torch.int32, device=self.device)
            if self._encoded.used:
                self._state[8] = self._encoded.used
        return self._state

    def _bookkeeping(self):
        return (self._block_infos.used, self._thread_infos.used, self._min_ints.used, self._scales.used, self.compressed_ctx_len)

    def _sync_sizes(self):
        """Learn from the device how many payload bytes the encodes queued so far have produced (waits for them).  If
        one of them failed, every store queued since the last one known to be good is taken back (their tokens return
        to the front of the tail) and the error is raised."""
        if self._enc_pending == 0:
            return
        p = self._probe
        if p is not None and p[1] == len(self._unverified):     # a copy of the device words behind the last store is on its way
            p[0].synchronize()
            if p[0].query() and int(self._arrived_words(p)[1]) == 0:
                self.waits += 1
                self.poll_stores()
                return
        self.waits += 1
        self._behind_the_last_store()
        try:
            _, max_tile, max_stream, _ = kvcomp_cuda.encode_result(self._state[:8], self._encoded.data.numel())
        except KvcompError:
            self._roll_back()
            raise
        self._probe = None
        self._accept(len(self._unverified), int(self._state[8].item()), max_tile, max_stream)

    def _accept(self, n_stores: int, used: int, max_tile: int, max_stream: int):
        """The first n_stores queued stores are done and good; `used` payload bytes lie in _encoded behind them."""
        done, self._unverified = self._unverified[:n_stores], self._unverified[n_stores:]
        self._encoded.used = used
        self._enc_pending = sum(u.worst for u in self._unverified)
        self.max_tile_bytes = max(self.max_tile_bytes, max_tile)
        self.max_stream_bytes = max(self.max_stream_bytes, max_stream)
        if done:
            self._verified = done[-1].books + (used,)
        if self._trim_after_sync and not self._unverified:
            self._trim_after_sync = False
            self._encoded.trim()                               # a byte per symbol was reserved; the stream is a fraction of it

    def _roll_back(self):
        """Back to the last store that is known to be good: the stores queued since then are dropped from the
        bookkeeping, the device's words say so too, and the tokens of those stores return to the front of the tail
        (rows that were not kept -- stores recorded into a graph -- are lost and leave ctx_len).  A store that cannot fail
        is good even if nobody has looked at it yet; where its payload ends is what its last tile says."""
        if self._verified is None:
            return
        good = 0
        while good < len(self._unverified) and self._unverified[good].certain:
            good += 1
        dropped = self._unverified[good:]
        if good:
            books = self._unverified[good - 1].books
            infos = self._block_infos.data[:books[0]].cpu().view(torch.int32)            # {offset, byte_num} per tile
            self.max_tile_bytes = max(self.max_tile_bytes, int((infos[1::2] & 0xffff).max()))
            # thread_infos: the byte of its tile where each lane's stream ends, above three bits
            ends = (self._thread_infos.data[:books[1]].cpu().view(torch.int16).int() & 0xffff).view(-1, 64) >> 3
            self.max_stream_bytes = max(self.max_stream_bytes, int(ends.diff(prepend=ends.new_zeros(len(ends), 1)).max()))
            self._verified = books + ((int(infos[-2]) & 0xffffffff) + (int(infos[-1]) & 0xffff),)
        (self._block_infos.used, self._thread_infos.used, self._min_ints.used, self._scales.used, self.compressed_ctx_len,
         self._encoded.used) = self._verified
        st = self._state
        st[1:5] = 0                                            # no error; the size hints start again from the host's
        st[4] = self._block_infos.used // 8
        st[8] = self._encoded.used
        self._enc_pending = 0
        rows = [u.rows for u in dropped if u.rows is not None]
        self.ctx_len -= sum(u.tokens for u in dropped if u.lost)
        if rows:
            if self._tail_len:
                rows.append(self._tail[:self._tail_len])
            self._tail = torch.cat(rows, dim=0)
            for t in rows:
                _lib.let_go(t)
            self._tail_len = self._tail.shape[0]
        if any(u.codebook for u in dropped):
            self.encode_codebook = self.decode_codebook = self._lut = self._lut_source = None
            self.tree_format, self.max_code_bits, self.pair_bits = kvcomp_cuda.TREE_I8, 0, 0
        self._unverified = []
        self._probe = None

    def _behind_the_last_store(self):
        """Order the current stream behind the last queued store, where that may have been queued on another one: one that found
        the outcome's words taken by a store on a stream of its own."""
        if self._unverified and self._unverified[-1].done is not None:
            torch.cuda.current_stream(self.device).wait_event(self._unverified[-1].done)

    def _issue_probe(self):
        """Ask for a copy of the device words without waiting for it (nothing is asked for while the stream is being
        recorded into a graph, or while an earlier copy is on its way on another stream; one on this stream is replaced
        by the newer one, which arrives after it in the same place and covers more stores)."""
        p = self._probe
        if not self._unverified or (p is not None and p[1] == len(self._unverified)) or torch.cuda.is_current_stream_capturing():
            return
        stream = _lib.stream_of(self._state)
        if p is not None and p[2] != stream:
            return
        if self._host_words is None:
            self._host_words = torch.empty(16, dtype=torch.int32, pin_memory=True)
        self._behind_the_last_store()
        self._host_words.copy_(self._state, non_blocking=True)
        ev = torch.cuda.Event()
        ev.record(torch.cuda.current_stream(self.device))
        self._probe = (ev, len(self._unverified), stream)

    def _ask_outcome(self):
        """The _Outcome that the encode about to be queued is to write, or None (as for _issue_probe, which then asks for a
        copy behind it where that is possible)."""
        if self.device.type != "cuda" or torch.cuda.is_current_stream_capturing():
            return None
        stream = _lib.stream_of(self._state)
        if self._probe is not None and self._probe[2] != stream:
            return None
        if self._outcome is None or (self._outcome.stream != stream and not self._outcome.query()):
            self._outcome = _Outcome()                         # (words that another stream may still write to are left to it)
        return self._outcome

    def _arrived_words(self, probe):
        return probe[0].words if isinstance(probe[0], _Outcome) else self._host_words

    def poll_stores(self):
        """Look, without waiting, at what the stores queued by async_store have left: sizes and size hints are brought
        up to date, and a store that failed on the device is reported here (KvcompError) with the context rolled back to
        the last good store.  Called by store() and by the attention operator; cheap when nothing is outstanding."""
        p = self._probe
        if p is None or torch.cuda.is_current_stream_capturing() or not p[0].query():      # (an event must not be asked for then)
            return
        w = self._arrived_words(p).tolist()
        self._probe = None
        if w[1] != 0:
            self._sync_sizes()                                 # takes the stores back and raises, with the library's message
            return
        self._accept(p[1], w[8], w[2], w[3])
        self._issue_probe()

    def _append_encoded(self, encoded_: torch.Tensor):
        self._sync_sizes()
        self._encoded.append(encoded_)
        if self._state is not None:
            self._state[8] = self._encoded.used

    @property
    def encoded_data(self) -> Optional[torch.Tensor]:
        """The reference's attribute (kvcomp_encode.py:56): the payload so far (waits for queued encodes)."""
        self._sync_sizes()
        return self._encoded.view

    @property
    def buffer(self) -> Optional[torch.Tensor]:
        """The uncompressed most recent tokens [t, B, H, D] (kvcomp_encode.py:61); a view of a preallocated area."""
        return None if self._tail is None else self._tail[:self._tail_len]

    def _tail_append(self, cache: torch.Tensor):
        n = cache.shape[0]
        if self._tail is None or self._tail_len + n > self._tail.shape[0]:
            # what a context keeps between stores is less than block_size + recent_size tokens; room for that plus
            # the tokens being appended (single tokens while decoding), with some slack against re-allocation
            cap = self._tail_len + n + self.block_size + 64
            grown = torch.empty((cap,) + tuple(cache.shape[1:]), dtype=cache.dtype, device=cache.device)
            if self._tail_len:
                grown[:self._tail_len] = self._tail[:self._tail_len]
            _lib.let_go(self._tail)
            self._tail = grown
        row = self._row_bytes
        if n and cache.is_cuda and not _lib.hooked():
            done = _lib.host().append_rows(self._tail, self._tail_len, cache, row)
            if done:
                if done < 0:
                    _lib.check(done)
                if self._tail_len == 0:                              # where views of an earlier tail may lie
                    torch.autograd.graph.increment_version((self._tail,))
                self._tail_len += n
                return
        to, src = self._tail.data_ptr() + self._tail_len * row, cache.data_ptr()
        if (n and (to | src | row) & 15 == 0 and cache.is_cuda and cache.is_contiguous() and
                not (cache.requires_grad or self._tail.requires_grad or _lib.hooked())):
            if self._tail_len == 0:                                  # where views of an earlier tail may lie
                torch.autograd.graph.increment_version((self._tail,))
            kvcomp_cuda.copy_rows(self._tail, to, src, n * row)      # (half the host time of an assignment to a slice)
        elif n:
            self._tail[self._tail_len:self._tail_len + n] = cache
        self._tail_len += n

    def _tail_drop_front(self, n: int):
        rest = self._tail_len - n
        if rest > 0:
            src = self._tail[n:self._tail_len]
            self._tail[:rest] = src.clone() if rest > n else src       # overlapping ranges go through a copy
        self._tail_len = rest

    # the reference's public tensor attributes (kvcomp_encode.py:56-61)
    block_infos = property(lambda self: self._block_infos.view)
    thread_infos = property(lambda self: self._thread_infos.view)
    quant_min_ints = property(lambda self: self._min_ints.view)
    quant_scales = property(lambda self: self._scales.view)

    def _check(self, cache: torch.Tensor):
        assert cache.dtype is torch.float16, "cache must be float16"
        shape = cache.shape
        assert shape[1] == self.batch_size, "batch size mismatch"
        assert shape[2] == self.head_num, "head num mismatch"
        assert shape[3] == self.head_dim, "head dim mismatch"

    def _scratch(self, sizes):
        dev = self.device
        for store, n in ((KVCompCtx.block_infos_buffer, sizes[0]), (KVCompCtx.thread_infos_buffer, sizes[1]),
                         (KVCompCtx.idx_offset_buffer, sizes[2]), (KVCompCtx.pre_alloc_compressed_data_buffer, sizes[3])):
            if dev not in store or store[dev].numel() < n:
                store[dev] = torch.empty(n, dtype=torch.uint8, device=dev)
        return (KVCompCtx.block_infos_buffer[dev], KVCompCtx.thread_infos_buffer[dev],
                KVCompCtx.idx_offset_buffer[dev], KVCompCtx.pre_alloc_compressed_data_buffer[dev])

    # With a codebook in place, whole blocks can go from fp16 to payload in one library call that never
    # materialises the symbols; callers that do not look at store()'s return value ask for it.
    fused_store = True

    def store(self, cache: torch.Tensor, want_symbols: bool = True):
        """kvcomp_encode.py:69-136: append [T_new, B, H, D]; compress the whole blocks that leave the tail.
        Returns the uint8 symbols that were compressed (None if nothing left the tail, or if want_symbols is
        False and they were never written out a byte each)."""
        self._check(cache)
        if self.device is None:
            self.device = cache.device
        assert self.device == cache.device, "device mismatch"
        if self._probe is not None:
            self.poll_stores()
        # cut_tensor_ctx_len_0 (utils/compute.py:59-72): the leading whole blocks of (tail + new tokens) that leave the
        # recent window are compressed, the rest is the new tail.  The blocks are taken from where they lie (the tail,
        # the incoming tensor, or -- when they span both -- a copy of just those tokens), so a long prompt never passes
        # through the tail and the tail stays a few blocks long.  Nothing of the context changes before the encoder
        # has succeeded: a failed store (a symbol without a code, a tile beyond 8191 bytes) leaves it as it was.
        n_new = cache.shape[0]
        n_blocks = blocks_to_compress(self._tail_len + n_new, self.block_size, self.recent_size)
        if n_blocks <= 0:
            self._tail_append(cache)
            self.ctx_len += n_new
            return None
        n_c = n_blocks * self.block_size
        from_tail = min(n_c, self._tail_len)
        if from_tail == 0:
            to_compress = cache[:n_c].contiguous()
        elif from_tail == n_c:
            to_compress = self._tail[:n_c]
        else:
            to_compress = torch.cat([self._tail[:from_tail], cache[:n_c - from_tail]], dim=0)
        sym = self._compress(to_compress, want_symbols)
        if n_c >= self._tail_len:
            rest = cache[n_c - self._tail_len:]
            self._tail_len = 0
            self._tail_append(rest)
        else:
            self._tail_drop_front(n_c)
            self._tail_append(cache)
        self.ctx_len += n_new
        return sym

    def _compress(self, to_compress: torch.Tensor, want_symbols: bool):
        """Quantize + encode whole blocks [n * block_size, B, H, D] and append the stream; returns the symbols on the
        two-step path.  State is only touched after the library calls have succeeded."""
        mask = dims_to_mask(self.quant_dims)
        if (not want_symbols and KVCompCtx.fused_store and self.async_store and self.encode_codebook is not None
                and kvcomp_cuda.store_fused_supported(self.is_k, mask, self.batch_size, self.head_num, self.head_dim)):
            T = to_compress.shape[0]
            capturing = torch.cuda.is_current_stream_capturing()
            large = T > self.ASYNC_KEEP_BLOCKS * self.block_size
            # the rows of a small store are kept until the store is seen to have succeeded (a copy: the caller's tensor
            # and the tail are both overwritten soon); a large one is waited for here, with its rows still in place
            keep = None if (large or capturing) else to_compress.clone()
            self._encode_direct(T, cache=to_compress, mask=mask, tables=self.encode_codebook,
                                table_bytes=self.encode_codebook.numel(), keep=keep, lost_if_dropped=capturing)
            if large and not capturing:
                self._trim_after_sync = True
                self._sync_sizes()
            else:
                self._issue_probe()
            return None
        if (not want_symbols and KVCompCtx.fused_store and self.encode_codebook is not None
                and kvcomp_cuda.store_fused_supported(self.is_k, mask, self.batch_size, self.head_num, self.head_dim)):
            self._store_fused(to_compress, mask)
            return None
        blocked = to_compress.reshape(-1, self.block_size, self.batch_size, self.head_num, self.head_dim)
        if self.encode_codebook is None and self.device_codebook:
            return self._first_chunk(blocked, want_symbols)
        quant_ints, min_ints, quant_scale = quant(blocked, self.quant_dims, self.quant_scale_rel)
        sizes = kvcomp_cuda.calculate_buffer_size(quant_ints, self.is_k, self.head_num, self.head_dim)
        KVCompCtx.buffer_ctx_len[self.device] = to_compress.shape[0]
        bi_buf, ti_buf, idx_buf, payload_buf = self._scratch(sizes)
        codebook = None
        if self.encode_codebook is None:     # first stored chunk defines the codebook (kvcomp_encode.py:99-103)
            counts = kvcomp_cuda.symbol_counts([quant_ints])
            if self.codebook_smoothing:
                counts[:self._smoothed_symbols()] += 1
            codebook = self._host_codebook(counts)
        enc_table = self.encode_codebook if codebook is None else codebook[0].to(self.device)
        fn = kvcomp_cuda.k_entropy_encode_cuda_export if self.is_k else kvcomp_cuda.v_entropy_encode_cuda_export
        encoded_, block_infos_, vec_infos_ = fn(quant_ints, enc_table, bi_buf, ti_buf, idx_buf, payload_buf,
                                                self._encoded.used, self.head_num, self.head_dim)
        if codebook is not None:
            self._set_codebook(*codebook[:2], tree_format=codebook[2])
        self.max_tile_bytes = max(self.max_tile_bytes, kvcomp_cuda.last_encode_max_tile_bytes)
        self.max_stream_bytes = max(self.max_stream_bytes, kvcomp_cuda.last_encode_max_stream_bytes)
        self._append_encoded(encoded_)
        self._block_infos.append(block_infos_)
        self._thread_infos.append(vec_infos_)
        self._min_ints.append(min_ints)
        self._scales.append(quant_scale)
        self.compressed_ctx_len += quant_ints.shape[0] * quant_ints.shape[1]
        return quant_ints

    # The first chunk's codebook comes from counts that the quantizer takes while it writes the symbols; False: from a
    # histogram pass over them, as in the reference.
    device_codebook = True
    # With a codebook in place, store(want_symbols=False) queues the fused quantize + encode and returns without
    # waiting for it: sizes and errors are learnt the next time something asks for them (encoded_data, get_cr, ...),
    # and a store that fails on the device is reported by the next store() or attention call that finds its outcome
    # (poll_stores: no wait), or by whatever waits for sizes: the context is then rolled back to the last good store,
    # with the failed stores' tokens back in the tail.  The caches that models use switch it on, together with
    # codebook_smoothing, which rules out symbols without a code.
    async_store = False
    # stores of up to this many blocks are queued without a wait; longer ones (a second chunk of a prompt) are waited for
    ASYNC_KEEP_BLOCKS = 8
    # a growing payload buffer takes up to this many bytes along of which it is not known yet whether they are payload (a copy
    # of this much takes about as long as a wait)
    COPY_PENDING = 8 << 20

    def _encode_direct(self, T: int, *, tables=None, table_bytes=0, symbols=None, cache=None, mask=0, most_bytes=None, keep=None,
                       lost_if_dropped=False, certain=False, codebook=False, prepared=None, longest_code=0, book=None):
        """Queue one encode whose outputs go straight to their final places in this context's buffers; nothing waits.
        Quantizes `cache` on the fly (fused store) or takes `symbols` whose parameters are in place already.  most_bytes:
        what the payload is known not to exceed; prepared, longest_code: what _prepare_encode returned, the codebook's longest code; book: instead of
        tables, a codebook that is still to be put in place, and where."""
        nb = T // self.block_size
        B, H, D = self.batch_size, self.head_num, self.head_dim
        sizes = kvcomp_cuda.buffer_sizes(T, B * H * D, self.is_k, H, D) if prepared is None else prepared.sizes
        state = self._device_state()
        if not self._unverified:
            self._sync_sizes()                                 # (a no-op unless sizes are outstanding for another reason)
            self._verified = self._bookkeeping() + (self._encoded.used,)
        if prepared is None:
            bi = self._block_infos.reserve(sizes[0], (), torch.uint8, self.device)
            ti = self._thread_infos.reserve(sizes[1], (), torch.uint8, self.device)
            mn = sc = None                                     # (symbols: their parameters are in place)
            if cache is not None:
                gshape = mask_keepdim_shape((nb, self.block_size, B, H, D), self._mask)
                mn = self._min_ints.reserve(nb, gshape[1:], torch.int8, self.device)
                sc = self._scales.reserve(nb, gshape[1:], torch.float16, self.device)
        worst = T * B * H * D if most_bytes is None else most_bytes       # the reference's pre-allocation: a byte per symbol
        if (self._encoded.data is None or
                self._encoded.used + self._enc_pending + worst > self._encoded.data.numel()):
            # growing copies the filled part, or -- while queued stores have yet to say how much that is -- what it can be at most
            if self._probe is not None:
                self.poll_stores()
            if self._enc_pending > self.COPY_PENDING or (self._enc_pending and torch.cuda.is_current_stream_capturing()):
                self._sync_sizes()
            self._encoded.reserve(worst, (), torch.uint8, self.device, self._enc_pending)
        # (a payload whose size is bounded is told so: what the buffer keeps for growing would make tiles look larger than they are)
        room = None if most_bytes is None else self._encoded.used + self._enc_pending + worst
        outcome = self._ask_outcome()
        before = None if outcome is None else (outcome.number, outcome.stream)
        told = None if outcome is None else outcome.ask(_lib.stream_of(state))
        try:
            if book is not None:
                kvcomp_cuda.encode_prepared_book(prepared, *book, self._encoded.data, told, room)
            elif prepared is not None:
                kvcomp_cuda.encode_prepared(prepared, tables, self._encoded.data, told, longest_code, room)
            else:
                kvcomp_cuda.encode_async(self.is_k, batch=B, head_num=H, head_dim=D, tokens=T, encode_tables=tables,
                                         table_bytes=table_bytes, block_infos=bi, thread_infos=ti, encoded=self._encoded.data,
                                         symbols=symbols, cache=cache, quant_mask=mask, eb=self.quant_scale_rel, min_ints=mn, scales=sc,
                                         stream_bytes=state[8:9], result=state[:8], outcome=told, room=room)
        except BaseException:
            if outcome is not None:
                with contextlib.suppress(RuntimeError):        # (the words must not go while a part of the call may write them)
                    torch.cuda.current_stream(self.device).synchronize()
                outcome.refused(*before)
            raise
        self._has_queued(T, sizes, worst, outcome, keep, lost_if_dropped, certain, codebook)

    def _has_queued(self, T: int, sizes, worst: int, outcome, keep=None, lost_if_dropped=False, certain=False, codebook=False):
        """The bookkeeping behind an encode of T tokens that has been queued."""
        nb = T // self.block_size
        self._block_infos.used += sizes[0]
        self._thread_infos.used += sizes[1]
        self._min_ints.used += nb
        self._scales.used += nb
        self._enc_pending += worst
        self.compressed_ctx_len += T
        done = None
        if outcome is None and self.device.type == "cuda" and not torch.cuda.is_current_stream_capturing():
            done = torch.cuda.Event()
            done.record(torch.cuda.current_stream(self.device))
        self._unverified.append(_QueuedStore(T, keep, self._bookkeeping(), worst, lost_if_dropped, certain, codebook, done))
        if outcome is not None:
            self._probe = (outcome, len(self._unverified), outcome.stream)

    def _prepare_encode(self, T: int, symbols: torch.Tensor, packed: bool):
        """For a first store, while the quantizer runs: the buffers of the encode and the launch that needs no codebook."""
        B, H, D = self.batch_size, self.head_num, self.head_dim
        sizes = kvcomp_cuda.buffer_sizes(T, B * H * D, self.is_k, H, D)
        bi = self._block_infos.reserve(sizes[0], (), torch.uint8, self.device)
        ti = self._thread_infos.reserve(sizes[1], (), torch.uint8, self.device)
        state = torch.empty(16, dtype=torch.int32, device=self.device)
        prepared = kvcomp_cuda.encode_prepare(self.is_k, batch=B, head_num=H, head_dim=D, tokens=T, symbols=symbols,
                                              block_infos=bi, thread_infos=ti, state=state, packed=packed)
        self._state = state                                    # (cleared, on this stream)
        self._ask_outcome()
        return prepared

    def _first_chunk(self, blocked: torch.Tensor, want_symbols: bool = True) -> Optional[torch.Tensor]:
        """The first stored chunk: quantized, its codebook built from the symbols just written (kvcomp_encode.py:86-103; the
        one thing that is waited for) and encoded with it.  The counts and the code lengths bound the payload to within a
        byte per lane stream, so the buffer is as large as the stream needs, and with them at hand neither a symbol without
        a code nor too small a buffer is possible; with codes of at most seven bits nor is a tile beyond 8191 bytes, so
        the encode need not be waited for either.  Symbols that nobody asked for go from the quantizer to the encoder two to a
        byte where there are at most sixteen of them, and are not returned."""
        nb, T, device = blocked.shape[0], blocked.shape[0] * self.block_size, self.device
        gshape = mask_keepdim_shape(blocked.shape, self._mask)
        min_ints = self._min_ints.reserve(nb, gshape[1:], torch.int8, device)
        quant_scale = self._scales.reserve(nb, gshape[1:], torch.float16, device)
        prepared = []

        fresh = self._state is None and self._encoded.used == 0
        smoothed = self._smoothed_symbols() if self.codebook_smoothing else 0
        # (just below 1/13, where the library's fp32 bound is 1/13, smoothing gives codes to seventeen symbols: packed ones would
        # always be written again a byte each)
        packed = (not want_symbols and fresh and smoothed <= 16 and
                  kvcomp_cuda.packed_symbols_supported(self.is_k, self._mask, blocked, self.quant_scale_rel))

        native, vectors = None, T * self.batch_size * self.head_num * self.head_dim // (self.head_dim if self.is_k else kvcomp_cuda.V_VEC_LEN)

        def meanwhile(symbols):
            nonlocal native
            if not fresh:
                return None
            prepared.extend((self._prepare_encode(T, symbols, packed), kvcomp_cuda.codebook_room(device)))
            if packed and self.async_store and not self._unverified and not _lib.hooked():
                self._sync_sizes()                             # (as _encode_direct)
                self._verified = self._bookkeeping() + (self._encoded.used,)
                outcome = self._ask_outcome()
                if outcome is not None:
                    native = _NativeFirst(*prepared, vectors, outcome, _lib.stream_of(self._state))
            return native
        quantize = kvcomp_cuda.quant_codebook_packed if packed else kvcomp_cuda.quant_codebook
        try:
            sym, book = quantize(blocked, self._mask, self.quant_scale_rel, min_ints, quant_scale, smoothed, meanwhile)
            if native is not None:
                _lib.check(native.failed)
        except BaseException:
            if native is not None:
                with contextlib.suppress(RuntimeError):        # (as in _encode_direct)
                    torch.cuda.current_stream(device).synchronize()
                native.refused()
            raise
        self.waits += 1
        if native is not None and native.payload is not None:
            enc, dec, lut = kvcomp_cuda.codebook_parts(book, prepared[1])
            self._encoded._hold(native.payload)
            self._has_queued(T, prepared[0].sizes, native.most, native.outcome, certain=True, codebook=True)
            self._issue_probe()
            self._take_book(book, enc, dec, lut)
            return None
        if native is not None:
            native.refused()                                   # (nothing of it has been queued)
        if packed and book.encode_bytes > 16 * 8:              # scales among fp16's smallest numbers: half a byte does not hold these symbols
            sym = quant(blocked, self.quant_dims, self.quant_scale_rel)[0]
            prepared, packed = [], False
        enc, dec, lut = kvcomp_cuda.codebook_parts(book, prepared[1]) if packed else kvcomp_cuda.put_codebook(book, device, *prepared[1:])
        cannot_fail = book.max_code_bits <= 7
        small = T <= self.ASYNC_KEEP_BLOCKS * self.block_size
        queued = self.async_store and (cannot_fail or small)
        self._encode_direct(T, symbols=sym, tables=enc, table_bytes=enc.numel(), most_bytes=book.payload_bits // 8 + vectors + 1,
                            keep=blocked.flatten(0, 1).clone() if queued and not cannot_fail else None, certain=cannot_fail, codebook=True,
                            prepared=prepared[0] if prepared else None, longest_code=book.max_code_bits,
                            book=(book, prepared[1]) if packed else None)
        if queued:
            self._issue_probe()
        else:
            self._sync_sizes()                                 # (a failure leaves the context as it was before the encode)
        self._take_book(book, enc, dec, lut)
        return None if packed else sym

    def _take_book(self, book, enc, dec, lut):
        self.tree_format, self.max_code_bits, self.pair_bits = book.tree_format, book.max_code_bits, book.pair_bits
        self.encode_codebook, self.decode_codebook = enc, dec
        self._lut, self._lut_source = lut, dec

    def _smoothed_symbols(self) -> int:
        return min(256, int(math.ceil(1.0 / self.quant_scale_rel)) + 3)      # symbols 0 .. ceil(1 / eb) + 2

    # The reference derives the one codebook of a stream from its first stored chunk alone, so a symbol that first
    # shows up later has no code (its encoder then emits nothing for it and the stream is corrupt; here the
    # encoder reports an error).  With smoothing, every symbol the error bound allows counts once more than it
    # occurs, so all of them get a code; the codebook then differs from the reference's for the same chunk.
    codebook_smoothing = False

    def _host_codebook(self, counts: torch.Tensor):
        """(encode table, decode tree, tree format) from 256 symbol counts, by the host builder: the reference's int8
        tree where the code fits it, the int16 tree where it does not (more than 64 symbols, or one above 127)."""
        try:
            shift, enc, dec = kvcomp_cuda.build_codebook_from_counts(counts, kvcomp_cuda.TREE_I8)
            fmt = kvcomp_cuda.TREE_I8
        except KvcompError:
            shift, enc, dec = kvcomp_cuda.build_codebook_from_counts(counts, kvcomp_cuda.TREE_I16)
            fmt = kvcomp_cuda.TREE_I16
        assert shift == 0, "shift must be 0"
        return enc, dec, fmt

    def _store_fused(self, to_compress: torch.Tensor, mask: int):
        """fp16 rows -> payload + metadata in one call (kvc_store_fused); same outputs as the two-step path."""
        T = to_compress.shape[0]
        nb = T // self.block_size
        gshape = mask_keepdim_shape((nb, self.block_size, self.batch_size, self.head_num, self.head_dim), mask)
        min_ints = torch.empty(gshape, dtype=torch.int8, device=self.device)
        quant_scale = torch.empty(gshape, dtype=torch.float16, device=self.device)
        sizes = kvcomp_cuda.buffer_sizes(T, self.batch_size * self.head_num * self.head_dim, self.is_k, self.head_num,
                                         self.head_dim)
        KVCompCtx.buffer_ctx_len[self.device] = T
        bi_buf, ti_buf, idx_buf, payload_buf = self._scratch(sizes)
        encoded_, block_infos_, vec_infos_ = kvcomp_cuda.store_fused(
            self.is_k, to_compress, mask, self.quant_scale_rel, self.encode_codebook, min_ints, quant_scale, bi_buf, ti_buf,
            idx_buf, payload_buf, self._encoded.used)
        self.max_tile_bytes = max(self.max_tile_bytes, kvcomp_cuda.last_encode_max_tile_bytes)
        self.max_stream_bytes = max(self.max_stream_bytes, kvcomp_cuda.last_encode_max_stream_bytes)
        self._append_encoded(encoded_)
        self._block_infos.append(block_infos_)
        self._thread_infos.append(vec_infos_)
        self._min_ints.append(min_ints)
        self._scales.append(quant_scale)
        self.compressed_ctx_len += T

    def _assert_ready(self):
        assert self.quant_min_ints is not None, "quant_min_ints is None"
        assert self.quant_scales is not None, "quant_scales is None"
        assert self.encoded_data is not None, "encoded_data is None"
        assert self.block_infos is not None, "huffman_block_info is None"
        assert self.thread_infos is not None, "huffman_thread_info is None"
        assert self.decode_codebook is not None, "decode_codebook is None"

    def get_decode_quant_ints(self) -> Tuple[torch.Tensor, float]:
        """kvcomp_encode.py:168-207: Huffman-decode the whole compressed part back to uint8 symbols."""
        self._assert_ready()
        decoded = torch.empty(self.compressed_ctx_len // self.block_size, self.block_size, self.batch_size,
                              self.head_num, self.head_dim, dtype=torch.uint8, device=self.device)
        fn = kvcomp_cuda.k_entropy_decode_cuda_export if self.is_k else kvcomp_cuda.v_entropy_decode_cuda_export
        t_ms = fn(self.encoded_data, self.block_infos, self.thread_infos, self.decode_codebook, decoded,
                  self.head_num, self.head_dim, self.tree_format)
        return decoded, t_ms

    @property
    def code_hint(self) -> int:
        """kvc_compressed_desc::max_code_bits of this context's codebook."""
        table = self.encode_codebook
        rows = 0 if table is None else table.shape[0]        # eight bytes per symbol
        return self.max_code_bits | self.pair_bits << 12 | (0 if rows == 0 or rows > 64 * 8 else 0x100 if rows > 17 * 8 else 0x300)

    def _build_lut(self):
        """The decode tables of the codebook that has just been put in place, on the stream that put it there: whoever is
        ordered behind that, on whatever stream, finds them built."""
        if self.decode_codebook.is_cuda:
            self._lut = kvcomp_cuda.build_lut(self.decode_codebook, self.tree_format)
            self._lut_source = self.decode_codebook

    def decode_lut(self) -> Optional[torch.Tensor]:
        """The decode tables of this context's codebook (kvc_build_lut); None before the first block has been compressed."""
        if self._lut_source is not self.decode_codebook:
            # a codebook assigned from outside, on a stream that nobody can name: the tables are waited for once, so that
            # other streams may read them.  While the stream is being recorded nothing is built yet: the graph builds tables
            # of its own, and they are not taken for ones that anyone else can use.
            self._lut = kvcomp_cuda.build_lut(self.decode_codebook, self.tree_format)
            if not torch.cuda.is_current_stream_capturing():
                torch.cuda.current_stream(self._lut.device).synchronize()
                self._lut_source = self.decode_codebook
        return self._lut

    def descriptor(self) -> "_lib.CompressedDesc":
        """kvc_compressed_desc of everything held; every call has its own, since the library reads it without the GIL.  Does
        not wait for queued stores: addresses and a bound of the payload are enough for the kernels.  Addresses and sizes
        come straight from the growing arrays, in one go: a tensor view or a ctypes assignment per field costs more host
        time than a short-context step takes on the device."""
        if self._probe is not None:
            self.poll_stores()                             # what queued stores have left, if it has arrived: no wait
        tokens, tail = self.compressed_ctx_len, self._tail_len
        tail_address = self._tail.data_ptr() if tail else 0
        desc = _lib.CompressedDesc()
        if tokens == 0:
            _DESC.pack_into(desc, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, self._mask, 0, 0, 0, 0, tail_address, tail)
            return desc
        lut = self._lut if self._lut_source is self.decode_codebook else self.decode_lut()
        infos, threads, mins, scales, encoded = self._block_infos, self._thread_infos, self._min_ints, self._scales, self._encoded
        # the kernels take the quantization parameters by pointer: they must cover every group of the stream
        groups = tokens // self.block_size * self._groups_per_block
        assert mins.used * mins.row == groups and scales.used * scales.row == groups, \
            "the context holds %d minima and %d scales for %d quantization groups" % (mins.used * mins.row, scales.used * scales.row, groups)
        _DESC.pack_into(desc, 0, lut.data_ptr(), 0, infos.data.data_ptr(), infos.used, threads.data.data_ptr(), threads.used,
                        encoded.data.data_ptr(), min(encoded.used + self._enc_pending, encoded.data.numel()),
                        mins.data.data_ptr(), scales.data.data_ptr(), self._mask,
                        self.max_tile_bytes, self.max_stream_bytes, self.code_hint, tokens, tail_address, tail)
        return desc

    _descriptor = property(descriptor)                     # (as an attribute: another one every time)

    # decode and dequantize in one kernel (no uint8 tensor in between); False = the reference's two steps
    fused_get = True

    def get_only_compressed(self) -> Tuple[torch.Tensor, float]:
        """kvcomp_encode.py:153-166: decode + dequantize the compressed part -> ([ctx_c, B, H, D] fp16, ms)."""
        if KVCompCtx.fused_get:
            self._assert_ready()
            return self._restore(with_tail=False)
        decoded, t_ms = self.get_decode_quant_ints()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        out = dequant(decoded, self.quant_min_ints, self.quant_scales, self.quant_dims)
        end.record()
        end.synchronize()
        return out.flatten(0, 1), t_ms + start.elapsed_time(end)

    def _restore(self, with_tail: bool) -> Tuple[torch.Tensor, float]:
        """The compressed part and (with_tail) the tail behind it, decoded straight into one tensor, and the milliseconds
        that took on the device."""
        desc = self.descriptor()
        tail = desc.tail_tokens if with_tail else 0
        out = torch.empty(desc.tokens + tail, self.batch_size, self.head_num, self.head_dim, dtype=torch.float16, device=self.device)
        t_ms = kvcomp_cuda.restore(self.is_k, desc, self.block_size, out, with_tail)
        return out, t_ms

    def get(self) -> Tuple[torch.Tensor, float]:
        """kvcomp_encode.py:138-151: compressed part followed by the uncompressed tail.  (While nothing has
        been compressed yet the tail is everything; the reference asserts in that state.)"""
        if self.compressed_ctx_len == 0:
            return self.buffer.clone(), 0.0
        if KVCompCtx.fused_get and not (self._tail_len and _lib.recorded(self._tail)):
            self._assert_ready()
            return self._restore(with_tail=True)
        out, t_ms = self.get_only_compressed()
        if self.buffer is not None and self.buffer.shape[0] > 0:
            out = torch.cat([out, self.buffer], dim=0)
        return out, t_ms

    def mat_vec_mul(self, B: torch.Tensor) -> Tuple[torch.Tensor, float]:
        """kvcomp_encode.py:209-280.  K: B = q [B, H, D] -> scores [B, H, ctx_c].  V: B = p [B, H, ctx_c] ->
        [1, B, H, D] (the per-128-token partials summed, as the reference does in PyTorch)."""
        self._assert_ready()
        assert B.dtype == torch.float16, "B must be float16"
        assert len(B.shape) == 3, "B must be 3D tensor"
        assert B.shape[0] == self.batch_size, "batch size mismatch"
        q_heads, tokens, part = B.shape[1], self.compressed_ctx_len, None
        assert q_heads % self.head_num == 0, "head num mismatch"
        if self.is_k:
            assert B.shape[2] == self.head_dim, "head dim mismatch"
            out = torch.empty(self.batch_size, q_heads, tokens, dtype=torch.float16, device=self.device)
        else:
            assert B.shape[2] == tokens, "ctx len mismatch"
            part = torch.empty(tokens // kvcomp_cuda.V_VEC_LEN, self.batch_size, q_heads, self.head_dim, dtype=torch.float16, device=self.device)
            out = torch.empty(1, self.batch_size, q_heads, self.head_dim, dtype=torch.float16, device=self.device)
        t_ms = kvcomp_cuda.mat_vec_mul(self.is_k, self.descriptor(), B.contiguous(), part, out, self.head_num, self.head_dim)
        return out, t_ms

    def build_codebook(self, tensors: List[torch.Tensor]):
        """kvcomp_encode.py:282-306: one codebook from the quantized whole blocks of sample tensors."""
        assert len(tensors) > 0, "tensors must not be empty"
        device_ = tensors[0].device
        sym = []
        for cache in tensors:
            self._check(cache)
            assert device_ == cache.device, "device mismatch"
            blocked_len = cache.shape[0] // self.block_size * self.block_size
            blocked = cache[:blocked_len].reshape(-1, self.block_size, self.batch_size, self.head_num, self.head_dim)
            sym.append(quant(blocked, self.quant_dims, self.quant_scale_rel)[0])
        enc, dec, fmt = self._host_codebook(kvcomp_cuda.symbol_counts(sym))
        if self.device is None:
            self.device = device_
            KVCompCtx.buffer_ctx_len[self.device] = 0
        self._set_codebook(enc, dec, tree_format=fmt)

    def _set_codebook(self, enc: torch.Tensor, dec: torch.Tensor, tree_format: int = kvcomp_cuda.TREE_I8):
        """enc / dec: CPU byte tensors from kvcomp_cuda.build_codebook."""
        self.tree_format, self.pair_bits = tree_format, 0
        lengths = enc.view(torch.int32)[1::2]
        self.max_code_bits = int(lengths.max())      # sizes the fused decoders' table in LDS
        self.encode_codebook = enc.to(self.device)
        self.decode_codebook = dec.to(self.device)
        self._build_lut()

    @property
    def shape(self):
        return torch.Size([self.compressed_ctx_len, self.batch_size, self.head_num, self.head_dim])

    def held_bytes(self) -> int:
        """Device memory this context holds, from the capacities of its buffers (not just their filled parts)."""
        n = 0 if self._tail is None else self._tail.numel() * self._tail.element_size()
        for g in (self._encoded, self._block_infos, self._thread_infos, self._min_ints, self._scales):
            if g.data is not None:
                n += g.data.numel() * g.data.element_size()
        for t in (self.encode_codebook, self.decode_codebook):
            if t is not None:
                n += t.numel()
        return n

    def compressed_bytes(self) -> int:
        """Denominator of get_cr (kvcomp_encode.py:318-324): everything a fused kernel has to read."""
        return (self.block_infos.numel() + self.thread_infos.numel() + self.encoded_data.numel() +
                self.quant_min_ints.numel() + self.quant_scales.numel() * 2)

    def get_cr(self):
        """kvcomp_encode.py:317-326"""
        original = 2 * self.batch_size * self.compressed_ctx_len * self.head_num * self.head_dim
        return original / self.compressed_bytes()
