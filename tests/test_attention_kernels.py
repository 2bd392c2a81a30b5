"""Which kernels decode attention takes a cache with: kvc_attention_kernels answers from the descriptors alone."""
import ctypes as C

import pytest

from kvcomp_amd import _lib

TWO_KERNELS, JOINT, WAVES = range(3)                   # KvcAttendRoute
COLUMNS, BYTES, LONG, PACKED, FMA = 0, 1, 2, 3, 4      # KVC_BOOK_*: columns with word entries, with byte entries, long codes, packed; none
BYTE_SYMBOLS = 0x300


def _desc(is_k, tokens, B, H, D, bits, mean, longest, pair_bits=0, symbols=BYTE_SYMBOLS):
    """mean: bytes of a stream; longest: of the longest one, 0 = not known"""
    tiles = tokens // 64 * B * H if is_k else tokens // 128 * B * H * D // 64
    return _lib.CompressedDesc(tokens=tokens, encoded_bytes=tiles * 64 * mean, max_tile_bytes=int(64 * mean * 1.05), max_stream_bytes=longest,
                               max_code_bits=bits | symbols | pair_bits << 12, quant_mask=1 if is_k else 0xE)


def _asked(B, H, rep, D, tokens, k=(7, 52, 59), v=(7, 32, 39), **kw):
    f = C.CDLL(_lib.LIB_PATH).kvc_attention_kernels
    f.argtypes = [C.POINTER(_lib.CompressedDesc)] * 2 + [C.c_int64] * 4
    _lib.lib()
    return f(C.byref(_desc(True, tokens, B, H, D, *k, **kw)), C.byref(_desc(False, tokens, B, H, D, *v, **kw)), B, H, H * rep, D)


def _kernels(*args, **kw):
    got = _asked(*args, **kw)
    return got & 15, got >> 4 & 15


def _route(*args, **kw):
    return _asked(*args, **kw) >> 8


@pytest.mark.parametrize("rep,D,first", [(1, 128, 2560), (2, 128, 2560), (2, 72, 2560), (4, 128, 2560), (4, 96, 2560), (8, 128, 2560), (8, 72, 2560)])
def test_columns_begin_where_they_pay(rep, D, first):
    """A wave of a small cache waits for its one tile, which the lanes' own loads make longer."""
    v = PACKED if rep == 8 else BYTES
    assert _kernels(1, 8, rep, D, (first // 8 - 2) * 64) == (PACKED, v)
    assert _kernels(1, 8, rep, D, first // 8 * 64) == (BYTES, v)


@pytest.mark.parametrize("rep,D", [(1, 96), (1, 72), (1, 64), (4, 72), (4, 64)])
def test_short_streams_lie_in_columns_from_the_first_tile(rep, D):
    for tokens in (128, 1024, 16384):
        assert _kernels(1, 8, rep, D, tokens, k=(7, 52 * D // 128, 59 * D // 128)) == (BYTES, BYTES)


@pytest.mark.parametrize("rep", [1, 2, 4])
def test_shorter_codes_and_products_that_are_not_rounded(rep):
    short = dict(k=(5, 38, 44), v=(5, 30, 36))
    assert _kernels(1, 8, rep, 128, 64 * 510, **short) == (PACKED, COLUMNS)
    assert _kernels(1, 8, rep, 128, 64 * 512, **short) == (COLUMNS, COLUMNS)
    assert _kernels(1, 8, rep, 128, 64 * 382, **short) == (PACKED, PACKED)
    was = _lib.set_option("fused_rounded", 0)
    try:
        assert _kernels(1, 8, rep, 128, 64 * 2046) == (PACKED, COLUMNS) and _kernels(1, 8, rep, 128, 64 * 2048) == (COLUMNS, COLUMNS)
        assert _kernels(1, 8, rep, 128, 64 * 510) == (PACKED, PACKED)
    finally:
        _lib.set_option("fused_rounded", was)


@pytest.mark.parametrize("rep,D", [(1, 128), (1, 96), (2, 128), (4, 128), (4, 96), (8, 128)])
def test_one_long_stream_does_not_size_every_waves_lds(rep, D):
    """A single token whose symbols are all rare: 112 bytes where the others have some 50."""
    v = PACKED if rep == 8 else BYTES
    even = dict(k=(7, 52 * D // 128, 59 * D // 128), v=(7, 32, 40))
    assert _kernels(4, 8, rep, D, 32768, **even) == (BYTES, v)
    odd = (7, 52 * D // 128, 112)
    assert _kernels(4, 8, rep, D, 32768, k=odd, v=even["v"])[0] == PACKED
    assert _kernels(4, 8, rep, D, 32768, k=even["k"], v=(7, 32, 112)) == (BYTES, PACKED)


@pytest.mark.parametrize("rep", [1, 2, 4])
def test_wider_entries_of_long_codes_keep_more_workgroups(rep):
    """Codes of 7 bits of symbols beyond 16, K of an error bound of 0.05: streams of 76 bytes leave five workgroups, of 44 six and more."""
    assert _kernels(4, 8, rep, 128, 16384, k=(7, 70, 76), symbols=0x100)[0] == PACKED
    assert _kernels(4, 8, rep, 72, 16384, k=(7, 39, 44), symbols=0x100)[0] == COLUMNS
    assert _kernels(4, 8, rep, 128, 16384, k=(7, 52, 67))[0] == BYTES


def test_a_stream_hint_that_is_not_there():
    """The tile's bytes decide then, as they are known or near their mean; a single stream would not be."""
    assert _kernels(4, 8, 1, 128, 32768, k=(7, 52, 0), v=(7, 32, 0)) == (PACKED, PACKED)


def test_a_layout_that_is_asked_for():
    for value, want in ((0, PACKED), (1, PACKED), (2, BYTES)):
        was = _lib.set_option("fused_skew", value)
        try:
            assert _kernels(1, 8, 2, 128, 512) == (want, want) and _kernels(4, 8, 2, 128, 32768) == (want, want)
            assert _kernels(1, 8, 2, 128, 512, k=(9, 52, 59), v=(9, 32, 39)) == (LONG, LONG)
        finally:
            _lib.set_option("fused_skew", was)


def test_other_codebooks():
    assert _kernels(4, 8, 2, 128, 32768, k=(9, 52, 59), v=(12, 60, 70)) == (LONG, LONG)
    assert _kernels(4, 8, 2, 128, 32768, k=(9, 52, 59), v=(12, 60, 70), symbols=0) == (FMA, FMA)      # an alphabet of any size
    assert _kernels(4, 8, 2, 128, 32768, symbols=0x100) == (COLUMNS, COLUMNS)
    assert _kernels(4, 8, 8, 128, 32768, symbols=0x100) == (PACKED, PACKED)
    assert _kernels(4, 8, 1, 96, 32768, k=(6, 42, 47), v=(6, 20, 24), pair_bits=7) == (BYTES, COLUMNS)


@pytest.mark.parametrize("rep,joint_up_to", [(1, 1536), (2, 1536), (4, 2048), (8, 3072)])
def test_a_wave_per_group_from_1536_groups_on(rep, joint_up_to):
    assert _route(8, 32, rep, 128, 128 * 6) == JOINT
    assert _route(8, 32, rep, 128, 128 * 7) == WAVES and _route(8, 32, rep, 128, 128 * 32) == WAVES
    # not its codes, its head size, its entries: a workgroup per group up to its own line, then two kernels
    for other in (dict(k=(5, 38, 44)), dict(v=(5, 30, 36)), dict(symbols=0x100), dict(pair_bits=7)):
        assert _route(8, 32, rep, 128, 128 * 7, **other) == (JOINT if 256 * 7 <= joint_up_to else TWO_KERNELS)
        assert _route(8, 32, rep, 128, 128 * 13, **other) == TWO_KERNELS
    assert _route(8, 32, rep, 64, 128 * 7) == (JOINT if 256 * 7 <= joint_up_to else TWO_KERNELS)


# K's and V's longest streams, the most groups (of 256 heads) that waves take with the workgroups these leave to a compute unit, what is
# taken behind those; 0: their LDS does not fit
@pytest.mark.parametrize("rep,k_longest,v_longest,most,behind", [
    (1, 59, 39, 99, WAVES), (1, 71, 39, 12, TWO_KERNELS), (1, 112, 39, 0, TWO_KERNELS), (1, 59, 112, 0, TWO_KERNELS), (2, 71, 39, 12, TWO_KERNELS),
    (4, 83, 39, 99, WAVES), (4, 95, 39, 8, TWO_KERNELS), (4, 112, 39, 0, TWO_KERNELS), (4, 59, 112, 0, TWO_KERNELS),
    (8, 71, 39, 99, WAVES), (8, 63, 73, 8, WAVES), (8, 63, 75, 0, TWO_KERNELS), (8, 112, 39, 0, TWO_KERNELS), (8, 59, 112, 0, TWO_KERNELS)])
def test_long_streams_leave_caches_to_the_kernels_that_took_them(rep, k_longest, v_longest, most, behind):
    joint = 1536 // 256 if rep <= 2 else 2048 // 256 if rep == 4 else 3072 // 256
    for groups in (7, 8, 9, 11, 12, 13, 32):             # a workgroup's four waves with groups of two heads, or of one
        want = WAVES if groups <= most else JOINT if groups <= joint else behind
        assert _route(8, 32, rep, 128, 128 * groups, k=(7, 52, k_longest), v=(7, 32, v_longest)) == want, groups
        was = _lib.set_option("attention_joint", 0)
        try:
            assert _route(8, 32, rep, 128, 128 * groups, k=(7, 52, k_longest), v=(7, 32, v_longest)) == TWO_KERNELS
        finally:
            _lib.set_option("attention_joint", was)


def test_two_heads_to_a_workgroup_only_where_they_fit():
    """Eight query heads, V's streams of 18 words: the columns of one head fit 64 KiB, those of two do not."""
    was = _lib.set_option("attention_joint", 2)
    try:
        for groups in (7, 8, 9):
            assert _route(8, 64, 8, 128, 128 * groups, k=(7, 52, 59), v=(7, 32, 69)) == WAVES
            assert _route(8, 64, 8, 128, 128 * groups, k=(7, 52, 59), v=(7, 32, 86)) == TWO_KERNELS
    finally:
        _lib.set_option("attention_joint", was)


def test_launches_that_are_asked_for():
    for value, want in ((0, TWO_KERNELS), (1, JOINT), (2, WAVES)):
        was = _lib.set_option("attention_joint", value)
        try:
            assert _route(1, 2, 2, 128, 384) == want and _route(8, 32, 2, 128, 4096) == want
        finally:
            _lib.set_option("attention_joint", was)
