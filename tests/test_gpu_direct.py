"""Unpartitioned joins (one launch of host-planned tiles: the hash join of a small build side and
the block nested-loop join) at the edges of their tables and tiles, and the deterministic order
when a skewed join has more tiles than the host estimated."""
import ctypes

import numpy as np
import pytest

import eating_one_amd as eo
from eating_one_amd import DeviceArray, _abi
from common import brute_join, same_multiset

pytestmark = pytest.mark.gpu


def _relations(nR, nS, keys):
    rng = np.random.default_rng(nR * 31 + nS)
    R = np.stack([rng.integers(-keys // 2, keys // 2 + 1, nR), np.arange(nR)], 1).astype(np.int32)
    S = np.stack([rng.integers(-keys // 2, keys // 2 + 1, nS), np.arange(nS) + 7], 1).astype(np.int32)
    return R, S


@pytest.mark.parametrize("lds", [0, 4096, 8192, 16384])
@pytest.mark.parametrize("nR,nS", [(1, 1), (2, 2047), (4352, 2049), (4353, 4096), (8704, 4097), (8705, 3),
                                   (17408, 8192), (17409, 8193), (52225, 20001)])
def test_direct_tiles_equal_brute_force(ctx, lds, nR, nS):
    R, S = _relations(nR, nS, max(nR, 4))
    want = brute_join(R, S)
    kw = dict(radix_bits=-1, lds_tuples=lds)
    assert same_multiset(ctx.hash_join(R, S, **kw), want)
    assert ctx.hash_join(R, S, count_only=True, **kw) == len(want)
    outer = ctx.hash_join(R, S, left_outer=True, **kw)
    null = outer[:, 0] == _abi.EO_NULL_PAYLOAD
    assert same_multiset(outer[~null], want)
    assert np.array_equal(np.sort(outer[null, 1]), np.sort(S[~np.isin(S[:, 0], R[:, 0]), 1]))
    if lds == 0:
        assert same_multiset(ctx.nlj_join(R, S), want)
        assert ctx.nlj_join(R, S, count_only=True) == len(want)
        rows = ctx.nlj_join(R, S, result16=True)
        assert same_multiset(rows[:, [0, 2]], want) and np.array_equal(rows[:, 1], rows[:, 3])


def test_direct_tiles_span_override_and_overflow(ctx):
    """S spans from the caller, and an output too small for the rows: the count is whole and the
    next call on the context starts from clean result words."""
    R, S = _relations(9000, 70000, 6000)
    want = brute_join(R, S)
    assert same_multiset(ctx.hash_join(R, S, radix_bits=-1, s_tile=8192), want)
    for fn in (ctx.lib.eo_hash_join, ctx.lib.eo_nlj_join):
        o, n = ctx.opts(), ctypes.c_uint64()
        out = np.full((100, 2), -5, dtype=np.int32)
        st = fn(ctx.handle, R.ctypes.data, len(R), S.ctypes.data, len(S), out.ctypes.data, 90, ctypes.byref(n),
                ctypes.byref(o))
        assert st == _abi.EO_ECAPACITY and n.value == len(want)
        assert (out[90:] == -5).all()
        assert ctx.hash_join(R, S, count_only=True) == len(want)


def test_deterministic_join_with_more_tiles_than_estimated(ctx):
    """Every key in one of 64 partitions: 35 R chunks by 123 S spans there, far above the estimate
    the count pass starts from."""
    rng = np.random.default_rng(8)
    nR, nS = 300_000, 1_000_000
    R = np.stack([rng.permutation(nR) << 6, np.arange(nR)], 1).astype(np.int32)
    S = np.stack([rng.integers(0, 2 * nR, nS) << 6, np.arange(nS)], 1).astype(np.int32)
    kw = dict(radix_bits=6, passes=1, lds_tuples=8192, s_tile=8192)
    hit = S[:, 0] >> 6 < nR
    for outer in (False, True):
        a = ctx.hash_join(R, S, deterministic=True, left_outer=outer, **kw)
        assert np.array_equal(a, ctx.hash_join(R, S, deterministic=True, left_outer=outer, **kw))
        inner = a[a[:, 0] != _abi.EO_NULL_PAYLOAD]
        assert np.array_equal(np.sort(inner[:, 1]), np.flatnonzero(hit))
        assert np.array_equal(R[inner[:, 0], 0], S[inner[:, 1], 0])
        assert len(a) - len(inner) == (np.count_nonzero(~hit) if outer else 0)


@pytest.mark.parametrize("bits,deterministic", [(1, True), (-1, True), (1, False)])
def test_too_many_tiles_are_refused(ctx, bits, deterministic):
    """All keys in two partitions: 2^32 and more tiles of 8704 x 8192 tuples, whose 32-bit numbers
    wrap.  The join is refused before a tile is probed, and the next one is answered."""
    n, chunk = 800_000_000, 1 << 20
    keys = np.zeros((chunk, 2), dtype=np.int32)
    keys[1::2, 0] = 1
    with eo.Context(0) as c:  # (its scratch is 26 GB)
        rel = DeviceArray(c, 8 * n)
        assert c.lib.eo_copy_h2d(c.handle, rel.ptr, keys.ctypes.data, 8 * chunk) == _abi.EO_OK
        have = chunk
        while have < n:
            k = min(have, n - have)
            assert c.lib.eo_copy_d2d(c.handle, rel.ptr + 8 * have, rel.ptr, 8 * k) == _abi.EO_OK
            have += k
        o = c.opts(where=_abi.EO_DEVICE, radix_bits=bits, lds_tuples=8192, s_tile=8192, deterministic=deterministic)
        cnt = ctypes.c_uint64()
        st = c.lib.eo_hash_join(c.handle, rel.ptr, n, rel.ptr, n, None, 0, ctypes.byref(cnt), ctypes.byref(o))
        assert st == _abi.EO_EINTERNAL
        R, S = _relations(3000, 9000, 2000)
        assert same_multiset(c.hash_join(R, S, deterministic=deterministic), brute_join(R, S))
        rel.close()


def _check_outer(join, R, S, **kw):
    want = brute_join(R, S)
    absent = S[~np.isin(S[:, 0], R[:, 0])]
    rows = join(R, S, left_outer=True, **kw)
    null = rows[:, 0] == _abi.EO_NULL_PAYLOAD
    assert same_multiset(rows[~null], want)
    assert np.array_equal(np.sort(rows[null, 1]), np.sort(absent[:, 1]))
    assert join(R, S, left_outer=True, count_only=True, **kw) == len(want) + len(absent)


@pytest.mark.parametrize("nR,nS", [(200_003, 1), (200_003, 63), (1 << 20, 1000), (70_001, 8193), (17409, 40_000)])
def test_outer_joins_of_a_large_build_side(ctx, nR, nS):
    """The R chunks of an unpartitioned left outer join run beside each other and mark what they
    match; the null rows follow."""
    R, S = _relations(nR, nS, 2 * nR)
    _check_outer(ctx.nlj_join, R, S)
    _check_outer(ctx.hash_join, R, S, radix_bits=-1)
    _check_outer(ctx.hash_join, R, S, radix_bits=-1, lds_tuples=4096)


@pytest.mark.parametrize("lds", [8192, 16384])
@pytest.mark.parametrize("flags", [0, _abi.EO_F_EXACT_PARTITIONS])
def test_outer_joins_of_one_large_partition(ctx, lds, flags):
    """R in one of 32 partitions, several tables and S spans there: the last chunk of a span writes
    its null rows; beside it partitions without R."""
    rng = np.random.default_rng(lds + flags)
    nR, nS = 60_000, 100_003
    R = np.stack([rng.integers(0, nR, nR) << 5, np.arange(nR)], 1).astype(np.int32)
    keys = rng.integers(0, 2 * nR, nS)
    S = np.stack([np.where(rng.random(nS) < 0.7, keys << 5, keys), np.arange(nS)], 1).astype(np.int32)
    _check_outer(ctx.hash_join, R, S, radix_bits=5, passes=1, lds_tuples=lds, s_tile=8192, flags=flags)


@pytest.mark.parametrize("nR,nS,lds", [(1000, 4000, 4096), (4353, 70_000, 4096), (1 << 16, 1 << 20, 16384)])
def test_stats_name_the_table_of_an_unpartitioned_join(ctx, nR, nS, lds):
    """The table that the time model chose, whichever the partitioned plan had: one with fewer
    tuples than the build side is several chunks of it."""
    R, S = _relations(nR, nS, nR)
    st = eo.JoinStats()
    ctx.hash_join(R, S, stats=st)
    assert st.radix_bits == 0 and st.lds_tuples == lds
    table = {4096: 4352, 8192: 8704, 16384: 17408}[lds]
    assert st.tiles % -(-nR // table) == 0
