"""GPU parity of the resident indexes (hash, sorted, learned) through the C ABI.

Oracles: joins/CPU_JOIN/inner_cpu (hash index) and joins/CPU_JOIN/sortIndex_cpu
(sorted index) restated in oracle/cpu_join.c; the learned model is checked probe
by probe against the plain binary search of the same index.
"""
import ctypes

import numpy as np
import pytest

import oracle
from eating_one_amd import _abi, gen
from common import brute_join, join_count_closed_form, same_multiset

pytestmark = pytest.mark.gpu


def test_hidx_c3_full(ctx):
    R, S = gen.c3()
    ix = ctx.hidx_build(R)
    try:
        got = ix.join(S)
        assert len(got) == join_count_closed_form(R, S)
        assert same_multiset(got, oracle.hidx_join(R, S, nbuckets=1 << 16))
        assert ix.join(S, count_only=True) == len(got)
    finally:
        ix.free()


@pytest.mark.parametrize("learned", [False, True])
def test_sidx_c3_full(ctx, learned):
    R, S = gen.c3()
    ix = ctx.sidx_build(R, learned=learned)
    try:
        got = ix.join(S)
        assert same_multiset(got, oracle.sidx_join(R, S))
        keys, pays = ix.export()
        ref = oracle.sidx_build(R)
        assert np.array_equal(keys, ref[:, 0])                  # sorted keys exactly
        assert np.array_equal(np.sort(R[ref[:, 1], 1]), np.sort(pays))
        # per key, the payload multiset matches the oracle's {val, adr} index
        o1 = np.lexsort((pays, keys))
        o2 = np.lexsort((R[ref[:, 1], 1], ref[:, 0]))
        assert np.array_equal(pays[o1], R[ref[:, 1], 1][o2])
    finally:
        ix.free()


def test_index_edge_cases(ctx):
    e = np.empty((0, 2), dtype=np.int32)
    one = np.array([[5, 9]], dtype=np.int32)
    R = np.array([[-(1 << 31), 0], [(1 << 31) - 1, 1], [0, 2], [-1, 3], [-1, 4]], dtype=np.int32)
    S = np.array([[(1 << 31) - 1, 0], [-(1 << 31), 1], [-1, 2], [7, 3]], dtype=np.int32)
    for build in (lambda r: ctx.hidx_build(r), lambda r: ctx.sidx_build(r), lambda r: ctx.sidx_build(r, learned=True)):
        ix = build(e)
        assert len(ix.join(one)) == 0
        ix.free()
        ix = build(one)
        assert len(ix.join(e)) == 0
        assert same_multiset(ix.join(one), np.array([[9, 9]]))
        ix.free()
        ix = build(R)
        assert same_multiset(ix.join(S), brute_join(R, S))
        ix.free()


@pytest.mark.parametrize("seed,nR,nS,kr", [(1, 5000, 7000, 300), (2, 100000, 50000, 1 << 20), (3, 70001, 3, 10)])
def test_indexes_random(ctx, seed, nR, nS, kr):
    R, S = gen.uniform(seed, nR, nS, kr, lo=-(kr // 2))
    want = brute_join(R, S)
    for ix in (ctx.hidx_build(R), ctx.sidx_build(R), ctx.sidx_build(R, learned=True)):
        try:
            assert same_multiset(ix.join(S), want)
        finally:
            ix.free()


def _check_learned(ctx, R, S):
    ix = ctx.sidx_build(R, learned=True)
    try:
        info = ix.info()
        assert info["learned"] and info["leaves"] == 4096
        keys, _ = ix.export()
        lb_bin = ix.lookup(S, _abi.EO_LOOKUP_BINARY)
        lb_lrn = ix.lookup(S, _abi.EO_LOOKUP_LEARNED)
        want = np.searchsorted(keys, S[:, 0], side="left").astype(np.uint64)
        assert np.array_equal(lb_bin, want), "binary search differs from numpy's lower bound"
        present = np.isin(S[:, 0], keys)
        assert np.array_equal(lb_lrn[present], lb_bin[present]), "learned position differs from binary search"
        # absent keys: the learned window holds no equal key
        pos = np.minimum(lb_lrn[~present], len(keys) - 1).astype(np.int64)
        assert not np.any(keys[pos] == S[~present, 0])
        assert same_multiset(ix.join(S), ix.join(S, binary_search=True))
        return info
    finally:
        ix.free()


def test_learned_index_c4_shape(ctx):
    R, S = gen.c4(nR=1 << 21, nS=1 << 22)
    info = _check_learned(ctx, R, S)
    assert info["max_err"] < 1 << 16


def test_learned_index_duplicates_and_uniform(ctx):
    R, S = gen.uniform(5, 1 << 20, 1 << 20, 1 << 18)
    _check_learned(ctx, R, S)


@pytest.mark.parametrize("kind", ["hash", "sorted", "learned"])
def test_index_join_fused_and_deterministic(ctx, kind):
    """Default one-pass index join (atomic output reservation) vs count/scan/write."""
    import ctypes
    from eating_one_amd import _abi
    R, S = gen.c3(seed=77, nR=50000, nS=80000, key_range=20000)
    ix = ctx.hidx_build(R) if kind == "hash" else ctx.sidx_build(R, learned=(kind == "learned"))
    want = oracle.hash_join(R, S, nparts=1 << 10)
    fused = ix.join(S)
    d1 = ix.join(S, deterministic=True)
    d2 = ix.join(S, deterministic=True)
    assert same_multiset(fused, want) and same_multiset(d1, want)
    assert np.array_equal(d1, d2)
    assert ix.join(S, count_only=True) == len(want)
    out = np.empty((len(want) - 5, 2), dtype=np.int32)
    n = ctypes.c_uint64()
    o = ctx.opts()
    st = ctx.lib.eo_index_join(ctx.handle, ix.handle, S.ctypes.data, len(S), out.ctypes.data, len(want) - 5,
                               ctypes.byref(n), ctypes.byref(o))
    assert st == _abi.EO_ECAPACITY and n.value == len(want)
    ix.free()


def test_sidx_import_from_reference_index_file(ctx, tmp_path):
    """A BUCKET index file read from disk gives the same index as building it on the device."""
    import eating_one_amd as eo
    R, S = gen.c3(seed=81, nR=70000, nS=90000, key_range=30000)
    bucket = R[np.argsort(R[:, 0], kind="stable")]
    path = tmp_path / "index"
    eo.write_ref_index(str(path), bucket)
    for learned in (False, True):
        imp = ctx.sidx_import(eo.read_ref_index(str(path)), learned=learned)
        built = ctx.sidx_build(R, learned=learned)
        k1, p1 = imp.export()
        k2, p2 = built.export()
        assert np.array_equal(k1, k2) and np.array_equal(k1, bucket[:, 0])
        assert same_multiset(imp.join(S), oracle.hash_join(R, S, nparts=1 << 10))
        if learned:
            assert imp.info()["max_err"] == built.info()["max_err"]
        imp.free()
        built.free()
    with pytest.raises(eo.EOError):
        ctx.sidx_import(R)  # not sorted


@pytest.mark.parametrize("nR", [1, 15, 16, 17, 512, 65536, 65537, 131073, 2097152, 2097153])
@pytest.mark.parametrize("dup", [1, 5, 40])
def test_sorted_index_directory_edges(ctx, nR, dup):
    """Sizes at the edges of the directory's lines and levels (16 entries and 32 keys a line, a
    top level of 4096 keys), runs of equal keys within, at the end of and across lines, probes
    below, between, equal to and above every key, and the key that pads the last line."""
    rng = np.random.default_rng(nR * 64 + dup)
    top = (1 << 31) - 1
    keys = np.repeat(np.arange((nR + dup - 1) // dup, dtype=np.int64) * 3 - nR, dup)[:nR]
    if nR > 15:
        keys[-(nR % 7 + 1):] = top  # the padding's key, also as a real one
    order = rng.permutation(nR)
    R = np.stack([keys[order], order], 1).astype(np.int32)
    probes = np.concatenate([keys[rng.integers(0, nR, 3000)], keys[rng.integers(0, nR, 500)] - 1,
                             [keys[0] - 5, keys[-1], min(keys[-1] + 1, top), top, -top - 1]])
    S = np.stack([probes, np.arange(len(probes))], 1).astype(np.int32)
    want = brute_join(R, S)
    for learned in (False, True):
        ix = ctx.sidx_build(R, learned=learned)
        try:
            pos = ix.lookup(S, _abi.EO_LOOKUP_BINARY)
            assert np.array_equal(pos, np.searchsorted(keys, S[:, 0], side="left").astype(np.uint64))
            assert same_multiset(ix.join(S), want)
            assert same_multiset(ix.join(S, deterministic=True), want)
        finally:
            ix.free()


@pytest.mark.parametrize("nS", [255, 257, (1 << 20) - 1, (1 << 20) + 1, (1 << 20) + 2049])
def test_index_join_probe_tiles(ctx, nS):
    """Probe counts at the edges of the tiles and of the choice between them."""
    R, S = gen.c3(seed=nS, nR=50000, nS=nS, key_range=200000)
    want = brute_join(R, S)
    for ix in (ctx.hidx_build(R), ctx.sidx_build(R)):
        try:
            assert same_multiset(ix.join(S), want)
            outer = ix.join(S, left_outer=True)
            null = outer[:, 0] == _abi.EO_NULL_PAYLOAD
            assert same_multiset(outer[~null], want)
            assert np.array_equal(np.sort(outer[null, 1]), np.flatnonzero(~np.isin(S[:, 0], R[:, 0])))
        finally:
            ix.free()


def test_index_memory_kept_for_the_next_build(ctx):
    """A freed index's block serves the next one of its size, not a much smaller one, while other
    indexes live: each keeps its own rows."""
    rng = np.random.default_rng(77)
    live = []
    for i, n in enumerate([50_000, 49_000, 50_000, 3_000, 50_001, 26_000]):
        R = np.stack([rng.integers(0, n, n), np.arange(n) + 10 ** 6 * i], 1).astype(np.int32)
        S = np.stack([rng.integers(0, 2 * n, n // 2), np.arange(n // 2)], 1).astype(np.int32)
        ix = ctx.hidx_build(R) if i % 2 else ctx.sidx_build(R)
        live.append((ix, S, brute_join(R, S)))
        if i in (1, 3):
            live.pop(0)[0].free()
        for other, S2, want in live:
            assert same_multiset(other.join(S2), want)
    for other, _, _ in live:
        other.free()


def test_index_info_counts_the_block_it_holds(ctx):
    """An index in a larger block kept from a freed one reports that block."""
    big = np.stack([np.arange(60_000), np.arange(60_000)], 1).astype(np.int32)
    ix = ctx.sidx_build(big)
    held = ix.info()["bytes"]
    ix.free()
    ix = ctx.sidx_build(big[:40_000])
    assert ix.info()["bytes"] == held
    ix.free()


def test_learned_lookups_come_from_the_model(ctx):
    """A lookup that the model predicts wrongly is answered wrongly: with every leaf's intercept
    moved, present keys are no longer found where the plain search finds them."""
    n = 100_000
    rng = np.random.default_rng(5)
    keys = np.unique(rng.integers(0, 2 ** 31 - 1, n)).astype(np.int32)
    R = np.stack([keys, np.arange(len(keys))], 1).astype(np.int32)
    ix = ctx.sidx_build(R, learned=True)
    binary = ix.lookup(R, _abi.EO_LOOKUP_BINARY)
    assert np.array_equal(binary, np.arange(len(keys), dtype=np.uint64))
    assert np.array_equal(ix.lookup(R, _abi.EO_LOOKUP_LEARNED), binary)
    # eo_index (api_index.cpp): ctx, kind, learned, n, log2nb, mem, ent, off, model
    word = lambda at: ctypes.c_uint64.from_address(ix.handle + at).value  # noqa: E731
    assert word(8) == _abi.EO_INDEX_SORTED | 1 << 32 and word(16) == len(keys)
    leaves = word(56) + (257 * 8 + 63) // 64 * 64  # behind 257 knots
    leaf = np.empty((4096, 8), dtype=np.int32)  # a, b, k0, pad, err_lo, err_hi, first, last
    assert ctx.lib.eo_copy_d2h(ctx.handle, leaf.ctypes.data, leaves, leaf.nbytes) == _abi.EO_OK
    assert leaf[:, 7].max() == len(keys) and leaf[:, 4:6].max() == ix.info()["max_err"]
    moved = leaf.copy()
    moved[:, 0] = (np.ascontiguousarray(leaf[:, 0]).view(np.float32) + np.float32(3 * (leaf[:, 4:6].max() + 1))).view(np.int32)
    assert ctx.lib.eo_copy_h2d(ctx.handle, leaves, moved.ctypes.data, moved.nbytes) == _abi.EO_OK
    wrong = ix.lookup(R, _abi.EO_LOOKUP_LEARNED)
    assert (wrong[:-4 * leaf[:, 4:6].max() - 8] > binary[:-4 * leaf[:, 4:6].max() - 8]).all()
    assert np.array_equal(ix.lookup(R, _abi.EO_LOOKUP_BINARY), binary)
    ix.free()


@pytest.mark.parametrize("n", [1, 17, 4096, 4097, 200_003])
def test_export_returns_the_entries(ctx, n):
    """Few entries are split on the host, more on the device."""
    rng = np.random.default_rng(n)
    R = np.stack([rng.integers(-n, n, n), np.arange(n)], 1).astype(np.int32)
    ix = ctx.sidx_build(R)
    keys, pays = ix.export()
    order = np.argsort(R[:, 0], kind="stable")
    assert np.array_equal(keys, R[order, 0]) and np.array_equal(pays, order)
    ix.free()


@pytest.mark.parametrize("dups", [15, 16, 17, 33, 500])
def test_deterministic_hash_join_of_long_buckets(ctx, dups):
    """Buckets of many duplicates, read two entries at a time from odd and even starts."""
    rng = np.random.default_rng(dups)
    keys = np.concatenate([np.repeat(np.arange(0, 40, 2), dups + rng.integers(0, 2, 20)), np.arange(1001, 1040)])
    R = np.stack([rng.permutation(keys), np.arange(len(keys))], 1).astype(np.int32)
    S = np.stack([rng.integers(0, 60, 300), np.arange(300)], 1).astype(np.int32)
    ix = ctx.hidx_build(R)
    rows = ix.join(S, deterministic=True)
    assert same_multiset(rows, brute_join(R, S))
    outer = ix.join(S, deterministic=True, left_outer=True)
    null = outer[:, 0] == _abi.EO_NULL_PAYLOAD
    assert same_multiset(outer[~null], rows)
    assert np.array_equal(np.sort(outer[null, 1]), np.flatnonzero(~np.isin(S[:, 0], R[:, 0])))
    ix.free()
