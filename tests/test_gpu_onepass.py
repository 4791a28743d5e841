"""Fused joins that partition both relations together in one pass: sampled and exact counts, sizes
at the edges of tiles and of the choice between the two, clumped and skewed keys, a sample that
proves too small, and left outer joins whose null rows come with the probe."""
import numpy as np
import pytest

import eating_one_amd as eo
from eating_one_amd import _abi
from common import brute_join, same_multiset
from test_gpu_sampled import _sampled_lines

pytestmark = pytest.mark.gpu


def _check(ctx, R, S, sampled, outer=True, **kw):
    want = brute_join(R, S)
    st = eo.JoinStats()
    assert same_multiset(ctx.hash_join(R, S, stats=st, **kw), want)
    assert st.sampled == sampled and st.passes == 1
    if not outer:
        return
    for wide in (False, True):
        rows = ctx.hash_join(R, S, left_outer=True, result16=wide, **kw)
        null = rows[:, 0] == _abi.EO_NULL_PAYLOAD
        assert same_multiset(rows[~null][:, [0, 2] if wide else [0, 1]], want)
        absent = S[~np.isin(S[:, 0], R[:, 0])]
        got = rows[null]
        if wide:
            assert (got[:, 1] == _abi.EO_NULL_PAYLOAD).all()
            assert same_multiset(got[:, [3, 2]], absent)
        else:
            assert np.array_equal(np.sort(got[:, 1]), np.sort(absent[:, 1]))
    assert ctx.hash_join(R, S, left_outer=True, count_only=True, **kw) == len(want) + len(absent)


def _relations(nR, nS, keys, seed):
    rng = np.random.default_rng(seed)
    R = np.stack([rng.integers(-keys, keys, nR), np.arange(nR)], 1).astype(np.int32)
    S = np.stack([rng.integers(-keys, keys, nS), np.arange(nS)], 1).astype(np.int32)
    return R, S


@pytest.mark.parametrize("bits", [1, 5, 8, 10])
@pytest.mark.parametrize("nR,nS", [(3, 5), (16384, 16385), (40001, 131072), (70001, 17)])
def test_exact_counts(ctx, bits, nR, nS):
    """Small relations are counted whole; at 1 bit R takes several LDS tables a partition (the
    null rows wait for the last of them)."""
    R, S = _relations(nR, nS, nR, bits * 7 + nR)
    for lds in (8192, 16384):
        _check(ctx, R, S, 0, radix_bits=bits, passes=1, lds_tuples=lds)


@pytest.mark.parametrize("bits", [7, 9, 10])
@pytest.mark.parametrize("nR,nS,sampled", [((1 << 20) - 1, (1 << 20) - 1, 0), (1 << 20, 30001, 1),
                                           (50001, (1 << 20) + 16385, 1), ((1 << 20) + 9, (1 << 21) + 131073, 1)])
def test_sampled_counts(ctx, bits, nR, nS, sampled):
    R, S = _relations(nR, nS, nR, bits + nS)
    _check(ctx, R, S, sampled, outer=bits == 9, radix_bits=bits, passes=1)


@pytest.mark.parametrize("run", [1, 2, 7, 16, 64, 300])
def test_clumped_keys_keep_the_sampled_layout(ctx, run):
    """Sorted and grouped probe keys widen the margins, they do not overflow them."""
    nR, nS = (1 << 20) + 5, (1 << 21) + 77
    R = np.stack([np.arange(nR), np.arange(nR)], 1).astype(np.int32)
    keys = np.repeat(np.random.default_rng(run).integers(0, 2 * nR, nS // run + 1), run)[:nS]
    S = np.stack([keys, np.arange(nS)], 1).astype(np.int32)
    _check(ctx, R, S, 1, outer=False, radix_bits=8, passes=1)


def test_hot_key(ctx):
    """Most of S in one partition: its spans spread over the chip."""
    rng = np.random.default_rng(3)
    nR, nS = 300_000, 1_500_001
    R = np.stack([rng.permutation(nR), np.arange(nR)], 1).astype(np.int32)
    keys = np.where(rng.random(nS) < 0.8, 12345, rng.integers(0, 2 * nR, nS))
    S = np.stack([keys, np.arange(nS)], 1).astype(np.int32)
    _check(ctx, R, S, 1)


def test_sample_too_small_redoes_the_join(ctx):
    """Every line the sample reads holds spread keys, every other line one hot key."""
    rng = np.random.default_rng(4)
    n = 1 << 20
    keys = np.full(n, 5)
    for t in range(n // 16384):
        for j in range(64):
            b = t * 16384 + _sampled_lines(t, j) * 16
            keys[b:b + 16] = rng.integers(0, 1 << 20, 16)
    S = np.stack([keys, np.arange(n)], 1).astype(np.int32)
    R = np.stack([rng.permutation(200_000), np.arange(200_000)], 1).astype(np.int32)
    _check(ctx, R, S, 2, radix_bits=6, passes=1)
    assert same_multiset(ctx.hash_join(R[:5000], S[:9000]), brute_join(R[:5000], S[:9000]))


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("order", ["random", "sorted", "one digit"])
@pytest.mark.parametrize("flags", [0, _abi.EO_F_EXACT_PARTITIONS])
def test_few_digits(ctx, bits, order, flags):
    """Few digits are counted in several copies each: waves of mixed and of single digits, tiles
    that end anywhere, in the reserving scatter (flags = 0) and the counted one."""
    nR, nS = 16384 + 129, 3 * 16384 + 77
    R, S = _relations(nR, nS, nR, bits)
    if order == "sorted":
        R, S = R[np.argsort(R[:, 0])], S[np.argsort(S[:, 0])]
        R[:, 0] >>= 1  # runs of equal digits
    elif order == "one digit":
        R[:, 0] &= -64
        S[:, 0] &= -64
    _check(ctx, R, S, 0, outer=False, radix_bits=bits, passes=1, flags=flags)


@pytest.mark.parametrize("nR,nS", [(70_000, 1), (70_000, 10), (1_000_003, 50), (5_000_000, 300)])
def test_planned_outer_join_of_few_probes(ctx, nR, nS):
    """Fewer probes than partitions, no plan given: the spans are one batch at least."""
    R, S = _relations(nR, nS, nR, nR + nS)
    want = brute_join(R, S)
    rows = ctx.hash_join(R, S, left_outer=True)
    null = rows[:, 0] == _abi.EO_NULL_PAYLOAD
    assert same_multiset(rows[~null], want)
    assert np.array_equal(np.sort(rows[null, 1]), np.sort(S[~np.isin(S[:, 0], R[:, 0]), 1]))
