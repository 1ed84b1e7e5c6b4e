"""The index's time keys: offsets from the first timestamp where most time
units of the span occur, ranks elsewhere, and slot words that hold a key's
offset in its edge's block.  Replay walks equal the oracle's bit for bit on
both sides of each rule."""
import numpy as np
import pytest

from tests import graphs
from tests.test_gpu_parity import WEIGHT_ARRAYS, _assert_index_equal, _pair, _walk_case

pytestmark = pytest.mark.gpu


def _units(rule, T):
    """T distinct time units: every unit of the span, every second one with a
    span of exactly 2 T units (still offsets), or one unit more (ranks)."""
    u = np.arange(T, dtype=np.int64)
    if rule != "dense":
        u = 2 * u
        u[-1] += 1 if rule == "half" else 2
    return u


@pytest.mark.parametrize("directed", [True, False])
@pytest.mark.parametrize("rule", ["dense", "half", "ranks"])
@pytest.mark.parametrize("t0", [0, -9_000, 1_600_000_000])
def test_walks_on_offset_and_rank_keys(rule, t0, directed):
    rng = np.random.default_rng(7)
    T, n = 15_000, 40_000
    units = _units(rule, T) + t0
    t = np.concatenate([units, rng.choice(units, n - T)])
    s, d, _ = graphs.powerlaw(2_000, n, s=1.4, seed=8)
    t = t[rng.permutation(n)]
    og, eng = _pair(directed, [(s, d, t)], weights=True, timescale_bound=30.0)
    _assert_index_equal(og, eng, weights=True)
    for name in WEIGHT_ARRAYS:
        w = eng.array(name)
        if w.size:
            og.set_weights(name, w)
    seeds = np.unique(s[:300]).astype(np.int32)
    # cutoffs before, inside and past the span, on and between its units
    cuts = rng.integers(units[0] - 50, units[-1] + 50, seeds.size)
    cuts[:4] = [units[0], units[0] + 1, units[-1], units[-1] + 1]
    cuts[4:6] = [-1, np.iinfo(np.int64).max - 1]
    for forward in (True, False):
        _walk_case(og, eng, "ExponentialIndex", "Linear", forward, "total", 20, 2_000, seed=1)
        _walk_case(og, eng, "ExponentialWeight", "ExponentialWeight", forward, "total", 20, 2_000,
                   seed=2)
        _walk_case(og, eng, "Linear", "Uniform", forward, "nodes", 16, 3, seed_nodes=seeds,
                   cutoffs=cuts, seed=3)


@pytest.mark.parametrize("gap", [1, 2])
@pytest.mark.parametrize("T", [1 << 19, (1 << 19) + 1])
def test_index_walks_at_the_rank_tables_limit(T, gap):
    """Without weights, gapped times are keyed by rank up to 2^19 unique
    timestamps and by offset past them; gapless ones always by offset."""
    rng = np.random.default_rng(27)
    n = T + 1_000
    units = gap * np.arange(T, dtype=np.int64) - 5_000
    t = np.concatenate([units, rng.choice(units, n - T)])[rng.permutation(n)]
    s, d, _ = graphs.powerlaw(3_000, n, s=1.4, seed=28)
    og, eng = _pair(True, [(s, d, t)])
    _assert_index_equal(og, eng)
    for forward in (True, False):
        _walk_case(og, eng, "ExponentialIndex", "Linear", forward, "total", 20, 2_000, seed=29)
        seeds = np.unique(s[:100]).astype(np.int32)
        cuts = rng.integers(units[0], units[-1] + 2, seeds.size)
        _walk_case(og, eng, "Linear", "Uniform", forward, "nodes", 16, 3, seed_nodes=seeds,
                   cutoffs=cuts, seed=30)


@pytest.mark.parametrize("gap", [False, True])
def test_weight_walks_on_key_blocks(gap):
    """22 + 22 + 22 bits do not fit a slot word: it holds 20 bits of the key's
    offset in its edge's block -- or, when one block would have to span a gap of
    2^21 units, no time at all (the edge's timestamp is looked up)."""
    rng = np.random.default_rng(17)
    e, T = 2_200_000, 2_150_000
    ids = np.concatenate([[0, (1 << 22) - 1],
                          rng.choice(np.arange(1, (1 << 22) - 1), 6_000, replace=False)])
    perm = rng.permutation(ids.size)
    s = ids[graphs.zipf_ids(rng, e, ids.size, 1.5, perm)].astype(np.int32)
    d = ids[graphs.zipf_ids(rng, e, ids.size, 1.5, perm)].astype(np.int32)
    units = np.arange(T, dtype=np.int64) if gap else 2 * np.arange(T, dtype=np.int64)
    if gap:
        units[-1] = 2 * T - 1
    units += 77
    t = np.concatenate([rng.permutation(units), rng.choice(units, e - T)])
    og, eng = _pair(True, [(s, d, t)], weights=True, timescale_bound=50.0)
    for name in WEIGHT_ARRAYS:
        og.set_weights(name, eng.array(name))
    for forward in (True, False):
        _walk_case(og, eng, "ExponentialWeight", "Uniform", forward, "total", 24, 10_000, seed=18)
        _walk_case(og, eng, "ExponentialIndex", "ExponentialWeight", forward, "total", 12, 5_000,
                   seed=19)
    assert eng.walk_stats()["slot_word_format"] == 1
