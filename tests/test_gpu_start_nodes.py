"""The start nodes of for_all_nodes and for_last_batch walks: ascending ids,
wpn walks each, at the edges of the id blocks, through the flags (ids no more
than the batch's entries) and through the sort (sparse ids)."""
import numpy as np
import pytest
import torch  # noqa: F401  (its HIP runtime comes up before the engine loads the system one)

from temporal_random_walk import capi

pytestmark = pytest.mark.gpu


def _starts(eng, mode, wpn):
    w = eng.sample(mode, 2, "Uniform", wpn, shuffle=False)
    assert np.all(w.lens == 2)  # undirected: every start has an edge
    return w.nodes[:, 0]


@pytest.mark.parametrize("max_id", [0, 1, 15, 16, 4_095, 4_096, 4_097, 70_000, 8_388_607, 8_400_001])
@pytest.mark.parametrize("n", [3, 500, 90_000])
def test_start_nodes_ascend(max_id, n):
    rng = np.random.default_rng(max_id + n)
    eng = capi.Engine(is_directed=False, global_seed=3)
    for batch in range(2):
        src = rng.integers(0, max_id + 1, n).astype(np.int32)
        dst = rng.integers(0, max_id + 1, n).astype(np.int32)
        src[0] = max_id
        eng.add_edges(src, dst, np.arange(n, dtype=np.int64) + batch * n)
        last = np.unique(np.concatenate([src, dst]))
        both = last if batch == 0 else np.union1d(both, last)
    np.testing.assert_array_equal(_starts(eng, "last_batch", 3), np.repeat(last, 3))
    np.testing.assert_array_equal(_starts(eng, "all_nodes", 2), np.repeat(both, 2))
    eng.close()


@pytest.mark.parametrize("max_id", [40, 300_000])
def test_last_batch_starts_of_a_directed_graph(max_id):
    rng = np.random.default_rng(4)
    src = rng.integers(0, max_id + 1, 5_000).astype(np.int32)
    dst = rng.integers(0, max_id + 1, 5_000).astype(np.int32)
    dst[0] = max_id
    eng = capi.Engine(is_directed=True, global_seed=3)
    eng.add_edges(src, dst, np.arange(5_000, dtype=np.int64))
    w = eng.sample("last_batch", 4, "Uniform", 1, shuffle=False)
    np.testing.assert_array_equal(w.nodes[:, 0], np.unique(src))
    eng.close()
