"""The build's radix sorts at the edges of their forms (one tile in one
workgroup, wide and narrow digits, one and two tiles per workgroup, the large
tile), through the arrays they order: the edge store is stable by timestamp
and the node index stable by (node, position), which numpy's stable argsort
gives exactly."""
import numpy as np
import pytest
import torch  # noqa: F401  (its HIP runtime comes up before the engine loads the system one)

from temporal_random_walk import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("directed", [True, False])
@pytest.mark.parametrize("n,ts_bits", [
    (1, 8), (2, 1), (64, 33), (1023, 20), (2047, 8), (2048, 9), (2049, 9), (4097, 33),
    (100_001, 20), (262_145, 27), (524_288, 20), (524_289, 20), (2_097_153, 30),
    (6_291_456, 17), (12_582_912, 12),
    (100_001, 40), (12_582_912, 40),  # the widest LDS tiles: 72 and 74 KiB
])
def test_store_and_node_index_order_at_the_sort_forms_edges(n, ts_bits, directed):
    if n > 6_291_456 and not directed:
        pytest.skip("the undirected index of half as many edges sorts as many entries")
    rng = np.random.default_rng(n + ts_bits)
    nodes = max(2, n // 7)
    src = rng.integers(0, nodes, n).astype(np.int32)
    src[rng.random(n) < 0.4] = nodes // 2  # a hub: rows of one digit
    dst = rng.integers(0, nodes, n).astype(np.int32)
    ts = rng.integers(0, 1 << ts_bits, n).astype(np.int64) - 5
    eng = capi.Engine(is_directed=directed)
    eng.add_edges(src, dst, ts)
    order = np.argsort(ts, kind="stable")
    s, d = src[order], dst[order]
    np.testing.assert_array_equal(eng.array("timestamps"), ts[order])
    np.testing.assert_array_equal(eng.array("sources"), s)
    np.testing.assert_array_equal(eng.array("targets"), d)
    if directed:
        out, inn = np.argsort(s, kind="stable"), np.argsort(d, kind="stable")
        np.testing.assert_array_equal(eng.array("node_ts_sorted_inbound_indices"), inn)
    else:  # entries 2i and 2i + 1 are edge i seen from its endpoints
        both = np.stack([s, d], axis=1).ravel()
        out = np.argsort(both, kind="stable") // 2
    np.testing.assert_array_equal(eng.array("node_ts_sorted_outbound_indices"), out)
    # the groups: runs of equal timestamps in the store, and of equal (node,
    # timestamp) in the node index
    t = ts[order]
    np.testing.assert_array_equal(eng.array("timestamp_group_offsets"), _starts(t[1:] != t[:-1], n))
    node = s[out] if directed else np.sort(both, kind="stable")
    starts = _starts((node[1:] != node[:-1]) | (t[out][1:] != t[out][:-1]), out.size)
    np.testing.assert_array_equal(eng.array("node_ts_group_outbound_offsets"), starts[:-1])
    first = np.searchsorted(node, np.arange(int(max(s.max(), d.max())) + 2))
    np.testing.assert_array_equal(eng.array("count_ts_group_per_node_outbound"),
                                  np.searchsorted(starts[:-1], first))
    eng.close()


def _starts(changes, n):
    """Positions starting a run (changes: where position i + 1 differs from i), then n."""
    return np.concatenate([[0], np.nonzero(changes)[0] + 1, [n]]).astype(np.uint64)
