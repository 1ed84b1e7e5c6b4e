"""Small host copies: batches and walk sets on both sides of the 2 MiB up to
which one kernel moves every array through a pinned buffer, and of the staged
chunks above it, with arrays that end inside a 16-byte unit."""
import numpy as np
import pytest
import torch

from temporal_random_walk import TemporalRandomWalk, capi
from tests import graphs

pytestmark = pytest.mark.gpu


# 16 bytes an edge without features: 131 072 edges are 2 MiB
@pytest.mark.parametrize("n", [1, 3, 257, 131_071, 131_072, 131_073, 600_001])
@pytest.mark.parametrize("dim", [0, 3])
def test_host_ingest_matches_device_ingest(n, dim):
    rng = np.random.default_rng(n)
    src = rng.integers(0, 1_000, n).astype(np.int32)
    dst = rng.integers(0, 1_000, n).astype(np.int32)
    ts = rng.integers(0, 5_000, n).astype(np.int64)
    feat = rng.standard_normal((n, dim)).astype(np.float32) if dim else None
    a, b, c = (capi.Engine(is_directed=True, global_seed=5) for _ in range(3))
    a.add_edges(src, dst, ts, feat)
    dv = [None if x is None else torch.from_numpy(x).cuda() for x in (src, dst, ts, feat)]
    torch.cuda.synchronize()
    b.add_edges_device(dv[0].data_ptr(), dv[1].data_ptr(), dv[2].data_ptr(), n,
                       dv[3].data_ptr() if dim else None, dim)
    c.prefetch_edges(src, dst, ts, feat)
    c.add_prefetched_edges()
    names = ["sources", "targets", "timestamps"] + (["edge_features"] if dim else [])
    for name in names:
        np.testing.assert_array_equal(a.array(name), b.array(name), err_msg=name)
        np.testing.assert_array_equal(c.array(name), b.array(name), err_msg=name)
    for e in (a, b, c):
        e.close()


# 20 bytes a slot: 6 553 walks of 16 are just below 2 MiB, 6 554 just above
@pytest.mark.parametrize("n,L", [(1, 2), (7, 3), (6_553, 16), (6_554, 16), (40_001, 21)])
def test_host_walks_match_device_walks(n, L):
    s, d, t = graphs.cfg1(n_nodes=1_000, n_edges=20_000, seed=9)
    eng = capi.Engine(is_directed=True, global_seed=77, shuffle_walk_order=False)
    eng.add_edges(s, d, t)
    host = eng.sample("total", L, "Linear", n)
    dev = eng.sample_device("total", L, "Linear", n)
    for got, ptr, shape in ((host.nodes, dev.nodes, (n, L)),
                            (host.timestamps, dev.timestamps, (n, L)),
                            (host.lens, dev.walk_lens, (n,)),
                            (host.edge_ids, dev.edge_ids, (n, L - 1))):
        want = capi.device_to_host(ptr, got.size, got.dtype)
        np.testing.assert_array_equal(got.reshape(shape), want.reshape(shape))
    # the class, which leaves the edge ids on the device
    tw = TemporalRandomWalk(is_directed=True, use_gpu=True, global_seed=77,
                            shuffle_walk_order=False)
    tw.add_multiple_edges(s, d, t)
    r = tw.get_random_walks_and_times(max_walk_len=L, walk_bias="Linear", num_walks_total=n,
                                      initial_edge_bias="Uniform")
    w = eng.sample("total", L, "Linear", n, initial_edge_bias="Uniform")
    np.testing.assert_array_equal(r[0], w.nodes)
    np.testing.assert_array_equal(r[1], w.timestamps)
    np.testing.assert_array_equal(r[2], w.lens)
    eng.close()
