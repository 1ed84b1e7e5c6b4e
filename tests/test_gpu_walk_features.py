"""Edge features of the walks: every slot's row is its edge's, zeros past the
walk's length, for dims on both sides of the 16-byte path and of the layout
pass's, slot counts that end inside a workgroup's run, and rows of several
layout chunks."""
import numpy as np
import pytest
import torch  # noqa: F401  (its HIP runtime comes up before the engine loads the system one)

from temporal_random_walk import capi
from tests import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 3, 4, 5, 8, 16, 20, 48, 260])
@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("n_walks,L", [(1, 2), (7, 40), (512, 3), (1025, 2), (65, 125), (5_001, 21)])
def test_walk_features_are_the_edges_rows(dim, forward, n_walks, L):
    s, d, t = graphs.cfg1(n_nodes=200, n_edges=3_000, seed=5)
    feat = np.random.default_rng(dim).standard_normal((3_000, dim), dtype=np.float32)
    eng = capi.Engine(is_directed=True, global_seed=11)
    eng.add_edges(s, d, t, feat)
    store = eng.array("edge_features").reshape(-1, dim)
    for layout in ("auto", "scratch"):
        w = eng.sample("total", L, "Uniform", n_walks, walk_layout=layout,
                       direction="Forward_In_Time" if forward else "Backward_In_Time")
        want = np.where((w.edge_ids >= 0)[..., None], store[w.edge_ids], np.float32(0))
        assert w.edge_features.shape == (n_walks, L - 1, dim)
        np.testing.assert_array_equal(w.edge_features, want)
    eng.close()
