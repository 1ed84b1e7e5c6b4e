"""The scratch of a radix sort serves every sort of fewer keys, whose plan may
ask for more than the larger sort's own (wider digits up to 2^19 keys, smaller
tiles below 12 582 912): the node-grouped walk order takes it once for all its
walks and sorts those still alive."""
import ctypes

import numpy as np
import pytest
import torch  # its HIP runtime comes up before the engine loads the system one

from temporal_random_walk import capi
from tests import graphs


@pytest.mark.parametrize("bits", [1, 8, 9, 17, 20, 24, 27, 31, 32, 40, 64])
def test_scratch_of_n_keys_serves_fewer(bits):
    lib = ctypes.CDLL(capi.LIB_PATH)
    need, have = lib._ZN3trw15radix_min_elemsEmi, lib._ZN3trw15radix_tmp_elemsEmi
    for f in (need, have):
        f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_size_t, ctypes.c_int]
    edges = [2_048, 1 << 19, 1 << 21, 3 << 22]
    sizes = sorted({max(0, e + d) for e in edges for d in (-2_048, -1, 0, 1, 2_047, 4_096)} |
                   {int(x) for x in np.geomspace(1, 2e8, 400)})
    most = 0
    for n in sizes:
        most = max(most, need(n, bits))
        assert need(n, bits) <= have(n, bits)
        assert most <= have(n, bits), f"{n} keys by {bits} bits"
        assert most <= need(n, bits), f"{n} keys by {bits} bits"


@pytest.mark.gpu
def test_node_grouped_walks_as_they_run_out():
    """1M walks over 20-bit ids end at different lengths, so that regroupings
    sort live counts on both sides of 2^19."""
    s, d, t = graphs.powerlaw(20_000, 300_000, s=1.4, seed=6)
    eng = capi.Engine(is_directed=True, global_seed=21)
    eng.add_edges(s * 50, d * 50, t)
    L, n = 20, 1_000_000
    rows = []
    for order in ("walk_id", "node_grouped"):
        w = eng.sample_device("total", L, "Uniform", n, walk_order=order)
        got = []
        for ptr, count, dt in ((w.nodes, n * L, torch.int32), (w.timestamps, n * L, torch.int64),
                               (w.walk_lens, n, torch.int64),
                               (w.edge_ids, n * (L - 1), torch.int64)):
            x = torch.empty(count, dtype=dt, device="cuda")
            capi.device_copy(x.data_ptr(), ptr, x.numel() * x.element_size())
            got.append(x)
        torch.cuda.synchronize()
        rows.append(got)
    alive = int((rows[0][2] > 9).sum())  # regrouped after 8 hops: about 370 000
    assert 260_000 <= alive <= 520_000
    for a, b in zip(*rows):
        assert torch.equal(a, b)
    eng.close()
