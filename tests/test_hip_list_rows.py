"""Padded list rows as the list kernels write them: rows of every length and slot count, slots
that do not fill 16-byte stores, list buffers that are not 16-byte aligned, rows too long to be
staged.  Lists, counts and true counts equal to the oracle's."""

import numpy as np
import pytest
import torch

from oracle.oracle import Oracle
from swarp_amd import NeighborGrid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,A,K,r,shift", [
    (3, 64, 32, 0.25, 0),    # one env per wave
    (2, 64, 64, 3.0, 0),     # every other agent listed: 63 of 64 slots
    (5, 13, 7, 0.9, 0),      # slots not a multiple of 4, pad slots, a partial last wave
    (9, 4, 4, 1.5, 0),
    (17, 7, 1, 1.0, 0),
    (4, 30, 8, 0.7, 1),      # a buffer on a 4-byte boundary
    (3, 20, 12, 0.8, 2),
    (2, 100, 12, 0.5, 1),    # one env per workgroup
    (2, 65, 31, 0.6, 0),
    (1, 700, 33, 0.3, 0),    # grid order
    (1, 520, 520, 1.0, 0),   # rows too long to be staged
    (1, 3000, 60, 0.1, 0),
    # one wave's rows: whole slots up to 16 of them, packed ids beyond
    (3, 64, 16, 3.0, 0),     # the longest whole rows, full
    (3, 64, 15, 3.0, 0),
    (4, 64, 17, 3.0, 0),     # packed, a store from two pieces and, past the end, the next row
    (4, 64, 18, 0.6, 0),
    (4, 61, 19, 3.0, 0),     # slots of the wave not a multiple of 4
    (5, 40, 33, 3.0, 2),     # packed, a 4-byte boundary
    (6, 13, 40, 3.0, 0),     # more slots than agents
    (7, 4, 20, 3.0, 0),
    (1, 64, 300, 3.0, 0),    # more slots than a store step
])
def test_rows(E, A, K, r, shift):
    rng = np.random.default_rng(A + K)
    pos = rng.uniform(-1, 1, size=(E, A, 2)).astype(np.float32)
    g = NeighborGrid(E, A, radius=r, max_neighbors=K, device="cuda:0", bounds=(-1.0, 1.0, -1.0, 1.0))
    buf = torch.full((E * A * K + shift + 8,), -7, dtype=torch.int32, device="cuda")
    idx = buf[shift:shift + E * A * K].view(E, A, K)
    cnt = torch.zeros(E, A, dtype=torch.int32, device="cuda")
    g.query_into(torch.tensor(pos, device="cuda"), idx, cnt)
    if g.method == "brute":
        oi, oc, ot = Oracle(np.float32).neighbors(pos, r, K)
    else:
        bins = g.uniform_bins
        oi, oc, ot, _ = Oracle(np.float32).neighbors_grid(pos, r, K, bins, (-1.0, -1.0, max(r, 2.0 / bins)))
    assert np.array_equal(idx.cpu().numpy(), oi) and np.array_equal(cnt.cpu().numpy(), oc)
    assert np.array_equal(g.neighbor_true_count.cpu().numpy(), ot)
    assert (buf[:shift] == -7).all() and (buf[shift + E * A * K:] == -7).all(), "wrote past the rows"
