"""Envs of more than 64 agents on the GPU, at the sizes where their kernels can go wrong:
edges of the reductions and tables, remainders, crowded cells, truncated lists.  Lists and
states must equal the oracle's bit for bit; a tape must not change a bit of a gradient."""

import numpy as np
import pytest
import torch

from oracle.oracle import Oracle
from swarp_amd import NeighborGrid

pytestmark = pytest.mark.gpu


def _bins(A):
    return max(4, min(128, int(np.ceil(np.sqrt(A)))))


@pytest.mark.parametrize("E,A,dtype,shift", [
    (8, 256, np.float32, 0),    # 2048 positions: the last size of one workgroup
    (1, 2049, np.float32, 0),   # one more: two boxes, the second of one position
    (37, 130, np.float64, 0),   # three boxes with a remainder
    (37, 130, np.float64, 1),   # a list buffer not aligned for float64: one workgroup
    (37, 130, np.float32, 1),   # 4-byte alignment suffices for float32
])
def test_batch_frame(E, A, dtype, shift):
    """The frame reduced over the batch, through the list buffer as scratch."""
    K, r = 5, 0.2
    rng = np.random.default_rng(A + E)
    pos = ((rng.random((E, A, 2)) * 2 - 1) * [3.0, 1.0]).astype(dtype)
    pos[E - 1, A - 1] = [4.5, -2.5]  # the extremes in the last position
    pos[0, 0] = [-4.0, 3.5]
    g = NeighborGrid(E, A, radius=r, max_neighbors=K, device="cuda:0",
                     dtype=torch.float32 if dtype == np.float32 else torch.float64,
                     method="uniform_grid")
    idx = torch.zeros(E * A * K + 1, dtype=torch.int32, device="cuda")[shift:shift + E * A * K]
    cnt = torch.zeros(E, A, dtype=torch.int32, device="cuda")
    g.query_into(torch.tensor(pos, device="cuda"), idx.view(E, A, K), cnt)
    oi, oc, _, ofr = Oracle(dtype).neighbors_grid(pos, r, K, _bins(A))
    assert np.array_equal(g.grid_frame().cpu().numpy(), ofr)
    assert np.array_equal(cnt.cpu().numpy(), oc)
    assert np.array_equal(idx.view(E, A, K).cpu().numpy(), oi)


@pytest.mark.parametrize("A,spread", [(65, 0.0), (200, 0.05), (1500, 0.3)])
def test_grid_lists_in_crowded_cells(A, spread):
    """Many agents in a cell (all of them at spread 0): the order within a cell is the agent
    order, whatever order they arrive in."""
    E, K, r = 2, 7, 0.2
    rng = np.random.default_rng(A)
    pos = (rng.random((E, A, 2)) * spread + [0.31, -0.4]).astype(np.float32)
    g = NeighborGrid(E, A, radius=r, max_neighbors=K, device="cuda:0", method="uniform_grid",
                     bounds=(-2.0, 2.0, -2.0, 2.0))
    g.build(torch.tensor(pos, device="cuda"))
    bins = _bins(A)
    oi, oc, ot, _ = Oracle(np.float32).neighbors_grid(pos, r, K, bins, (-2.0, -2.0, max(r, 4.0 / bins)))
    assert np.array_equal(g.neighbor_idx.cpu().numpy(), oi)
    assert np.array_equal(g.neighbor_count.cpu().numpy(), oc)
    assert np.array_equal(g.neighbor_true_count.cpu().numpy(), ot)
