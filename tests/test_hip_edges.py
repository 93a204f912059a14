"""The COO graph of padded lists (``NeighborGrid.edge_index``: tile sums, then the edges)
against ``swarp_edge_index`` with torch's prefix sums and against the lists themselves.  Bar:
equal."""

import pytest
import torch

from swarp_amd import NeighborGrid, _lib

pytestmark = pytest.mark.gpu


def _lists(E, A, K, seed, fill):
    """A grid with lists of random lengths (`fill`: the share of rows that hold any)."""
    g = NeighborGrid(E, A, radius=0.3, max_neighbors=K, device="cuda:0")
    gen = torch.Generator("cpu").manual_seed(seed)
    cnt = torch.randint(0, K + 1, (E, A), generator=gen)
    cnt[torch.rand(E, A, generator=gen) >= fill] = 0
    idx = torch.randint(0, A, (E, A, K), generator=gen)
    g.neighbor_idx.copy_(idx)
    g.neighbor_count.copy_(cnt)
    keep = torch.arange(K) < cnt[..., None]
    e, a, k = keep.nonzero(as_tuple=True)
    return g, torch.stack([e * A + idx[e, a, k], e * A + a])


@pytest.mark.parametrize("E,A,K,fill", [
    (1, 1, 1, 1.0),
    (1, 511, 4, 1.0),        # one agent short of a workgroup
    (3, 171, 5, 0.7),        # 513 agents, rows that are not whole 16-byte pieces
    (4, 512, 16, 0.5),       # exactly one tile
    (683, 3, 8, 0.4),        # 2049 agents: a tile and one
    (7, 1000, 6, 0.01),      # mostly empty
    (40000, 60, 4, 0.3),     # more agents than 1024 tiles of 2048
])
def test_edges_match_the_lists(E, A, K, fill):
    g, want = _lists(E, A, K, E + A + K, fill)
    for _ in range(2):
        got = g.edge_index()
        assert got.dtype == torch.int64 and torch.equal(got.cpu(), want)
    cnt = g.neighbor_count.reshape(-1)
    off = (torch.cumsum(cnt, 0, dtype=torch.int64) - cnt).contiguous()
    ref = torch.full_like(got, -1)
    _lib.check(_lib.load().swarp_edge_index(
        E, A, K, g.neighbor_idx.data_ptr(), cnt.data_ptr(), off.data_ptr(), want.shape[1],
        ref.data_ptr(), _lib.stream_of(ref.device)))
    assert torch.equal(got, ref)


@pytest.mark.parametrize("E,A,K,fill", [
    (2100, 1000, 2, 0.5),   # just above 1024 tiles of 2048: two parts a workgroup
    (6001, 701, 3, 0.3),    # three, a ragged end
    (4100, 1023, 1, 1.0),   # a last workgroup with one agent of its second part
])
def test_more_agents_than_single_part_workgroups(E, A, K, fill):
    test_edges_match_the_lists(E, A, K, fill)


def test_no_edges_and_another_stream():
    g, _ = _lists(5, 300, 4, 1, 0.0)
    assert g.edge_index().shape == (2, 0)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        h, want = _lists(5, 300, 4, 2, 1.0)
        got = h.edge_index()
    s.synchronize()
    assert torch.equal(got.cpu(), want)
