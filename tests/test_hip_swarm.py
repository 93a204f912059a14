"""Envs of more than 64 agents on the GPU, at the sizes where their kernels can go wrong:
edges of the reductions and tables, remainders, crowded cells, truncated lists.  Lists and
states must equal the oracle's bit for bit; a tape must not change a bit of a gradient."""

import numpy as np
import pytest
import torch

from hip_helpers import hip_run, make_stepper, oracle_run, rel
from oracle.oracle import Oracle, pack_state
from swarp_amd import NeighborGrid
from swarp_amd.config import AgentConfig, DynamicsModel, WorldConfig

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


@pytest.mark.parametrize("E,A,T,S,half,kw", [
    (5, 65, 6, 4, 2.2, {}),                               # just past a wavefront, sparse
    (3, 256, 5, 3, 4.0, {}),                              # four waves, sparse
    (2, 200, 4, 4, 0.9, {}),                              # candidate lists overflow: full traversal
    (3, 130, 5, 2, 1.6, dict(max_neighbors=3)),           # lists truncated among few candidates
    (2, 90, 5, 2, 0.8, dict(neighbor_radius=0.3, max_neighbors=5)),
    (2, 128, 6, 1, 1.5, {}),                              # one substep: no skin
    (2, 600, 4, 2, 5.0, {}),                              # uniform grid, sparse
    (2, 600, 4, 3, 1.7, dict(max_neighbors=4)),           # uniform grid, truncated and overflowing
    (2, 70, 6, 3, 1.5, dict(neighbor_method="uniform_grid", uniform_bins=5)),
    (2, 1030, 3, 2, 7.0, {}),                             # two agents per thread
    (1, 1500, 3, 2, 8.0, dict(neighbor_method="brute")),
    (1, 2060, 2, 2, 9.0, {}),                             # four agents per thread
    (1, 3584, 2, 2, 12.0, dict(neighbor_method="brute")),  # the largest env: the shortest lists
    (2, 100, 4, 2, 1.6, dict(f64=True)),
    (1, 2048, 2, 2, 10.0, dict(f64=True, neighbor_method="brute")),
    (3, 80, 5, 4, 1.5, dict(shift=40000.0)),              # far from the origin: coarse positions
    (3, 96, 5, 4, 2.0, dict(fast=6.0)),                   # agents outrun the skin
    (3, 96, 5, 2, 1.1, dict(mixed=True)),                 # diff-drive and bicycle
])
def test_swarm_rollout(E, A, T, S, half, kw):
    """States bit-exact with the oracle (float64: 1e-12), gradients within the bars; with and
    without the tape the same bits."""
    kw = dict(kw)
    dt = np.float64 if kw.pop("f64", False) else np.float32
    shift, fast, mixed = kw.pop("shift", 0.0), kw.pop("fast", 0.0), kw.pop("mixed", False)
    rng = np.random.default_rng(A + S)
    cfgs = [AgentConfig(radius=0.05) for _ in range(A)]
    if mixed:
        cfgs = [AgentConfig(model=DynamicsModel.DIFF_DRIVE if k % 2 else
                            DynamicsModel.KINEMATIC_BICYCLE, radius=0.05) for k in range(A)]
    ad, nf = 2, 5
    s0 = {"pos": rng.uniform(-half, half, size=(E, A, 2)) + shift,
          "theta": rng.uniform(-np.pi, np.pi, size=(E, A))}
    acts = rng.uniform(-1, 1, size=(T, E, A, 2))
    bounds = (shift - half, shift + half, shift - half, shift + half)
    if fast:  # drones keep their initial velocity, whatever max_speed says
        cfgs = [AgentConfig(model=DynamicsModel.DRONE, radius=0.1) for _ in range(A)]
        ad, nf, bounds = 4, 9, None
        s0["vel"] = rng.uniform(-fast, fast, size=(E, A, 2))
        s0["attitude"] = np.broadcast_to([0.0, 0.0, 0.0, 1.0], (E, A, 4))
        acts = rng.uniform(0, 10, size=(T, E, A, 4))
    s0, acts = pack_state(s0).astype(dt), acts.astype(dt)
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025, bounds=bounds,
                        **kw)
    w = rng.normal(size=(T, E, A, 16)) * (0.01 if fast else 1.0)
    if nf == 5:
        w[..., 7:] = 0.0
    td = torch.float32 if dt == np.float32 else torch.float64
    on = make_stepper(cfgs, world, 0.05, S, td)
    off = make_stepper(cfgs, world, 0.05, S, td)
    off.use_tape = False
    assert on.wide and on.tape_bytes(E, ad, T) > 0 and off.tape_bytes(E, ad, T) == 0
    a, b = hip_run(on, s0, acts, w, dt), hip_run(off, s0, acts, w, dt)
    for x, y in zip(a, b):
        assert np.array_equal(x, y), "the tape changes a result"
    o = oracle_run(cfgs, world, 0.05, S, s0, acts, w, dt)
    cols = slice(0, 16 if fast else 7)
    if dt == np.float32:
        assert np.array_equal(a[0][..., cols], o[0][..., cols])
    else:
        assert rel(a[0][..., cols], o[0][..., cols]) <= 1e-12
    tol = 1e-5 if dt == np.float32 else 1e-12  # the gradient bars of test_hip_wide.py
    assert rel(a[2], o[2]) <= tol and rel(a[1][..., cols], o[1][..., cols]) <= tol
