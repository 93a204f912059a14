"""The lane tape of movable-body rollouts (forces and touching agents of the few lanes that
feel any, shapes touched): a backward that reads it against one that evaluates the forces
again.  Bar: equal bit for bit, as for every tape."""

import numpy as np
import pytest
import torch

from cases import nav_agents
from hip_helpers import TDT, make_stepper
from test_hip_v_bodies import _pushers, _ring_extra, _world, cross_obs, hip_body_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,A,S,extra,world,shapes,dtype", [
    (5, 64, 4, 0, {}, False, np.float32),                    # one env per wave, one body
    (5, 64, 5, 3, {}, False, np.float32),                    # a fifth substep: a second read of four
    (4, 64, 2, 0, dict(max_neighbors=3), False, np.float32), # truncated lists
    (9, 13, 4, 4, dict(max_neighbors=2), False, np.float32), # four envs per wave, some truncated
    (7, 5, 1, 2, {}, False, np.float32),
    (6, 12, 3, 4, {}, True, np.float32),                     # boxes and segments among the shapes
    (3, 64, 2, 75, dict(max_neighbors=8), False, np.float32),  # more than 64 shapes
    (4, 30, 4, 3, dict(max_neighbors=4), False, np.float64),
])
def test_lane_tape_matches_recompute(E, A, S, extra, world, shapes, dtype):
    s0, acts = _pushers(E, A, 29 + A, spread=0.8)
    obs = cross_obs(E, (0.0, 0.0), extra=_ring_extra(extra, radius=0.6) if extra else ())
    n = obs["pos"].shape[1]
    if shapes:
        ty = np.arange(n) % 3
        obs["type"] = ty.astype(np.int32)
        obs["half"] = np.where((ty > 0)[:, None], [0.12, 0.06], 0.0)
        obs["angle"] = np.zeros((E, n))
    td = TDT[dtype]
    runs = []
    for tape in ("lanes", "records", None):
        st = make_stepper(nav_agents(A), _world(**world), 0.05, S, td, obs=obs, n_envs=E)
        st.use_tape = tape is not None
        records = acts.shape[0] * S * E * st.n_body_roots * 12 * (4 if td == torch.float32 else 8)
        if tape == "lanes":
            assert st.ob_tape_bytes(E, 2, acts.shape[0]) > records
        if tape == "records":  # a tape of the body records alone is taken as well
            st.ob_tape_bytes = lambda *a: records
        runs.append(hip_body_run(st, s0, acts, td, seed=3)[0])
    names = ("agent states", "obstacle states", "d/d pos0", "d/d ob0", "d/d actions")
    for other in runs[1:]:
        for name, x, y in zip(names, runs[0], other):
            assert np.array_equal(x, y), f"{name} differ"
    assert np.abs(runs[0][4]).max() > 0


def test_agent_at_the_centre_of_a_shape():
    """An agent exactly at a round shape's centre exerts no force on it, yet the derivative is
    the largest a contact has (the offset divided by the contact law's smallest distance): the
    tape has to name the shape.  No other agent is near the body."""
    E, A, td = 3, 4, torch.float32
    s0, acts = _pushers(E, A, 5, spread=0.8)
    s0[:, :, 0:2] = [[0.0, 0.0], [0.9, 0.9], [-0.9, 0.9], [0.9, -0.9]]
    runs = []
    for tape in (True, False):
        st = make_stepper(nav_agents(A), _world(), 0.05, 2, td, obs=cross_obs(E, (0.0, 0.0)),
                          n_envs=E)
        st.use_tape = tape
        runs.append(hip_body_run(st, s0, acts[:1], td, seed=3)[0])
    for name, x, y in zip(("agent states", "obstacle states", "d/d pos0", "d/d ob0", "d/d actions"),
                          *runs):
        assert np.array_equal(x, y), f"{name} differ"
    assert np.abs(runs[1][3]).max() > 1e3  # the contact's derivative reaches the body
