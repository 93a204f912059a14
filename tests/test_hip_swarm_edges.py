"""Envs of more than 64 agents at the edges of the candidate search and the touch record:
exactly as many touching agents as a pass or a record word holds and one more, agents outside
the search's frame, rollouts too short for the whole skin, crowds that overflow the whole skin
but not a quarter of it, per-env parameter rows.  States equal the oracle's bit for bit, a tape
changes no bit, gradients within the bars of test_hip_swarm.py."""

import numpy as np
import pytest
import torch

from cases import oracle_cfg, params_of
from hip_helpers import hip_run, make_stepper, oracle_run, rel
from oracle.oracle import Oracle, pack_state
from swarp_amd import per_env_float_template
from swarp_amd.config import AgentConfig, WorldConfig

pytestmark = pytest.mark.gpu


def _clusters(E, A, size, half, rng):
    """Agents in clusters of `size` that all touch each other (pairwise within 0.04 of a reach
    of 0.125), the clusters on a lattice 0.5 apart."""
    n = -(-A // size)
    side = int(np.ceil(np.sqrt(n)))
    at = np.stack(np.meshgrid(np.arange(side), np.arange(side)), -1).reshape(-1, 2)[:n] * 0.5 - half
    pos = np.repeat(at, size, axis=0)[:A]
    pos = pos[rng.permutation(A)]  # a cluster's indices lie apart
    return pos + rng.uniform(-0.014, 0.014, size=(E, A, 2))


def _check(cfgs, world, S, s0, acts, seed):
    T, E, A = acts.shape[:3]
    w = np.random.default_rng(seed).normal(size=(T, E, A, 16))
    w[..., 7:] = 0.0
    on = make_stepper(cfgs, world, 0.05, S, torch.float32)
    off = make_stepper(cfgs, world, 0.05, S, torch.float32)
    off.use_tape = False
    a, b = hip_run(on, s0, acts, w, np.float32), hip_run(off, s0, acts, w, np.float32)
    for x, y in zip(a, b):
        assert np.array_equal(x, y), "the tape changes a result"
    o = oracle_run(cfgs, world, 0.05, S, s0, acts, w, np.float32)
    assert np.array_equal(a[0][..., :7], o[0][..., :7])
    assert rel(a[2], o[2]) <= 1e-5 and rel(a[1][..., :7], o[1][..., :7]) <= 1e-5


@pytest.mark.parametrize("method", ["brute", "uniform_grid"])
@pytest.mark.parametrize("size,K", [
    (5, 16),    # 4 touching agents: one pass, a full first word
    (6, 16),    # 5: a second pass, a second word
    (9, 16),    # 8: the record's last
    (10, 16),   # 9: one more than it holds
    (14, 16),   # four passes
    (10, 6),    # truncated, the cap within the second pass
    (10, 8),    # truncated at a whole number of passes
    (12, 11),   # exactly K listed: not truncated
])
def test_touching_clusters(size, K, method):
    E, A, half = 2, 96, 2.6
    rng = np.random.default_rng(size + K)
    s0 = pack_state({"pos": _clusters(E, A, size, half, rng)}).astype(np.float32)
    acts = rng.uniform(-1, 1, size=(3, E, A, 2)).astype(np.float32)
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025,
                        bounds=(-half, half, -half, half), max_neighbors=K, neighbor_method=method)
    _check([AgentConfig(radius=0.05) for _ in range(A)], world, 2, s0, acts, size)


@pytest.mark.parametrize("A,T,S,rho,kw", [
    (80, 1, 1, 15.0, {}),                                 # one substep: no skin
    (80, 1, 1, 60.0, dict(neighbor_radius=0.3)),          # overflows without any
    (150, 1, 4, 15.0, dict(neighbor_radius=0.3)),         # three eighths of the skin
    (70, 2, 3, 60.0, {}),                                 # overflows: straight to the traversal
    (200, 3, 3, 30.0, {}),                                # overflows the whole skin, not a quarter
    (200, 3, 3, 90.0, {}),                                # overflows both
    (70, 3, 3, 30.0, dict(neighbor_method="uniform_grid", uniform_bins=6)),
    (600, 2, 2, 30.0, {}),                                # uniform grid
])
def test_crowds(A, T, S, rho, kw):
    E, half = 2, float(np.sqrt(A / rho) / 2)
    rng = np.random.default_rng(A + T)
    s0 = pack_state({"pos": rng.uniform(-half, half, size=(E, A, 2))}).astype(np.float32)
    acts = rng.uniform(-1, 1, size=(T, E, A, 2)).astype(np.float32)
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025,
                        bounds=(-half, half, -half, half), max_neighbors=32, **kw)
    _check([AgentConfig(radius=0.05) for _ in range(A)], world, S, s0, acts, A)


@pytest.mark.parametrize("method", ["brute", "uniform_grid"])
def test_agents_outside_the_frame(method):
    """Most agents lie beyond the bounds, where the search's cells are clamped."""
    E, A, half = 2, 130, 0.5
    rng = np.random.default_rng(3)
    s0 = pack_state({"pos": rng.uniform(-4, 4, size=(E, A, 2))}).astype(np.float32)
    acts = rng.uniform(-1, 1, size=(4, E, A, 2)).astype(np.float32)
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025,
                        bounds=(-half, half, -half, half), max_neighbors=8, neighbor_method=method)
    _check([AgentConfig(radius=0.05) for _ in range(A)], world, 2, s0, acts, 3)


@pytest.mark.parametrize("A,method", [(90, "brute"), (90, "uniform_grid"), (1100, "brute")])
def test_per_env_rows(A, method):
    """Every env with its own radii, masses and speeds, against the oracle run env by env."""
    E, T, S, half = 3, 3, 2, float(np.sqrt(A) / 5)
    rng = np.random.default_rng(A)
    cfgs = [AgentConfig(radius=0.05) for _ in range(A)]
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025,
                        bounds=(-half, half, -half, half), max_neighbors=8, neighbor_method=method)
    rows = np.array(per_env_float_template(cfgs, E))
    rows[..., 0] *= rng.uniform(0.5, 1.0, size=(E, A))
    rows[..., 1] = rng.uniform(0.5, 2.0, size=(E, A))
    rows[..., 2] = rng.uniform(0.4, 1.0, size=(E, A))
    rows = rows.astype(np.float32).astype(np.float64)
    s0 = pack_state({"pos": rng.uniform(-half, half, size=(E, A, 2))}).astype(np.float32)
    acts = rng.uniform(-1, 1, size=(T, E, A, 2)).astype(np.float32)
    w = rng.normal(size=(T, E, A, 16))
    w[..., 7:] = 0.0
    out = []
    for tape in (True, False):
        st = make_stepper(cfgs, world, 0.05, S, torch.float32)
        st.use_tape = tape
        st.set_agent_params_per_env(rows)
        assert st.desc(E, 2).params_per_env == 1
        out.append(hip_run(st, s0, acts, w, np.float32))
    for x, y in zip(*out):
        assert np.array_equal(x, y), "the tape changes a result"
    O = Oracle(np.float32)
    _, tag, mode = params_of(cfgs)
    for e in range(E):
        cfg = oracle_cfg(cfgs, world, 0.05, S, 1, 2)
        one = lambda x, ax: np.ascontiguousarray(np.take(x, [e], axis=ax))  # noqa: E731
        p = rows[e].astype(np.float32)
        states = O.rollout(cfg, p, tag, mode, None, one(s0, 0), one(acts, 1))
        g0, ga = O.rollout_adj(cfg, p, tag, mode, None, one(s0, 0), one(acts, 1), states, one(w, 1), None)
        assert np.array_equal(out[0][0][:, e:e + 1, :, :7], states[..., :7].astype(np.float64)), f"env {e}"
        assert rel(out[0][2][:, e:e + 1], ga) <= 1e-5
        assert rel(out[0][1][e:e + 1, :, :7], g0[..., :7]) <= 1e-5
