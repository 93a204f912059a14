"""A tape that memory is not there for is left out: the rollout runs and its backward gives the
same bits.  On the CPU the choice of a buffer, with torch's allocator and the device's memory
replaced; on the GPU whole rollouts whose tape's allocation fails."""

import numpy as np
import pytest
import torch

from swarp_amd import autograd
from swarp_amd.autograd import _tape_buffer

GiB = 1 << 30


class _Memory:
    """Stands in for the allocator: allocations above `most` bytes fail, `free` is what the
    device reports."""

    def __init__(self, monkeypatch, most, free):
        self.asked = []
        empty = torch.empty

        def fake(*shape, **kw):
            if kw.get("dtype") is not torch.uint8:
                return empty(*shape, **kw)
            self.asked.append(shape[0])
            if shape[0] > most:
                raise torch.OutOfMemoryError("no memory")
            return empty(*shape, **kw) if shape[0] < GiB else empty(1, **kw).expand(shape[0])

        monkeypatch.setattr(torch, "empty", fake)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (free, 288 * GiB))
        monkeypatch.setattr(torch.cuda, "memory_reserved", lambda dev: 5 * GiB)
        monkeypatch.setattr(torch.cuda, "memory_allocated", lambda dev: 4 * GiB)


@pytest.mark.parametrize("sizes,most,free,want", [
    ((1000, 10), 10**6, 0, 1000),             # small ones are not weighed
    ((1000, 10), 100, 0, 10),                 # the allocation fails: the records alone
    ((1000, 10), 5, 0, None),
    ((0,), 10**6, 0, None),
    ((2 * GiB,), 99 * GiB, 15 * GiB, 2 * GiB),     # an eighth of 15 + 1 free
    ((2 * GiB,), 99 * GiB, 15 * GiB - 8, None),
    ((2 * GiB, 10), 99 * GiB, 4 * GiB, 10),
])
def test_choice_of_a_buffer(monkeypatch, sizes, most, free, want):
    mem = _Memory(monkeypatch, most, free)
    got = _tape_buffer(sizes, "cpu")
    assert (None if got is None else got.numel()) == want
    assert want is None or mem.asked[-1] == want


def _no_memory_above(monkeypatch, most):
    empty = torch.empty

    def fake(*shape, **kw):
        if kw.get("dtype") is torch.uint8 and shape[0] > most:
            raise torch.OutOfMemoryError("no memory")
        return empty(*shape, **kw)

    monkeypatch.setattr(autograd.torch, "empty", fake)


@pytest.mark.gpu
def test_swarm_without_memory_for_its_tape(monkeypatch):
    from hip_helpers import hip_run, make_stepper
    from oracle.oracle import pack_state
    from swarp_amd.config import AgentConfig, WorldConfig

    E, A, T = 2, 80, 3
    rng = np.random.default_rng(0)
    s0 = pack_state({"pos": rng.uniform(-1, 1, size=(E, A, 2))}).astype(np.float32)
    acts = rng.uniform(-1, 1, size=(T, E, A, 2)).astype(np.float32)
    w = rng.normal(size=(T, E, A, 16))
    w[..., 7:] = 0.0
    world = WorldConfig(collision_k=100.0, collision_c=1.0, collision_margin=0.025,
                        bounds=(-1.0, 1.0, -1.0, 1.0), max_neighbors=16)
    st = make_stepper([AgentConfig(radius=0.05) for _ in range(A)], world, 0.05, 2, torch.float32)
    assert st.tape_bytes(E, 2, T) > 0
    a = hip_run(st, s0, acts, w, np.float32)
    _no_memory_above(monkeypatch, 0)
    b = hip_run(st, s0, acts, w, np.float32)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("keeps", ["records", "nothing"])
def test_bodies_without_memory_for_their_tape(monkeypatch, keeps):
    from cases import nav_agents
    from hip_helpers import make_stepper
    from test_hip_v_bodies import _pushers, _world, cross_obs, hip_body_run

    E, A, S, td = 3, 20, 2, torch.float32
    s0, acts = _pushers(E, A, 7, spread=0.8)
    runs = []
    for short in (False, True):
        st = make_stepper(nav_agents(A), _world(), 0.05, S, td, obs=cross_obs(E, (0.0, 0.0)),
                          n_envs=E)
        full, records = st.ob_tape_sizes(E, 2, acts.shape[0])
        if short:
            _no_memory_above(monkeypatch, records if keeps == "records" else 0)
        runs.append(hip_body_run(st, s0, acts, td, seed=3)[0])
    for x, y in zip(*runs):
        assert np.array_equal(x, y)
