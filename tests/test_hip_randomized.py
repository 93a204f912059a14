"""Per-env parameter rows on the specialised holonomic kernels: every env steps with its own
masses, speeds and radii.  States bit-exact with the oracle run env by env and with the
generic kernels; gradients within the parity bar of the oracle's."""

import numpy as np
import pytest
import torch

from cases import nav_agents, nav_world, oracle_cfg, params_of
from hip_helpers import hip_run, make_stepper, rel
from oracle.oracle import Oracle, pack_state
from swarp_amd import per_env_float_template

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,A,T,S,dtype", [
    (7, 16, 6, 4, np.float32),   # a partial last wave, the row-rotation scan
    (5, 13, 5, 1, np.float32),   # padded slots
    (9, 4, 4, 2, np.float32),
    (3, 32, 4, 5, np.float32),   # more substeps than the tape keeps
    (2, 64, 4, 4, np.float32),
    (6, 10, 4, 3, np.float64),
])
def test_per_env_rows(E, A, T, S, dtype):
    rng = np.random.default_rng(10 * E + A)
    cfgs = nav_agents(A)
    # radii up to the template's, so that the world's neighbour radius covers every env
    world = nav_world(A, world_size=0.6)
    rows = np.array(per_env_float_template(cfgs, E))
    rows[..., 0] *= rng.uniform(0.5, 1.0, size=(E, A))
    rows[..., 1] = rng.uniform(0.5, 2.0, size=(E, A))
    rows[..., 2] = rng.uniform(0.4, 1.0, size=(E, A))
    rows = rows.astype(dtype).astype(np.float64)
    s0 = pack_state({"pos": rng.uniform(-0.6, 0.6, size=(E, A, 2)),
                     "vel": rng.uniform(-0.3, 0.3, size=(E, A, 2))}).astype(dtype)
    acts = rng.uniform(-1, 1, size=(T, E, A, 2)).astype(dtype)
    w = rng.normal(size=(T, E, A, 16))
    w[..., 7:] = 0.0
    td = torch.float32 if dtype == np.float32 else torch.float64
    out = []
    for specialised in (True, False):
        st = make_stepper(cfgs, world, 0.05, S, td)
        st.use_specialised = specialised
        st.set_agent_params_per_env(rows)
        assert st.desc(E, 2).holo_velocity_only == int(specialised)
        out.append(hip_run(st, s0, acts, w, dtype))
    assert np.array_equal(out[0][0][..., :7], out[1][0][..., :7]), "states differ from the generic kernels'"
    O = Oracle(dtype)
    p, t, m = params_of(cfgs)
    for e in range(E):
        cfg = oracle_cfg(cfgs, world, 0.05, S, 1, 2)
        one = lambda x, ax: np.ascontiguousarray(np.take(x, [e], axis=ax))  # noqa: E731
        states = O.rollout(cfg, rows[e].astype(dtype), t, m, None, one(s0, 0), one(acts, 1))
        g0, ga = O.rollout_adj(cfg, rows[e].astype(dtype), t, m, None, one(s0, 0), one(acts, 1),
                               states, one(w, 1), None)
        hs, hg0, hga = out[0][0][:, e:e + 1], out[0][1][e:e + 1], out[0][2][:, e:e + 1]
        if dtype == np.float32:
            assert np.array_equal(hs[..., :7], states[..., :7].astype(np.float64)), f"env {e}"
        else:
            assert rel(hs[..., :7], states[..., :7]) <= 1e-12
        tol = 1e-5 if dtype == np.float32 else 1e-12
        assert rel(hga, ga) <= tol and rel(hg0[..., :7], g0[..., :7]) <= tol, f"env {e}"
