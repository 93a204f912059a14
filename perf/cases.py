"""What a user of the simulator runs, as cases that can be timed and compared.

A case is one pass through the public entry points:

* ``train``  a BPTT rollout: ``rollout`` over T env steps, a loss, ``backward`` -- forward and
  backward of the physics step.  ``fleet`` says what is stepped: ``holonomic`` point agents
  between soft walls (the navigation worlds), ``mixed`` differential-drive and bicycle agents
  among static circles, boxes and segments, ``drone`` quadrotors, ``body`` agents pushing a
  movable compound body with neighbour lists, overflow flags and the COO graph of every step;
* ``env``    one no-grad ``Environment.step`` of the navigation scenario (step, lists,
  observations, reward): what a policy's sampling loop calls;
* ``graph``  the radius graph of a state: ``NeighborGrid.build``, ``overflow_view``,
  ``edge_index`` -- what a graph policy asks for between steps.

Sizes are those of the repository's benchmark workloads (``bench.py``), of its throughput
table (``swarp_amd/throughput.py``) and of its tests, with odd ones beside them; ``draw``
spreads over the same ranges.
"""

import math

import numpy as np
import torch

from swarp_amd import (
    AgentConfig,
    DynamicsModel,
    Environment,
    NavigationScenario,
    NeighborGrid,
    Obstacles,
    Stepper,
    TorchState,
    WorldConfig,
    per_env_float_template,
    rollout,
)

DEV = "cuda:0"
R = 0.05                       # agent radius of the 2-D fleets
K_CONTACT, C_CONTACT = 100.0, 1.0
EPS2 = 1.0e-10                 # the contact law's smallest squared distance
BODY_OFFSETS = ((0.0, 0.0), (0.2, 0.0), (-0.2, 0.0), (0.0, 0.2), (0.0, -0.2))
BODY_R, BODY_MASS = 0.1, 1.0


def listed():
    return [
        # a policy's sampling loop at the smallest size of the throughput table: launch latency
        {"name": "env_1000x4", "kind": "env", "envs": 1000, "agents": 4, "half": 1.0},
        # the same loop at the table's largest size: lists and observations written to memory
        {"name": "env_16000x64", "kind": "env", "envs": 16000, "agents": 64, "half": 2.0},
        # the smallest training call (64 envs x 4 agents, 10 steps): host and launch latency
        _train("train_64x4", "holonomic", 64, 4, 10, 1, 1.0),
        # the benchmark workload: 16000 envs x 16 agents, 4 substeps, 32-step BPTT
        _train("train_16000x16", "holonomic", 16000, 16, 32, 4, 2.0),
        # odd sizes in float64 (gradient checking, system identification), padded agent slots
        _train("train_777x13_f64", "holonomic", 777, 13, 9, 3, 1.5, dtype="float64"),
        # domain randomization: a parameter row per env and agent, a loss over the whole path
        _train("train_3000x16_random", "holonomic", 3000, 16, 16, 4, 2.0, per_env=True,
               loss="path"),
        # mixed fleet among static obstacles, 20-step BPTT (benchmark workload)
        _train("train_4096x32_mixed", "mixed", 4096, 32, 20, 4, 2.0, obstacles=8),
        # quadrotors, 64-step BPTT (benchmark workload)
        _train("train_8192x8_drone", "drone", 8192, 8, 64, 1, 0.0),
        # agents pushing a movable body, lists and COO graph of every step (benchmark workload)
        _train("train_16000x64_body", "body", 16000, 64, 16, 4, 3.0),
        # swarms: more agents than a wavefront holds, index-ordered lists, loss over the path
        _train("train_500x200_swarm", "holonomic", 500, 200, 8, 4, 3.5, loss="path"),
        # large swarms: more than 512 agents, for which the lists follow the uniform grid
        _train("train_48x2000_swarm", "holonomic", 48, 2000, 8, 2, 11.0),
        # the radius graph of large swarms for a graph policy (uniform grid, frame from the batch)
        {"name": "graph_200x1000", "kind": "graph", "envs": 200, "agents": 1000, "half": 8.0,
         "radius": 0.4, "cap": 16},
    ]


def _train(name, fleet, envs, agents, steps, substeps, half, dtype="float32", per_env=False,
           loss="final", obstacles=0):
    c = {"kind": "train", "fleet": fleet, "envs": envs, "agents": agents, "steps": steps,
         "substeps": substeps, "half": half, "dtype": dtype, "per_env": per_env, "loss": loss,
         "obstacles": obstacles}
    return dict(c, name=name) if name else c


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("env", "holonomic", "holonomic", "mixed", "drone", "body", "swarm", "swarm",
                       "graph"))
    if kind == "env":
        A = _log(rng, 2, 64)
        return {"kind": "env", "envs": _log(rng, 50, 16000), "agents": A,
                "half": round(max(1.0, math.sqrt(A) / 4), 2)}
    if kind == "graph":
        A = _log(rng, 40, 3000)
        return {"kind": "graph", "envs": min(_log(rng, 4, 4000), 200000 // A), "agents": A,
                "half": round(math.sqrt(A) / 4, 2), "radius": round(rng.uniform(0.15, 0.45), 3),
                "cap": rng.choice((8, 16, 24, 32))}
    if kind == "holonomic":
        A, T, S = _log(rng, 2, 64), _log(rng, 1, 40), rng.choice((1, 1, 2, 3, 4, 4, 6))
        f64 = rng.random() < 0.25
        most = 16000 * 16 * 32 * 4 // (A * T * S * (4 if f64 else 1))
        return _train("", kind, max(1, min(_log(rng, 16, 16000), most)), A, T, S,
                      round(max(1.0, math.sqrt(A) / 3), 2), "float64" if f64 else "float32",
                      rng.random() < 0.3, rng.choice(("final", "path")))
    if kind == "mixed":
        A, T, S = _log(rng, 4, 64), _log(rng, 2, 20), rng.choice((1, 2, 4))
        most = 4096 * 32 * 20 * 4 // (A * T * S)
        return _train("", kind, max(1, min(_log(rng, 32, 4096), most)), A, T, S,
                      round(max(1.5, math.sqrt(A) / 3), 2), obstacles=rng.randint(1, 12))
    if kind == "drone":
        A, T, S = _log(rng, 2, 32), _log(rng, 2, 64), rng.choice((1, 1, 2))
        most = 8192 * 8 * 64 // (A * T * S)
        return _train("", kind, max(1, min(_log(rng, 32, 8192), most)), A, T, S, 0.0)
    if kind == "body":
        A, T, S = _log(rng, 6, 64), _log(rng, 2, 16), rng.choice((1, 2, 4))
        return _train("", kind, _log(rng, 64, 12000), A, T, S, 3.0)
    A, T, S = _log(rng, 65, 3000), _log(rng, 2, 10), rng.choice((1, 2, 4))
    most = 500 * 200 * 8 * 4 // (A * T * S)
    return _train("", "holonomic", max(1, min(_log(rng, 4, 1000), most)), A, T, S,
                  round(math.sqrt(A) / 4, 2), "float32", False, rng.choice(("final", "path")))


# ------------------------------------------------------------------------------- inputs


def _gen(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) + case["envs"] + case["agents"])

    def u(*shape, lo=-1.0, hi=1.0):
        return torch.rand(*shape, generator=g, device=DEV) * (hi - lo) + lo

    return g, u


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, u = _gen(case, seed)
    E, A, h = case["envs"], case["agents"], case["half"]
    dt = getattr(torch, case.get("dtype", "float32"))
    if case["kind"] == "graph":
        return {"pos": u(E, A, 2, lo=-h, hi=h)}
    if case["kind"] == "env":
        # the actions come back on themselves, so that the agents stay where they are however
        # often the loop goes round
        acts = [u(E, A, 2) for _ in range(8)]
        return {"pos": u(E, A, 2, lo=-h, hi=h), "goals": u(E, A, 2, lo=-h, hi=h),
                "theta": u(E, A, lo=-math.pi, hi=math.pi),
                "actions": acts + [-a for a in reversed(acts)]}
    T, fleet = case["steps"], case["fleet"]
    if fleet == "drone":
        # rotor thrusts over their range, attitudes within 0.1 rad of level, 1 m up
        ax = torch.randn(E, A, 3, generator=g, device=DEV)
        ax = ax / ax.norm(dim=-1, keepdim=True)
        ang = u(E, A, 1, lo=0.0, hi=0.1)
        w = math.sqrt(A) * 0.25
        return {"pos": u(E, A, 2, lo=-w, hi=w),
                "attitude": torch.cat([ax * torch.sin(ang / 2), torch.cos(ang / 2)], -1),
                "goals": u(E, A, 2), "actions": u(T, E, A, 4, lo=0.0, hi=10.0)}
    x = {"pos": u(E, A, 2, lo=-h, hi=h).to(dt), "goals": u(E, A, 2, lo=-h, hi=h).to(dt),
         "actions": u(T, E, A, 2).to(dt)}
    if case["per_env"]:
        x["mass"] = u(E, A, lo=0.8, hi=1.25).to(dt)
        x["max_speed"] = u(E, A, lo=0.5, hi=1.0).to(dt)
    if fleet == "mixed":
        N = case["obstacles"]
        shape = [(0, 1, 0, 2)[k % 4] for k in range(N)]
        # shared extents, per-env poses: circles, axis-aligned boxes, segments of any angle
        rc, bx, sl = u(N, lo=0.05, hi=0.2), u(N, 2, lo=0.05, hi=0.3), u(N, lo=0.1, hi=0.4)
        t = torch.tensor(shape, device=DEV)
        zero = torch.zeros_like(rc)
        x.update(
            theta=u(E, A, lo=-math.pi, hi=math.pi), o_type=t, o_pos=u(E, N, 2, lo=-h, hi=h),
            o_rad=torch.where(t == 0, rc, torch.where(t == 2, zero + 0.02, zero)),
            o_half=torch.where((t == 1).unsqueeze(-1), bx,
                               torch.where((t == 2).unsqueeze(-1), torch.stack([sl, zero], -1),
                                           torch.zeros_like(bx))),
            o_ang=u(E, N, lo=-math.pi, hi=math.pi) * (t == 2))
    if fleet == "body":
        x["goals"] = u(E, 2, lo=-2.0, hi=2.0)
    return x


def _world(case):
    """Constants of the case's world: what its WorldConfig holds."""
    E, A, h = case["envs"], case["agents"], case["half"]
    if case.get("fleet") == "drone":
        return dict(r=0.1, margin=0.02, dt=0.02, bounds=None, reach=0.22, cap=32)
    w = dict(r=R, margin=0.5 * R, dt=0.05, bounds=(-h, h, -h, h), reach=2.5 * R,
             cap=min(32, max(4, A)))
    if case.get("fleet") == "body":
        w.update(reach=0.3, cap=16)
    return w


def _near(A, radius, half):
    """Agents within the radius of an agent, on average."""
    return A * math.pi * radius ** 2 / (2 * half) ** 2


def _edge_buffer(rows, cap, near):
    """The fixed-size buffer a batched consumer takes a graph in (unused columns are -1)."""
    return torch.full((2, int(rows * min(cap, 2 * near + 3))), -1, dtype=torch.int64, device=DEV)


def _into(buf, edges):
    buf[:, :edges.shape[1]] = edges
    return buf


def _inertia():
    m = BODY_MASS / len(BODY_OFFSETS)
    return sum(0.5 * m * BODY_R ** 2 + m * (a * a + b * b) for a, b in BODY_OFFSETS)


# ------------------------------------------------------------------------------ the cases


def prepare(case, seed):
    x, w = _inputs(case, seed), _world(case)
    E, A = case["envs"], case["agents"]
    if case["kind"] == "graph":
        return {"case": case, "pos": x["pos"],
                "edges": _edge_buffer(E * A, case["cap"], _near(A, case["radius"], case["half"])),
                "grid": NeighborGrid(E, A, radius=case["radius"], max_neighbors=case["cap"],
                                     device=DEV)}
    if case["kind"] == "env":
        env = Environment(NavigationScenario(n_agents=A, world_size=case["half"]), n_envs=E,
                          device=DEV, dt=0.05, substeps=1, seed=0)
        env.reset(seed=0)
        env.world.write_state(pos=x["pos"], theta=x["theta"])
        env.world.goals.copy_(x["goals"])
        with torch.no_grad():
            env.step(torch.zeros_like(x["actions"][0]))
        return {"case": case, "env": env, "actions": x["actions"], "at": 0}
    fleet = case["fleet"]
    if fleet == "mixed":
        cfgs = [AgentConfig(model=DynamicsModel.DIFF_DRIVE if k < A // 2
                            else DynamicsModel.KINEMATIC_BICYCLE, radius=R) for k in range(A)]
    elif fleet == "drone":
        cfgs = [AgentConfig(model=DynamicsModel.DRONE, radius=w["r"]) for _ in range(A)]
    else:
        cfgs = [AgentConfig(radius=R, max_speed=1.0, max_accel=2.0) for _ in range(A)]
    world = WorldConfig(collision_k=K_CONTACT, collision_c=C_CONTACT, collision_margin=w["margin"],
                        bounds=w["bounds"], bounds_mode="soft", neighbor_radius=w["reach"],
                        max_neighbors=w["cap"])
    dtype = getattr(torch, case["dtype"])
    st = Stepper(cfgs, dt=w["dt"], substeps=case["substeps"], device=DEV, dtype=dtype, world=world)
    if case["per_env"]:
        table = torch.from_numpy(np.ascontiguousarray(per_env_float_template(cfgs, E)))
        table[..., 1], table[..., 2] = x["mass"].double().cpu(), x["max_speed"].double().cpu()
        st.set_agent_params_per_env(table)
    if fleet == "mixed":
        st.set_obstacles(Obstacles(pos=x["o_pos"], radius=x["o_rad"], shape=x["o_type"].int(),
                                   angle=x["o_ang"], half_extents=x["o_half"]))
    s = {"case": case, "stepper": st, "goals": x["goals"]}
    if fleet == "body":
        n = len(BODY_OFFSETS)
        offs = torch.tensor(BODY_OFFSETS, device=DEV)
        st.set_obstacles(Obstacles(
            pos=offs.expand(E, n, 2).contiguous(), radius=torch.full((n,), BODY_R),
            kind=torch.ones(n, dtype=torch.int32), body=torch.zeros(n, dtype=torch.int32),
            mass=torch.full((n,), BODY_MASS), inertia=torch.full((n,), _inertia()),
            body_offset=offs))
        s.update(ob0=st.ob_state.clone(), grid=st.grid(E),
                 edges=[_edge_buffer(E * A, w["cap"], _near(A, w["reach"], case["half"]))
                        for _ in range(case["steps"])])
    z = torch.zeros(E, A, device=DEV, dtype=dtype)
    z2 = torch.zeros(E, A, 2, device=DEV, dtype=dtype)
    theta = x["theta"] if "theta" in x else z.clone()
    pos = x["pos"].clone().requires_grad_(True)
    tail = ()
    if fleet == "drone":
        tail = (torch.ones_like(z), z.clone(), x["attitude"], torch.zeros(E, A, 3, device=DEV))
    s.update(state=TorchState(pos, theta, z2, z.clone(), z.clone(), *tail),
             actions=x["actions"].clone().requires_grad_(True))
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "graph":
        g = s["grid"]
        g.build(s["pos"])
        over = g.overflow_view()
        idx, cnt = g.torch_views()
        return {"idx": idx, "count": cnt, "overflow": over,
                "edges": _into(s["edges"], g.edge_index())}
    if case["kind"] == "env":
        with torch.no_grad():
            a = s["actions"][s["at"] % len(s["actions"])]
            s["at"] += 1
            obs, reward, terminated, truncated, info = s["env"].step(a)
        return {"obs": obs, "reward": reward, "terminated": terminated, "truncated": truncated,
                "info": info}
    st, s0, a, goals = s["stepper"], s["state"], s["actions"], s["goals"]
    a.grad = s0.pos.grad = None
    if case["fleet"] == "body":
        return _run_body(s)
    final, traj = rollout(st, s0, a)
    out = {"pos": final.pos, "theta": final.theta, "vel": final.vel, "speed": final.speed,
           "ang_vel": final.ang_vel}
    if case["loss"] == "path":
        loss = sum(((x.pos - goals) ** 2).sum() for x in traj)
        out["path"] = [x.pos for x in traj]
    else:
        loss = ((final.pos - goals) ** 2).sum()
    if case["fleet"] == "drone":
        loss = loss + ((final.z - 1.0) ** 2).sum()
        out.update(z=final.z, vz=final.vz, attitude=final.attitude, body_rates=final.body_rates)
    loss.backward()
    return dict(out, loss=loss, d_actions=a.grad, d_pos=s0.pos.grad)


def _run_body(s):
    st, s0, a, grid = s["stepper"], s["state"], s["actions"], s["grid"]
    n = len(BODY_OFFSETS)
    ob = st.ob_state = s["ob0"].clone().requires_grad_(True)
    final, traj = rollout(st, s0, a)
    body = st.ob_trajectory[-1][:, 6 * n:6 * n + 2]
    loss = ((body - s["goals"]) ** 2).sum()
    edges, over = [], []
    with torch.no_grad():
        for x, buf in zip(traj, s["edges"]):
            grid.build(x.pos)
            over.append(grid.overflow_view())
            edges.append(_into(buf, grid.edge_index()))
    loss.backward()
    return {"pos": final.pos, "vel": final.vel, "speed": final.speed, "bodies": st.ob_trajectory,
            "edges": edges, "overflow": over, "loss": loss, "d_actions": a.grad,
            "d_pos": s0.pos.grad, "d_bodies": ob.grad}


def work(case):
    """Bytes: every input read once, every output written once (a rollout's outputs are the
    states after each of its steps and the gradients).  Operations: membership of each pair
    that a cell search cannot rule out, the contact and integration arithmetic of one agent
    and substep, twice that for the reverse."""
    E, A = case["envs"], case["agents"]
    EA = E * A
    pairs = min(A - 1, 16)
    if case["kind"] == "graph":
        edges = EA * min(case["cap"], _near(A, case["radius"], case["half"]))
        return {"bytes": EA * (8 + 4 * case["cap"] + 8 + 1) + 16 * edges, "flops": 6.0 * EA * pairs}
    if case["kind"] == "env":
        # state, action, goal, baseline in; state, lists, observations, reward terms out
        return {"bytes": EA * 4 * (7 + 2 + 2 + 1 + 7 + min(32, max(4, A)) + 19 + 8),
                "flops": EA * (6.0 * pairs + 100)}
    T, S = case["steps"], case["substeps"]
    item = 8 if case["dtype"] == "float64" else 4
    sf, ad = (16, 4) if case["fleet"] == "drone" else (7, 2)
    b = EA * item * (T * (2 * ad + sf) + 3 * sf)
    ops = 6.0 * pairs * T + 3 * T * S * (120 if case["fleet"] == "drone" else 40)
    if case["per_env"]:
        b += EA * item * 22
    if case["fleet"] == "mixed":
        b += E * case["obstacles"] * 24
        ops += 30.0 * T * S * case["obstacles"]
    if case["fleet"] == "body":
        edges = min(16.0, _near(A, 0.3, case["half"]))
        b += T * E * 4 * 12 * len(BODY_OFFSETS) + T * EA * (1 + 4 * 18 + 16 * edges)
        ops += 40.0 * T * S * len(BODY_OFFSETS)
    return {"bytes": float(b), "flops": EA * ops}


def tolerance(case):
    if case["kind"] == "graph":
        return "exact"
    if case["kind"] == "env":
        # float32 steps of + - * / sqrt; cos and sin of the heading to an ulp
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-5}
    if case["dtype"] == "float64":
        return {"rel": 1e-11}
    # Float32 against 64 bits: states 1e-6, gradients up to 3e-3 over a long chain of substeps
    # (1.6e-3 over a shorter one) -- a contact that begins a rounding earlier or later turns the
    # gradient of its two agents, and every later substep carries it on.
    return {"rel": 1.2e-2 if case["steps"] * case["substeps"] > 48 else 6e-3, "differ": 1e-5}


# ----------------------------------------------------------------- the same in 64 bits


def _law(d, rv, md, dd):
    """Soft contact: force on self at offset d = self - other, relative velocity rv."""
    d2 = (d * d).sum(-1)
    dist = d2.clamp_min(EPS2).sqrt()
    n = d / dist.unsqueeze(-1)
    coef = ((K_CONTACT * (md - dist) - C_CONTACT * (rv * n).sum(-1)) / dd).clamp_min(0.0)
    return torch.where((md - dist > 0).unsqueeze(-1), coef.unsqueeze(-1) * n, torch.zeros_like(n))


def _agent_pairs(p, v, w, dd, radius):
    """Contact forces of the agents on each other: only pairs that touch exert any, found by
    sorting along x."""
    E, A = p.shape[:2]
    md = 2 * radius + w["margin"]
    with torch.no_grad():
        xs, order = p[..., 0].sort(dim=1)
        ys = p[..., 1].gather(1, order)
        ei, ii, jj = [], [], []
        for k in range(1, A):
            near = xs[:, k:] - xs[:, :-k] < md
            if k % 8 == 1 and not bool(near.any()):
                break
            e, a = (near & ((ys[:, k:] - ys[:, :-k]).abs() < md)).nonzero(as_tuple=True)
            ei.append(e)
            ii.append(order[e, a])
            jj.append(order[e, a + k])
        if not ei:
            return torch.zeros_like(p)
        e, i, j = torch.cat(ei), torch.cat(ii), torch.cat(jj)
    fi = _law(p[e, i] - p[e, j], v[e, i] - v[e, j], md, torch.ones((), device=DEV, dtype=p.dtype))
    out = torch.zeros_like(p)
    out = out.index_put((e, i), fi / dd[e, i].unsqueeze(-1), accumulate=True)
    return out.index_put((e, j), -fi / dd[e, j].unsqueeze(-1), accumulate=True)


def _walls(p, v, w, dd, radius):
    if w["bounds"] is None:
        return 0.0
    x0, x1, y0, y1 = w["bounds"]
    lo, hi = p.new_tensor([x0, y0]), p.new_tensor([x1, y1])
    reach, ddv = radius + w["margin"], dd.unsqueeze(-1)

    def side(pen, vn):
        c = ((K_CONTACT * pen - C_CONTACT * vn) / ddv).clamp_min(0.0)
        return torch.where(pen > 0, c, torch.zeros_like(c))

    return side(reach - (p - lo), v) - side(reach - (hi - p), -v)


def _obstacles(p, v, w, dd, x):
    """Static circles, boxes and segments (capsules), all still."""
    f, reach = 0.0, R + w["margin"]
    for o, ty in enumerate(x["o_type"].tolist()):
        c, ro = x["o_pos"][:, None, o].double(), float(x["o_rad"][o])
        hx, hy = (float(t) for t in x["o_half"][o])
        if ty == 0:
            f = f + _law(p - c, v, reach + ro, dd)
            continue
        a = x["o_ang"][:, None, o].double()
        ca, sa = a.cos(), a.sin()
        d = p - c
        if ty == 2:
            u = torch.stack([ca, sa], -1)
            t = (d * u).sum(-1).clamp(-hx, hx)
            f = f + _law(d - t.unsqueeze(-1) * u, v, reach + ro, dd)
            continue
        lx, ly = ca * d[..., 0] + sa * d[..., 1], -sa * d[..., 0] + ca * d[..., 1]
        ox, oy = lx - lx.clamp(-hx, hx), ly - ly.clamp(-hy, hy)
        out = ox * ox + oy * oy > EPS2
        one = torch.ones_like(lx)
        s_out = torch.where(out, ox * ox + oy * oy, one).sqrt()
        qx, qy = lx.abs() - hx, ly.abs() - hy
        xf = qx > qy
        sx, sy = torch.where(lx >= 0, one, -one), torch.where(ly >= 0, one, -one)
        s = torch.where(out, s_out, torch.where(xf, qx, qy))
        nlx = torch.where(out, ox / s_out, torch.where(xf, sx, 0 * one))
        nly = torch.where(out, oy / s_out, torch.where(xf, 0 * one, sy))
        n = torch.stack([ca * nlx - sa * nly, sa * nlx + ca * nly], -1)
        coef = ((K_CONTACT * (reach - s) - C_CONTACT * (v * n).sum(-1)) / dd).clamp_min(0.0)
        f = f + torch.where((reach - s > 0).unsqueeze(-1), coef.unsqueeze(-1) * n,
                            torch.zeros_like(n))
    return f


def _clamp_norm(a, lim):
    n = (a * a).sum(-1)
    over = n > lim * lim
    s = torch.where(over, lim / torch.where(over, n, torch.ones_like(n)).sqrt(), torch.ones_like(n))
    return a * s.unsqueeze(-1)


def _holonomic(s, a, f, h, x):
    mass = x["mass"].double() if "mass" in x else torch.ones_like(s["theta"])
    lim = x["max_speed"].double() if "max_speed" in x else torch.ones_like(s["theta"])
    vel = _clamp_norm(a, lim) + f * (h / mass).unsqueeze(-1)
    sq = (vel * vel).sum(-1)
    still = sq == 0
    speed = torch.where(still, torch.zeros_like(sq), torch.where(still, torch.ones_like(sq), sq).sqrt())
    return dict(s, pos=s["pos"] + vel * h, vel=vel, speed=speed, ang_vel=torch.zeros_like(speed))


def _mixed(s, a, f, h):
    A = a.shape[1]
    dd, bi = slice(0, A // 2), slice(A // 2, A)
    th = s["theta"]
    sd = a[:, dd, 0].clamp(-1.0, 1.0)
    wd = a[:, dd, 1].clamp(-math.pi, math.pi)
    steer = a[:, bi, 1].clamp(-math.pi / 4, math.pi / 4)
    sb = (s["speed"][:, bi] + a[:, bi, 0].clamp(-1.0, 1.0) * h).clamp(-1.0, 1.0)
    beta = torch.atan(torch.tan(steer) * 0.5)  # l_r / (l_f + l_r), both 0.1
    wb = sb / 0.2 * torch.cos(beta) * torch.tan(steer)
    speed, turn = torch.cat([sd, sb], 1), torch.cat([wd, wb], 1)
    head = torch.cat([th[:, dd], th[:, bi] + beta], 1)
    vel = speed.unsqueeze(-1) * torch.stack([head.cos(), head.sin()], -1) + f * h
    return dict(s, pos=s["pos"] + vel * h, theta=th + turn * h, vel=vel, speed=speed, ang_vel=turn)


def _drone(s, a, f, h):
    f0, f1, f2, f3 = a.clamp(0.0, 10.0).unbind(-1)
    thrust = f0 + f1 + f2 + f3
    qx, qy, qz, qw = s["attitude"].unbind(-1)
    acc = torch.stack([2 * (qx * qz + qw * qy) * thrust, 2 * (qy * qz - qw * qx) * thrust,
                       thrust - 2 * (qx * qx + qy * qy) * thrust - 9.81], -1)
    bx, by, bz = s["body_rates"].unbind(-1)
    b = torch.stack([bx + (0.15 * (f1 - f3) - 0.01 * by * bz) / 0.01 * h,
                     by + (0.15 * (f2 - f0) + 0.01 * bz * bx) / 0.01 * h,
                     bz + 0.02 * (f0 - f1 + f2 - f3) / 0.02 * h], -1)
    nx, ny, nz = b.unbind(-1)
    q = s["attitude"] + 0.5 * h * torch.stack([
        qw * nx + qy * nz - qz * ny, qw * ny - qx * nz + qz * nx,
        qw * nz + qx * ny - qy * nx, -qx * nx - qy * ny - qz * nz], -1)
    vel, vz = s["vel"] + acc[..., :2] * h + f * h, s["vz"] + acc[..., 2] * h
    return dict(s, pos=s["pos"] + vel * h, vel=vel, z=s["z"] + vz * h, vz=vz, body_rates=b,
                attitude=q / q.norm(dim=-1, keepdim=True))


def _body(p, v, dd, ob, h):
    """Forces of the compound body's circles on the agents and the body's own substep.
    `ob` [E, 12 N]: per shape its pose and velocity, then the state of the body rooted there."""
    n = len(BODY_OFFSETS)
    E = p.shape[0]
    shapes, bodies = ob[:, :6 * n].view(E, n, 6), ob[:, 6 * n:].view(E, n, 6)
    off, md = ob.new_tensor(BODY_OFFSETS), 2 * R + BODY_R + 0.5 * R - R
    b = bodies[:, 0]

    def install(c, th, vel, om):
        ca, sa = th.cos().unsqueeze(-1), th.sin().unsqueeze(-1)
        w = torch.stack([ca * off[:, 0] - sa * off[:, 1], sa * off[:, 0] + ca * off[:, 1]], -1)
        r = torch.stack([-w[..., 1], w[..., 0]], -1)
        return w, c.unsqueeze(1) + w, vel.unsqueeze(1) + om[:, None, None] * r

    f = sum(_law(p - shapes[:, None, k, :2], v - shapes[:, None, k, 3:5], md, dd) for k in range(n))
    w, c, cv = install(b[:, :2], b[:, 2], b[:, 3:5], b[:, 5])
    react = torch.stack([-_law(p - c[:, None, k], v - cv[:, None, k], md, dd).sum(1)
                         for k in range(n)], 1)
    tau = (w[..., 0] * react[..., 1] - w[..., 1] * react[..., 0]).sum(1)
    decay = 1.0 - 10.0 * h
    vel = (b[:, 3:5] + react.sum(1) / BODY_MASS * h) * decay
    om = (b[:, 5] + tau / _inertia() * h) * decay
    c2, th2 = b[:, :2] + vel * h, b[:, 2] + om * h
    _, sc, sv = install(c2, th2, vel, om)
    ones = torch.ones(E, n, 1, device=DEV, dtype=ob.dtype)
    new = torch.cat([sc, th2[:, None, None] * ones, sv, om[:, None, None] * ones], -1)
    root = torch.cat([c2, th2.unsqueeze(-1), vel, om.unsqueeze(-1)], -1)
    nb = torch.cat([root.unsqueeze(1), bodies[:, 1:]], 1)
    return f, torch.cat([new.reshape(E, 6 * n), nb.reshape(E, 6 * n)], -1)


def _step(s, a, case, w, x, substeps):
    h = w["dt"] / substeps
    mass = x["mass"].double() if "mass" in x else torch.ones_like(s["theta"])
    dd = 1.0 + C_CONTACT * h / mass
    for _ in range(substeps):
        p, v = s["pos"], s["vel"]
        f = _agent_pairs(p, v, w, dd, w["r"]) + _walls(p, v, w, dd, w["r"])
        if "o_type" in x:
            f = f + _obstacles(p, v, w, dd, x)
        ob = s.get("ob")
        if ob is not None:
            fo, ob = _body(p, v, dd, ob, h)
            f = f + fo
        fleet = case.get("fleet", "holonomic")
        if fleet == "mixed":
            s = _mixed(s, a, f, h)
        elif fleet == "drone":
            s = _drone(s, a, f, h)
        else:
            s = _holonomic(s, a, f, h, x)
        if ob is not None:
            s["ob"] = ob
    return s


def exact(case, seed):
    if case["kind"] == "graph":
        return None  # whole numbers
    x, w = _inputs(case, seed), _world(case)
    z = torch.zeros(case["envs"], case["agents"], device=DEV, dtype=torch.float64)
    z2 = torch.zeros(*z.shape, 2, device=DEV, dtype=torch.float64)
    s = {"pos": x["pos"].double(), "theta": x["theta"].double() if "theta" in x else z, "vel": z2,
         "speed": z, "ang_vel": z}
    if case["kind"] == "env":
        with torch.no_grad():
            return _exact_env(case, x, w, s, z2)
    if case["fleet"] == "drone":
        s.update(z=z + 1.0, vz=z, attitude=x["attitude"].double(),
                 body_rates=torch.zeros(*z.shape, 3, device=DEV, dtype=torch.float64))
    pos = s["pos"] = s["pos"].requires_grad_(True)
    acts = x["actions"].double().requires_grad_(True)
    leaves = [acts, pos]
    if case["fleet"] == "body":
        off = z2.new_tensor(BODY_OFFSETS).float().double()
        n = len(BODY_OFFSETS)
        ob = torch.zeros(case["envs"], 12 * n, device=DEV, dtype=torch.float64)
        for k in range(n):
            ob[:, 6 * k:6 * k + 2] = off[k]
        s["ob"] = ob.requires_grad_(True)
        leaves.append(ob)
    path, obs = [], []
    for a in acts:
        s = _step(s, a, case, w, x, case["substeps"])
        path.append(s["pos"])
        obs.append(s.get("ob"))
    goals = x["goals"].double()
    if case["fleet"] == "body":
        n6 = 6 * len(BODY_OFFSETS)
        loss = ((s["ob"][:, n6:n6 + 2] - goals) ** 2).sum()
    elif case["loss"] == "path":
        loss = sum(((p - goals) ** 2).sum() for p in path)
    else:
        loss = ((s["pos"] - goals) ** 2).sum()
    if case["fleet"] == "drone":
        loss = loss + ((s["z"] - 1.0) ** 2).sum()
    grads = torch.autograd.grad(loss, leaves)
    out = {"loss": loss, "d_actions": grads[0], "d_pos": grads[1]}
    if case["fleet"] == "body":
        return dict(out, pos=s["pos"], vel=s["vel"], speed=s["speed"], bodies=torch.stack(obs),
                    d_bodies=grads[2])
    out.update({k: v for k, v in s.items() if k != "ob"})
    if case["loss"] == "path":
        out["path"] = path
    return out


def _exact_env(case, x, w, s, zero):
    s = _step(s, zero, case, w, x, 1)
    before = (s["pos"] - x["goals"]).norm(dim=-1)
    s = _step(s, x["actions"][0].double(), case, w, x, 1)
    p, v, g = s["pos"], s["vel"], x["goals"].double()
    E, A = p.shape[:2]
    dist = (p - g).norm(dim=-1)
    d = ((p[:, :, None, 0] - p[:, None, :, 0]) ** 2 + (p[:, :, None, 1] - p[:, None, :, 1]) ** 2).sqrt()
    d.diagonal(dim1=1, dim2=2).fill_(math.inf)
    listed_ = d <= w["reach"]
    touch = (d < 2 * R).sum(-1).double()
    rows = [p, v, torch.stack([s["theta"].cos(), s["theta"].sin(), s["ang_vel"]], -1), g - p]
    rp, rv, ok = [], [], []
    first = torch.where(listed_, torch.arange(A, device=DEV), A).sort(-1).values[..., :2]
    for k in range(min(2, max(4, A))):
        if k < A:
            j = first[..., k]
        else:
            j = torch.full((E, A), A, device=DEV)
        there = (j < A).unsqueeze(-1)
        at = j.clamp_max(A - 1).unsqueeze(-1).expand(-1, -1, 2)
        rp.append((p.gather(1, at) - p) * there)
        rv.append((v.gather(1, at) - v) * there)
        ok.append(there.double())
    reward = -touch + (before - dist)
    goal = (dist < R).all(-1, keepdim=True)
    return {"obs": torch.cat(rows + rp + rv + ok, -1), "reward": reward + 5.0 * goal,
            "info": {"dist_to_goal": dist, "collisions": touch}}
