"""Timing cases of the MLS-MPM engine: what a user's program has it do.

frame     one step of a simulation program's loop, as the mpm program runs it:
          `Engine.advance` to the next saved frame (240 frames a second: 42
          substeps at dt = 1e-4, 83 at dt = 5e-5) and `Engine.download` of the
          particles that the frame is written from. Repeated passes go on from
          the state the last one left, as that loop does. With more substeps
          it stands for a program that saves less often.
batch     the same for many independent scenes at once (`Batch.advance`), as a
          parameter sweep or a data generator runs them.
rollout   `diff.rollout` of the differentiable substep: "grad" false is a
          forward run alone (evaluation), true a training step (a loss on the
          final positions, gradients of state, mu and lambda).
step      one differentiable substep and its adjoint through
          `DiffStepper.forward` / `.backward`, as a program with a time loop of
          its own calls them.
mesh      the surface mesh of one saved frame (`Engine.mesh`).

Inputs are states in the middle of a run: bodies that move with a swirl (a
rapid one for snow) and a shear, deformed by a few tenths of a per cent. The liquid starts undeformed
(F = I), as its scenes do. Sizes are those of mpm_amd.scenes' workloads and of
the benchmark, or lie in between.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mpm_amd import (BOUNDARY_CELLS, BOUNDARY_FRACTION, COMPAT_FIXED, COMPAT_REFERENCE,
                     MATERIAL_FIXED_COROTATED, MATERIAL_JELLY, MATERIAL_SNOW, MATERIAL_WC_LIQUID,
                     Batch, Engine, Params, make_material)
from mpm_amd.diff import DiffStepper, rollout

GRAVITY = -9.8
SCENES = ("elastic", "snow", "liquid", "mixed")


def listed():
    return [
        # the smallest scene (the benchmark's elastic sphere): every kernel of
        # a substep is a few microseconds, launches and latency count
        dict(name="frame_elastic_10k", kind="frame", scene="elastic", particles=10_000, N=16, substeps=42,
             sort_every=16),
        # an odd size with four materials in one scene, on a grid that the
        # 4^3 node blocks do not divide
        dict(name="frame_mixed_77k", kind="frame", scene="mixed", particles=77_773, N=45, substeps=42,
             sort_every=16),
        # the snow scene (two stacked spheres, ~45 particles a cell), a frame
        # with the engine's default sort interval
        dict(name="frame_snow_500k", kind="frame", scene="snow", particles=500_000, N=64, substeps=42,
             sort_every=16),
        # a dense elastic body at a longer sort interval
        dict(name="frame_elastic_200k", kind="frame", scene="elastic", particles=200_000, N=64, substeps=42,
             sort_every=32),
        # the dam break, the benchmark's headline scene: a frame of 83 substeps
        dict(name="frame_liquid_1m", kind="frame", scene="liquid", particles=1_000_000, N=128, substeps=83,
             sort_every=16),
        # the dam break run on, at its tuned sort interval
        dict(name="run_liquid_1m", kind="frame", scene="liquid", particles=1_000_000, N=128, substeps=1000,
             sort_every=48),
        # a sweep of independent scenes, sizes and grids mixed as in the
        # benchmark's batch; one frame of each
        dict(name="batch_24", kind="batch", scenes=24, max_particles=120_000, substeps=42, sort_every=16),
        # the differentiable elastic cube: a forward run, and a training step
        dict(name="rollout_32k", kind="rollout", side=32, N=32, substeps=100, every=20, grad=False),
        dict(name="rollout_grad_32k", kind="rollout", side=32, N=32, substeps=100, every=20, grad=True),
        # a training step on a small, ragged cube: launches count
        dict(name="rollout_grad_2k", kind="rollout", side=13, N=24, substeps=33, every=10, grad=True),
        # the smallest differentiable call: one substep and its adjoint
        dict(name="step_4k", kind="step", side=16, N=32),
        # a saved frame's surface at the mesher's default settings
        dict(name="mesh_liquid_1m", kind="mesh", scene="liquid", particles=1_000_000, N=128, side=250, radius=5),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frame", "frame", "frame", "batch", "rollout", "rollout", "step", "mesh"])
    if kind == "frame":
        scene = rng.choice(SCENES)
        n = log_int(3_000, 1_000_000)
        # 2 to 60 particles a cell of the body, which fills about a tenth of the box
        N = int(min(128, max(16, round((n / (0.1 * rng.uniform(2.0, 60.0))) ** (1 / 3)))))
        k = log_int(8, 400 if scene == "liquid" else 48)
        return dict(kind="frame", scene=scene, particles=n, N=N, substeps=k, sort_every=rng.choice([16, 32, 48, 96]))
    if kind == "batch":
        return dict(kind="batch", scenes=rng.randint(3, 24), max_particles=log_int(8_000, 120_000),
                    substeps=rng.randint(16, 48), sort_every=rng.choice([16, 24]))
    if kind == "rollout":
        side = rng.randint(6, 32)
        return dict(kind="rollout", side=side, N=rng.randint(16, 40), substeps=rng.randint(12, 100),
                    every=rng.randint(8, 24), grad=rng.random() < 0.6)
    if kind == "step":
        return dict(kind="step", side=rng.randint(6, 40), N=rng.randint(16, 48))
    n = log_int(10_000, 1_000_000)
    return dict(kind="mesh", scene=rng.choice(SCENES), particles=n, N=rng.choice([48, 64, 96, 128]),
                side=rng.randint(40, 250), radius=rng.randint(1, 5))


# ---------------------------------------------------------------- inputs

def _ball(rng, n, center, r):
    d = rng.standard_normal((n, 3), dtype=np.float32)
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-9)
    u = rng.random((n, 1), dtype=np.float32) ** (1.0 / 3.0)
    return np.asarray(center, np.float32) + np.float32(r) * u * d


def _box(rng, n, lo, hi):
    lo, hi = np.asarray(lo, np.float32), np.asarray(hi, np.float32)
    return lo + rng.random((n, 3), dtype=np.float32) * (hi - lo)


def _materials(volume):
    """Kind and constants of the scenes' materials, by name."""
    return {
        "elastic": dict(kind=MATERIAL_SNOW, volume=volume, density=1000.0, E=1e4, nu=0.3, hardening=0.0,
                        clamp_lo=0.0, clamp_hi=1e30),
        "snow": dict(kind=MATERIAL_SNOW, volume=volume, density=400.0, E=1.4e5, nu=0.2, hardening=10.0,
                     clamp_lo=1.0 - 2.5e-2, clamp_hi=1.0 + 7.5e-3),
        "liquid": dict(kind=MATERIAL_WC_LIQUID, volume=volume, density=1000.0, E=0.0, nu=0.0, hardening=0.0,
                       clamp_lo=0.0, clamp_hi=0.0, bulk_modulus=4e4),
        "jelly": dict(kind=MATERIAL_JELLY, volume=volume, density=1000.0, E=2e4, nu=0.3, hardening=10.0),
        "corotated": dict(kind=MATERIAL_FIXED_COROTATED, volume=volume, density=1000.0, E=2e4, nu=0.3,
                          hardening=0.0),
    }


def _scene(scene, n, N, rng):
    """A scene's parameters, material constants and particle arrays (float32)."""
    # (in the reference's mode, particles with an index past N^3 are held back)
    params = dict(dt=1e-4, N=N, gravity=GRAVITY, boundary_mode=BOUNDARY_FRACTION, boundary=0.05,
                  compat=COMPAT_REFERENCE if n <= N ** 3 else COMPAT_FIXED)
    mat = np.zeros(n, np.uint8)
    if scene == "elastic":
        x, volume, names = _ball(rng, n, (0.5, 0.5, 0.5), 0.15), 4 / 3 * math.pi * 0.15 ** 3, ["elastic"]
        params.update(boundary_mode=BOUNDARY_CELLS, boundary=3, compat=COMPAT_FIXED)
    elif scene == "snow":
        r1, r2 = 0.2, 0.13
        n1 = int(round(n * r1 ** 3 / (r1 ** 3 + r2 ** 3)))
        x = np.concatenate([_ball(rng, n1, (0.5, 0.32, 0.5), r1), _ball(rng, n - n1, (0.5, 0.64, 0.5), r2)])
        volume, names = 4 / 3 * math.pi * (r1 ** 3 + r2 ** 3), ["snow"]
    elif scene == "liquid":
        x, volume, names = _box(rng, n, (0.07, 0.07, 0.07), (0.47, 0.65, 0.93)), 0.4 * 0.58 * 0.86, ["liquid"]
        params.update(dt=5e-5)
    else:
        names = ["elastic", "snow", "liquid", "jelly", "corotated"]
        at = [(0.3, 0.3, 0.35), (0.7, 0.32, 0.36), (0.32, 0.34, 0.7), (0.68, 0.3, 0.68), (0.5, 0.68, 0.5)]
        count = [n // 5 + (i < n % 5) for i in range(5)]
        x = np.concatenate([_ball(rng, c, a, 0.14) for c, a in zip(count, at)])
        mat = np.repeat(np.arange(5, dtype=np.uint8), count)
        volume = 5 * 4 / 3 * math.pi * 0.14 ** 3
    known = _materials(volume / n)
    materials = [known[m] for m in names]
    # a swirl about the vertical axis and a shear, with their gradient as C
    w, s = {"snow": 6.0, "mixed": 3.0}.get(scene, 1.0) * (2.0 + rng.random()), 1.0 + rng.random()
    G = np.array([[0.3 * s, s, w], [0.2 * s, -0.5 * s, 0.1 * s], [-w, 0.3 * s, 0.2 * s]], np.float32)
    v = (x - np.float32(0.5)) @ G.T + np.array([0.1, -0.6, 0.05], np.float32)
    C = np.broadcast_to(G, (n, 3, 3)).copy()
    F = np.broadcast_to(np.eye(3, dtype=np.float32), (n, 3, 3)).copy()
    Jp = np.ones(n, np.float32)
    if scene != "liquid":
        solid = np.ones(n, bool) if scene != "mixed" else mat != 2
        for a in range(3):
            for b in range(3):
                wave = np.sin((11.0 + 3 * a + 2 * b) * x[:, b] + 5.0 * x[:, (b + 1) % 3] + a)
                F[:, a, b] += np.where(solid, (0.004 * wave).astype(np.float32), np.float32(0))
        Jp += np.where(solid, (0.01 * np.sin(17.0 * x[:, 1])).astype(np.float32), np.float32(0))
    return params, materials, dict(x=x, v=v.astype(np.float32), C=C, F=F, Jp=Jp, material=mat)


def _batch_scenes(case, rng):
    out = []
    for j in range(case["scenes"]):
        # sizes log-uniform from 5,000 to the largest, the same for every seed
        u = (0.5 + j * 0.6180339887) % 1.0
        n = int(round(5_000 * (case["max_particles"] / 5_000) ** u))
        out.append(_scene(("elastic", "snow", "liquid")[j % 3], n, (32, 48, 64)[j * 7 % 9 // 3], rng))
    return out


def _cube(case, seed):
    """The elastic cube: state planes (24, n), mu, lambda, target positions."""
    rng = np.random.default_rng(seed)
    side = case["side"]
    n, h = side ** 3, 0.3 / side
    g = (np.arange(side) + 0.5) * h + 0.35
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(n, 3)
    x = (x + (rng.random((n, 3)) - 0.5) * 0.5 * h).astype(np.float32)
    G = (rng.uniform(-1.5, 1.5, (3, 3)) + np.diag([0.5, -0.5, 0.3])).astype(np.float32)
    v = ((x - np.float32(0.5)) @ G.T + np.array([0.2, -0.5, 0.1])).astype(np.float32)
    C = np.broadcast_to(G, (n, 3, 3))
    F = (np.eye(3) + 0.01 * np.sin(9.0 * x[:, :, None] + 7.0 * x[:, None, :] + 1.0)).astype(np.float32)
    E = np.exp(math.log(1e4) + 0.1 * rng.standard_normal(n))
    st = np.concatenate([x.T, v.T, C.reshape(n, 9).T, F.reshape(n, 9).T]).astype(np.float32)
    mu, lam = (E / 2.6).astype(np.float32), (E * 0.3 / (1.3 * 0.4)).astype(np.float32)
    target = (x + 0.02 * np.sin(8.0 * x[:, ::-1])).T.astype(np.float32)
    volume = float(np.float32(h ** 3))
    mass = float(np.float32(1000.0) * np.float32(volume))
    params = dict(dt=1e-4, N=case["N"], gravity=GRAVITY, boundary_mode=BOUNDARY_FRACTION, boundary=0.05,
                  compat=COMPAT_FIXED)
    return params, mass, volume, n, dict(st=st, mu=mu, lam=lam, target=target)


# ---------------------------------------------------------------- the passes

def _engine(params, materials, p, sort_every):
    e = Engine(Params(**params))
    e.set_materials([make_material(**m) for m in materials])
    e.set_option("sort_every", sort_every)
    e.add_particles(p["x"], p["material"], p["v"], p["C"], p["F"], p["Jp"])
    e.upload()
    return e


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("frame", "mesh"):
        e = _engine(*_scene(case["scene"], case["particles"], case["N"], np.random.default_rng(seed)),
                    case.get("sort_every", 16))
        if kind == "mesh":
            e.advance(16)  # a frame is meshed after some substeps
            # the vertex buffer that a viewer keeps, empty past the last triangle
            return dict(case=case, engine=e, buffer=np.zeros((20 * case["side"] ** 2, 3, 3), np.float32), used=0)
        return dict(case=case, engine=e)
    if kind == "batch":
        engines = [_engine(*s, case["sort_every"]) for s in _batch_scenes(case, np.random.default_rng(seed))]
        return dict(case=case, engines=engines, batch=Batch(engines))
    params, mass, volume, n, p = _cube(case, seed)
    s = dict(case=case, stepper=DiffStepper(Params(**params), mass, volume, n))
    s.update({k: torch.from_numpy(a).cuda() for k, a in p.items()})
    if kind == "rollout" and case["grad"]:
        for k in ("st", "mu", "lam"):
            s[k].requires_grad_(True)
    if kind == "step":
        s["tape"] = s["stepper"].new_tape()
        s["out"], s["adj_in"] = torch.empty_like(s["st"]), torch.empty_like(s["st"])
        s["adj_mu"], s["adj_lam"] = torch.empty_like(s["mu"]), torch.empty_like(s["lam"])
        s["adj_out"] = _step_adjoint(s["st"])
    return s


def _step_adjoint(st):
    """The adjoint of a substep's result that a loss on all of it would give."""
    return torch.sin(3.0 * st + torch.arange(24, device=st.device, dtype=st.dtype)[:, None]).contiguous()


def _loss(st, target):
    return 100.0 * ((st[0:3] - target) ** 2).sum()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        state["engine"].advance(case["substeps"])
        return state["engine"].download()
    if kind == "batch":
        state["batch"].advance(case["substeps"])
        # one array of each kind over the scenes
        got = [e.download() for e in state["engines"]]
        return {k: np.concatenate([g[k] for g in got]) for k in got[0]}
    if kind == "mesh":
        tri, buf = state["engine"].mesh(case["side"], case["radius"])["triangles"], state["buffer"]
        n = tri.shape[0]
        buf[:n] = tri
        buf[n:state["used"]] = 0.0
        state["used"] = n
        return dict(triangles=buf, count=n)
    if kind == "rollout":
        st = rollout(state["stepper"], state["st"], state["mu"], state["lam"], case["substeps"], case["every"])
        if not case["grad"]:
            return dict(state=st)
        g = torch.autograd.grad(_loss(st, state["target"]), [state["st"], state["mu"], state["lam"]])
        return dict(state=st.detach(), grad_state=g[0], grad_mu=g[1], grad_lam=g[2])
    s = state
    s["adj_mu"].zero_()
    s["adj_lam"].zero_()
    s["stepper"].forward(s["st"], s["out"], s["mu"], s["lam"], s["tape"])
    s["stepper"].backward(s["st"], s["mu"], s["lam"], s["tape"], s["adj_out"], s["adj_in"], s["adj_mu"], s["adj_lam"])
    return dict(out=s["out"], adj_in=s["adj_in"], adj_mu=s["adj_mu"], adj_lam=s["adj_lam"])


def work(case):
    """Bytes: a substep reads and writes what a particle carries from one to
    the next (x, F, Jp, material; the liquid's F follows from Jp) and writes
    and reads the nodes its bodies cover; the state at the end goes to the
    caller. Operations: about 1,200 a particle and substep, and 1,300 more
    where the polar rotation is needed."""
    kind = case["kind"]
    if kind in ("frame", "batch"):
        k = case["substeps"]
        if kind == "frame":
            sizes = [(case["scene"], case["particles"], case["N"])]
        else:  # the mean of the log-uniform sizes
            hi, lo = case["max_particles"], 5_000
            mean = (hi - lo) / math.log(hi / lo)
            sizes = [(("elastic", "snow", "liquid")[j % 3], mean, 48) for j in range(case["scenes"])]
        b = f = 0.0
        for scene, n, N in sizes:
            covered = {"elastic": 0.02, "snow": 0.06, "liquid": 0.22, "mixed": 0.08}[scene]
            b += k * ((33 if scene == "liquid" else 105) * n + 2 * 16 * covered * N ** 3) + 101 * n
            f += k * (1200 if scene == "liquid" else 2500) * n
        return dict(bytes=b, flops=f)
    if kind == "mesh":
        v = case["side"] ** 3
        return dict(bytes=12 * case["particles"] + 8 * v + 60 * 6 * case["side"] ** 2,
                    flops=8 * (2 * case["radius"] + 3) ** 3 * case["particles"] * 0.5)
    n, nodes = case["side"] ** 3, 0.06 * case["N"] ** 3
    forward = 2 * 96 * n + 8 * n + 2 * 16 * nodes
    if kind == "step":
        return dict(bytes=forward + (4 * 96 + 24) * n + 2 * 16 * nodes, flops=(2500 + 6000) * n)
    k = case["substeps"]
    # the forward carries x and F; the backward needs each substep's state once
    # more and carries the adjoint
    b = k * (2 * 48 * n + 2 * 16 * nodes) + 2 * 96 * n
    if case["grad"]:
        b += k * (3 * 96 * n + 2 * 16 * nodes) + 2 * 96 * n
    return dict(bytes=b, flops=k * n * (2500 + (8500 if case["grad"] else 0)))


# ---------------------------------------------------------------- in 64 bits

def _f32(v):
    return float(np.float32(v))


def _det(m):
    return (m[:, 0, 0] * (m[:, 1, 1] * m[:, 2, 2] - m[:, 1, 2] * m[:, 2, 1]) -
            m[:, 0, 1] * (m[:, 1, 0] * m[:, 2, 2] - m[:, 1, 2] * m[:, 2, 0]) +
            m[:, 0, 2] * (m[:, 1, 0] * m[:, 2, 1] - m[:, 1, 1] * m[:, 2, 0]))


def _inv_t(m):
    """Inverse transpose of 3x3 matrices: the cofactors over the determinant."""
    r0, r1, r2 = m[:, 0], m[:, 1], m[:, 2]
    c = torch.stack([torch.linalg.cross(r1, r2), torch.linalg.cross(r2, r0), torch.linalg.cross(r0, r1)], 1)
    return c / (r0 * c[:, 0]).sum(1)[:, None, None]


def _rotation(F):
    """Polar rotation of F (det F > 0) by Newton's iteration."""
    R = F
    for _ in range(8):
        R = 0.5 * (R + _inv_t(R))
    return R


def _mm(a, b):
    return (a[:, :, :, None] * b[:, None, :, :]).sum(2)


def _clamp_stretch(F, lo, hi):
    """F = U s V^T with s clamped to [lo, hi], by Jacobi rotations on F^T F."""
    S = _mm(F.transpose(1, 2), F)
    V = torch.eye(3, dtype=F.dtype, device=F.device).expand_as(F).clone()
    for _ in range(5):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            apq, d = S[:, p, q], S[:, q, q] - S[:, p, p]
            off = apq.abs() > 1e-300
            tau = d / torch.where(off, 2 * apq, torch.ones_like(apq))
            t = torch.where(tau >= 0, 1.0, -1.0) / (tau.abs() + torch.sqrt(1 + tau * tau))
            t = torch.where(off, t, torch.zeros_like(t))
            c = 1 / torch.sqrt(1 + t * t)
            s = t * c
            J = torch.eye(3, dtype=F.dtype, device=F.device).expand_as(F).clone()
            J[:, p, p], J[:, q, q], J[:, p, q], J[:, q, p] = c, c, s, -s
            S = _mm(_mm(J.transpose(1, 2), S), J)
            V = _mm(V, J)
    sv = torch.sqrt(torch.diagonal(S, dim1=1, dim2=2))
    FV = _mm(F, V)
    return _mm(FV * (sv.clamp(lo, hi) / sv)[:, None, :], V.transpose(1, 2))


class _Stencil:
    def __init__(self, x, dx, N):
        xg = x / dx
        base = (xg - 0.5).to(torch.int64)
        f = xg - base
        w = torch.stack([0.5 * (1.5 - f) ** 2, 0.75 - (f - 1) ** 2, 0.5 * (f - 0.5) ** 2], 2)  # (n, 3 axes, 3)
        o = torch.arange(3, device=x.device)
        d = (base[:, :, None] + o) * dx - x[:, :, None]
        n = x.shape[0]
        self.w = (w[:, 0, :, None, None] * w[:, 1, None, :, None] * w[:, 2, None, None, :]).reshape(n, 27)
        b = base[:, :, None] + o
        self.node = ((b[:, 0, :, None, None] * N + b[:, 1, None, :, None]) * N + b[:, 2, None, None, :]).reshape(n, 27)
        self.d = torch.stack([d[:, 0, :, None, None].expand(n, 3, 3, 3), d[:, 1, None, :, None].expand(n, 3, 3, 3),
                              d[:, 2, None, None, :].expand(n, 3, 3, 3)], -1).reshape(n, 27, 3)
        self.inside = bool((base >= 0).all()) and bool((base + 2 < N).all())


def _walls(params, device):
    N, b = params["N"], params["boundary"]
    i = torch.arange(N, device=device)
    if params["boundary_mode"] == BOUNDARY_CELLS:
        low, high = i < b, i >= N - b
    else:
        f = i.to(torch.float32) / np.float32(N)
        low, high = f < _f32(b), f > np.float32(1.0) - np.float32(b)
    side = low | high
    sticky = side[:, None, None] | high[None, :, None] | side[None, None, :]
    return sticky.expand(N, N, N).reshape(-1), low[None, :, None].expand(N, N, N).reshape(-1)


def _substep(x, v, C, stress, mass, volume, params, walls, chunk=1 << 18):
    """One substep of particles of mass (n,): the new x, v, C and I + dt C, or
    None where a stencil reaches past the grid. `stress`: Kirchhoff stress."""
    N, dt = params["N"], _f32(params["dt"])
    dx = _f32(1.0 / N)
    dinv = 4.0 / dx ** 2
    n = x.shape[0]
    parts = [slice(a, min(n, a + chunk)) for a in range(0, n, chunk)]
    A = -dinv * dt * volume * stress + mass[:, None, None] * C
    grid = torch.zeros(N ** 3, 4, dtype=x.dtype, device=x.device)
    kept = []
    for p in parts:
        s = _Stencil(x[p], dx, N)
        if not s.inside:
            return None
        mom = (mass[p, None] * v[p])[:, None, :] + (A[p][:, None] * s.d[:, :, None, :]).sum(-1)
        val = torch.cat([mom, mass[p, None, None].expand(-1, 27, 1)], 2) * s.w[:, :, None]
        grid = grid.index_add(0, s.node.reshape(-1), val.reshape(-1, 4))
        kept.append(s if len(parts) == 1 else None)
    full = grid[:, 3] > 0
    vel = grid[:, :3] / torch.where(full, grid[:, 3], torch.ones_like(grid[:, 3]))[:, None]
    sticky, floor = walls
    vy = vel[:, 1] + dt * _f32(params["gravity"])
    vy = torch.where(floor, vy.clamp(min=0.0), vy)
    vel = torch.stack([vel[:, 0], vy, vel[:, 2]], 1)
    vel = torch.where((full & ~sticky)[:, None], vel, torch.zeros_like(vel))
    vs, Cs = [], []
    for p, s in zip(parts, kept):
        s = s or _Stencil(x[p], dx, N)
        wg = s.w[:, :, None] * vel[s.node]
        vs.append(wg.sum(1))
        Cs.append(dinv * (wg[:, :, :, None] * s.d[:, :, None, :]).sum(1))
    v, C = torch.cat(vs), torch.cat(Cs)
    return x + dt * v, v, C, torch.eye(3, dtype=x.dtype, device=x.device) + dt * C


def _corotated(F, mu, lam, J):
    eye = torch.eye(3, dtype=F.dtype, device=F.device)
    return ((2 * mu)[:, None, None] * _mm(F - _rotation(F), F.transpose(1, 2)) +
            (lam * (J - 1) * J)[:, None, None] * eye)


def _simulate(params, materials, p, substeps):
    """The engine's state after `substeps`, in 64 bits, or None."""
    dev = torch.device("cuda")
    x, v, C, F, Jp = (torch.from_numpy(p[k]).to(dev, torch.float64) for k in ("x", "v", "C", "F", "Jp"))
    mats, walls = torch.from_numpy(p["material"]).to(dev), _walls(params, dev)
    volume = _f32(materials[0]["volume"])  # one for all materials of a scene
    density = torch.tensor([m["density"] for m in materials], dtype=torch.float32, device=dev)
    mass = (density * volume).to(torch.float64)[mats.long()]
    fixed = params["compat"] == COMPAT_FIXED
    if not fixed and x.shape[0] - 1 > params["N"] ** 3:
        return None  # the reference's bound on particle indices holds some back
    of = [slice(None) if len(materials) == 1 else torch.nonzero(mats == i)[:, 0] for i in range(len(materials))]
    one = np.float32(1)
    for _ in range(substeps):
        tau = torch.zeros_like(F)
        for sel, m in zip(of, materials):
            f, j = F[sel], Jp[sel]
            if m["kind"] == MATERIAL_WC_LIQUID:
                tau[sel] = (_f32(m["bulk_modulus"]) * (j - 1) * j)[:, None, None] * torch.eye(3, dtype=F.dtype, device=dev)
                continue
            E, nu = np.float32(m["E"]), np.float32(m["nu"])
            e = torch.ones_like(j)
            if m["kind"] != MATERIAL_FIXED_COROTATED:
                e = torch.exp(_f32(m["hardening"]) * (1 - j))
            mu, lam = float(E / (2 * (one + nu))), float(E * nu / ((one + nu) * (one - 2 * nu)))
            tau[sel] = _corotated(f, mu * e, lam * e, _det(f) if fixed else j)
        got = _substep(x, v, C, tau, mass, volume, params, walls)
        if got is None:
            return None
        x, v, C, A = got
        F = _mm(A, F)
        for sel, m in zip(of, materials):
            if m["kind"] == MATERIAL_WC_LIQUID:
                J = _det(F[sel])
                Jp[sel] = J
                F[sel] = (torch.sign(J) * J.abs() ** (1 / 3))[:, None, None] * torch.eye(3, dtype=F.dtype, device=dev)
            elif m["kind"] == MATERIAL_JELLY:
                Jp[sel] = Jp[sel].clamp(0.6, 20.0)
            elif m["kind"] == MATERIAL_SNOW:
                f = F[sel]
                old = _det(f)
                if m["clamp_hi"] < 1e29:
                    f = _clamp_stretch(f, _f32(m["clamp_lo"]), _f32(m["clamp_hi"]))
                    F[sel] = f
                Jp[sel] = (Jp[sel] * old / _det(f)).clamp(0.6, 20.0)
    return dict(x=x, v=v, C=C, F=F, Jp=Jp, material=None)


def _differentiable(params, mass, volume, p, substeps):
    """State planes, mu and lambda as 64-bit leaves, and the planes after
    `substeps`; None for those where a stencil reaches past the grid."""
    dev = torch.device("cuda")
    leaves = [torch.from_numpy(p[k]).to(dev, torch.float64).requires_grad_(True) for k in ("st", "mu", "lam")]
    st, mu, lam = leaves
    n = st.shape[1]
    walls, m = _walls(params, dev), torch.full((n,), mass, dtype=torch.float64, device=dev)
    x, v, C, F = st[0:3].T, st[3:6].T, st[6:15].T.reshape(n, 3, 3), st[15:24].T.reshape(n, 3, 3)
    for _ in range(substeps):
        got = _substep(x, v, C, _corotated(F, mu, lam, _det(F)), m, volume, params, walls)
        if got is None:
            return leaves, None
        x, v, C, A = got
        F = _mm(A, F)
    return leaves, torch.cat([x.T, v.T, C.reshape(n, 9).T, F.reshape(n, 9).T])


def exact(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "frame":
        if case["particles"] * case["substeps"] > 9e7:
            return None  # too long
        return _simulate(*_scene(case["scene"], case["particles"], case["N"], rng), case["substeps"])
    if kind == "batch":
        got = [_simulate(*s, case["substeps"]) for s in _batch_scenes(case, rng)]
        if any(g is None for g in got):
            return None
        return {k: None if k == "material" else torch.cat([g[k] for g in got]) for k in got[0]}
    if kind == "mesh":
        return None  # the triangles are those of a 32-bit field, bit for bit
    params, mass, volume, n, p = _cube(case, seed)
    if kind == "step":
        leaves, st = _differentiable(params, mass, volume, p, 1)
        if st is None:
            return None
        g = torch.autograd.grad(st, leaves, _step_adjoint(torch.from_numpy(p["st"]).cuda()).double())
        return dict(out=st.detach(), adj_in=g[0], adj_mu=g[1], adj_lam=g[2])
    if case["grad"] and n * case["substeps"] > 4e6:
        return None  # too much to keep for the gradient
    with torch.set_grad_enabled(case["grad"]):
        leaves, st = _differentiable(params, mass, volume, p, case["substeps"])
        if st is None:
            return None
        if not case["grad"]:
            return dict(state=st.detach())
        g = torch.autograd.grad(_loss(st, torch.from_numpy(p["target"]).cuda().double()), leaves)
    return dict(state=st.detach(), grad_state=g[0], grad_mu=g[1], grad_lam=g[2])
