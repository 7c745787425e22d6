"""The work that a program using birdflow_hip has it do, as cases that can be timed.

A case is a batch of steps of one simulation (or one gradient of it) through
birdflow_hip's public calls, and what the program reads back after the batch:
the load history, the density and velocity fields, the body's state.  The
simulation is made in prepare(): configuration, geometry and start state are in
place, as they are in a program that then steps for hours.

Kinds:
  box       periodic box of decaying modes, no walls (the shear-wave workload)
  fixed     fixed obstacle written by the caller, far-field or inlet / outlet
            faces, half-way or interpolated walls, optional sponge
  sphere    translating sphere, one step at a time (a coupled loop)
  plate     flapping plate as a recorded frame sequence, 12 triangles
  bird      articulated bird, 40,000 triangles, on-device kinematics
  flight    analytic bird in free flight (the reference's product path)
  wing      prescribed Li & Nabawy wing with its link table
  gradient  adjoint gradient of the plate's mean lift, 8 parameters
  response  adjoint sensitivity dJ/df of a fixed obstacle's load
"""
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch
import torch.utils.checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "numi-gpu-physics_amd"))

import birdflow_hip as bh  # noqa: E402
from birdflow_hip import workloads  # noqa: E402

STORAGE = {"fp32": bh.STORAGE_FP32, "fp16": bh.STORAGE_FP16_OFFSET, "bf16": bh.STORAGE_BF16_OFFSET}
COLLISION = {"trt": bh.COLLISION_TRT, "limited": bh.COLLISION_TRT_SYMMETRIC_LIMITER,
             "regularized": bh.COLLISION_REGULARIZED, "rr3": bh.COLLISION_RR3}
WALLS = {"halfway": bh.WALL_HALFWAY, "sdf": bh.WALL_INTERPOLATED_SDF, "half": bh.WALL_INTERPOLATED_HALF,
         "links": bh.WALL_INTERPOLATED_LINKS, "ray": bh.WALL_INTERPOLATED_RAY}
PERIODIC = ((bh.BC_PERIODIC, bh.BC_PERIODIC),) * 3
OPEN = ((bh.BC_FARFIELD, bh.BC_FARFIELD),) * 3
CHANNEL = ((bh.BC_FARFIELD, bh.BC_OUTLET),) + PERIODIC[:2]
STREAM = ((bh.BC_FARFIELD, bh.BC_FARFIELD),) + PERIODIC[:2]
FACES = {"periodic": PERIODIC, "open": OPEN, "channel": CHANNEL, "stream": STREAM}


def case(name, kind, nx, ny, nz, steps, storage="fp32", collision="trt", walls="halfway", faces="periodic",
         sponge=0.0):
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, steps=steps, storage=storage, collision=collision, walls=walls,
             faces=faces, sponge=sponge)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the translating-sphere canonical, driven as a host-coupled loop drives it: one step, its load, the fields
        case("sphere, one step", "sphere", 24, 24, 24, 1, walls="half"),
        # the shear-wave accuracy workload: 64^3, periodic, many steps per call
        case("box 64", "box", 64, 64, 64, 200),
        # the fixed-wing diagnostic (80 x 80 x 48, sponge on every face): a grid that is not whole tiles
        case("fixed wing 80", "fixed", 80, 80, 48, 200, faces="open", sponge=0.04),
        # an obstacle on an odd grid, channel faces, interpolated walls, 16-bit storage
        case("obstacle, ragged, bf16", "fixed", 203, 117, 91, 100, storage="bf16", collision="regularized",
             walls="sdf", faces="channel"),
        # the flapping plate at its stated size, one recorded frame per step
        case("plate 256", "plate", 256, 128, 128, 200, collision="rr3", walls="sdf", faces="channel"),
        # free flight of the analytic bird: geometry, loads and body update follow each other every step
        case("free flight 320", "flight", 320, 200, 168, 100, faces="open", sponge=0.04),
        # the prescribed wing at the resolution of its lift validation (16 cells per chord)
        case("wing 160", "wing", 160, 160, 128, 200, walls="links", faces="open", sponge=0.04),
        # the headline workload: the articulated bird, FP32
        case("bird 512", "bird", 512, 256, 256, 200, collision="rr3", walls="sdf", faces="channel"),
        # the same bird with exact link fractions, as a smaller design study runs it
        case("bird 384, exact roots", "bird", 384, 192, 192, 100, collision="rr3", walls="ray", faces="channel"),
        # the precision case: 16-bit offsets on a grid that FP32 studies avoid (113M cells)
        case("bird 768, fp16", "bird", 768, 384, 384, 100, storage="fp16", collision="rr3", walls="sdf",
             faces="channel"),
        # shape optimization: gradient of the plate's mean lift, checkpoints every 25 steps
        case("gradient 256", "gradient", 256, 128, 128, 100, collision="rr3", walls="sdf", faces="stream"),
        # sensitivity of an obstacle's load to the flow state, small grid
        case("response 96", "response", 96, 48, 40, 40, collision="rr3", walls="sdf", faces="stream"),
    ]


def draw(rng):
    """One more case: any kind, sizes log-uniform over the kind's range, odd ones among them."""
    def size(lo, hi):
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return v if rng.random() < 0.5 else max(8, v // 8 * 8)
    kind = rng.choice(["box", "fixed", "fixed", "sphere", "plate", "bird", "bird", "flight", "wing", "gradient",
                       "response"])
    storage = rng.choice(["fp32", "fp32", "fp16", "bf16"])
    if kind == "sphere":
        return case(None, kind, size(24, 64), size(24, 64), size(24, 64), rng.choice([1, 2, 4]), walls="half")
    if kind == "box":
        return case(None, kind, size(32, 320), size(32, 160), size(32, 160), rng.randint(50, 200), storage,
                    rng.choice(["trt", "limited", "regularized", "rr3"]))
    if kind == "fixed":
        return case(None, kind, size(48, 320), size(48, 200), size(40, 160), rng.randint(50, 150), storage,
                    rng.choice(["trt", "regularized", "rr3"]), rng.choice(["halfway", "sdf"]),
                    rng.choice(["open", "channel", "stream"]), rng.choice([0.0, 0.04]))
    if kind == "plate":
        nx = size(128, 384)
        return case(None, kind, nx, nx // 2 + rng.randint(0, 9), nx // 2 + rng.randint(0, 9), rng.randint(50, 200),
                    storage, "rr3", "sdf", "channel")
    if kind == "bird":
        nx = size(256, 640)
        return case(None, kind, nx, nx // 2 + rng.randint(0, 9), nx // 2 + rng.randint(0, 9), rng.randint(20, 60),
                    storage, "rr3", rng.choice(["sdf", "sdf", "ray"]), "channel")
    if kind == "flight":
        nx = size(192, 448)
        return case(None, kind, nx, nx * 5 // 8 + rng.randint(0, 9), nx // 2 + rng.randint(0, 9), rng.randint(20, 100),
                    "fp32", rng.choice(["trt", "trt", "limited"]), "halfway", "open", 0.04)
    if kind == "wing":
        nx = size(96, 384)
        return case(None, kind, nx, nx + rng.randint(0, 9), nx // 2 + nx // 4 + rng.randint(0, 9), rng.randint(30, 100),
                    storage, "trt", "links", "open", 0.04)
    if kind == "gradient":
        nx = size(128, 256)
        return case(None, kind, nx, nx // 2 + rng.randint(0, 9), nx // 2 + rng.randint(0, 9), rng.randint(50, 100),
                    storage, "rr3", rng.choice(["sdf", "sdf", "ray"]), "stream")
    return case(None, kind, size(48, 128), size(40, 64), size(32, 64), rng.randint(20, 40), "fp32",
                rng.choice(["trt", "regularized", "rr3"]), "sdf", "stream")


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def shape_of(c):
    return c["nx"], c["ny"], c["nz"]


def omegas(tau, magic=3.0 / 16.0):
    return 1.0 / tau, 1.0 / (0.5 + magic / (tau - 0.5))


def config(c, tau, **kw):
    op, om = omegas(tau)
    kw.setdefault("sponge_width", 8.0 if min(shape_of(c)) > 64 else 4.0)
    return bh.SolverConfig(shape=shape_of(c), omega_plus=op, omega_minus=om, storage=STORAGE[c["storage"]],
                           collision=COLLISION[c["collision"]], wall_rule=WALLS[c["walls"]],
                           boundary=FACES[c["faces"]], sponge_strength=c["sponge"], **kw)


def modes(c, seed, speed=0.02, count=6):
    """Populations [19 N] FP32 at the equilibrium of a few random smooth
    velocity modes (made on the device when there is one)."""
    nx, ny, nz = shape_of(c)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = np.random.default_rng(seed)
    ax = [2.0 * math.pi * torch.arange(n, device=dev, dtype=torch.float32) / n for n in (nx, ny, nz)]
    u = torch.zeros(3, nz, ny, nx, device=dev)
    for _ in range(count):
        k = rng.integers(-2, 3, 3)
        amp, ph = rng.normal(size=3), rng.uniform(0.0, 2.0 * math.pi)
        wave = torch.sin(float(k[2]) * ax[2][:, None, None] + float(k[1]) * ax[1][None, :, None]
                         + float(k[0]) * ax[0][None, None, :] + float(ph))
        for i in range(3):
            u[i] += float(amp[i]) * wave
    u *= speed / max(float(u.abs().max()), 1e-12)
    return equilibria(torch.ones(nz, ny, nx, device=dev), u).reshape(-1).cpu().numpy()


def obstacle(c, seed):
    """A tilted, slowly turning ellipsoid in the first third of the grid:
    (mask [N], wall [N, 4] = wall velocity and signed distance in cells, centre)."""
    nx, ny, nz = shape_of(c)
    rng = np.random.default_rng(seed)
    center = np.array([0.33 * nx, 0.5 * ny, 0.5 * nz]) + rng.uniform(-1.0, 1.0, 3)
    radii = min(ny, nz) * np.array([0.16, 0.2, 0.11]) * rng.uniform(0.9, 1.1, 3)
    tilt, spin = rng.uniform(0.2, 0.6), rng.uniform(-1.0, 1.0, 3) * 0.02 / radii.max()
    x = (np.arange(nx, dtype=np.float32) + np.float32(0.5) - np.float32(center[0]))[None, None, :]
    y = (np.arange(ny, dtype=np.float32) + np.float32(0.5) - np.float32(center[1]))[None, :, None]
    z = (np.arange(nz, dtype=np.float32) + np.float32(0.5) - np.float32(center[2]))[:, None, None]
    ct, st = np.float32(math.cos(tilt)), np.float32(math.sin(tilt))
    a, b, d = (ct * x + st * z) / np.float32(radii[0]), y / np.float32(radii[1]), (ct * z - st * x) / np.float32(radii[2])
    r = np.sqrt(a * a + b * b + d * d)
    # first-order signed distance: level set over the length of its gradient
    grad = np.sqrt((a / radii[0]) ** 2 + (b / radii[1]) ** 2 + (d / radii[2]) ** 2).astype(np.float32)
    sd = np.where(r > 1e-3, (r - 1.0) * r / np.maximum(grad, np.float32(1e-6)), -radii.min()).astype(np.float32)
    w = spin.astype(np.float32)
    wall = np.empty((nz, ny, nx, 4), np.float32)
    wall[..., 0], wall[..., 1], wall[..., 2] = w[1] * z - w[2] * y, w[2] * x - w[0] * z, w[0] * y - w[1] * x
    wall[..., 3] = sd
    mask = (sd <= 0.0).astype(np.uint8)
    return mask.ravel(), wall.reshape(-1, 4), center


def plate_theta(seed):
    """Heave 8 cells and pitch 30 degrees with second harmonics of a quarter,
    each of the 8 values drawn +-20 %."""
    base = np.array([8.0, 0.0, 2.0, 0.0, np.radians(30.0), np.pi / 2, np.radians(7.5), np.pi / 2])
    return base * (1.0 + 0.2 * np.random.default_rng(seed).uniform(-1.0, 1.0, 8))


PLATE_PERIODS = 20


def plate_frames(c, seed):
    """The plate's recorded frames and their parameter tangents: whole
    periods of 800 steps, one after the other."""
    s = c["nx"] / 256.0
    theta = plate_theta(seed)
    theta[0], theta[2] = theta[0] * s, theta[2] * s
    seq, _, tan = workloads.parametric_plate(theta, 799, center=(64.0 * s, c["ny"] / 2, c["nz"] / 2),
                                             span=48.0 * s, chord=16.0 * s)
    pts = np.tile(seq.points, (PLATE_PERIODS, 1, 1))
    return (dataclasses.replace(seq, points=pts, times=np.arange(len(pts), dtype=np.float32)),
            np.tile(tan.astype(np.float32), (1, PLATE_PERIODS, 1, 1)))


@functools.lru_cache(maxsize=16)
def bird_mesh(nx, ny, nz):
    s = nx / 512.0
    return workloads.synthetic_bird_articulated(
        seed=7, center=(160.0 * s, ny / 2, nz / 2), body_radii=(40.0 * s, 14.0 * s, 14.0 * s), half_span=100.0 * s,
        root_chord=40.0 * s, tip_chord=12.0 * s, tail=(30.0 * s, 20.0 * s), period=1200.0 * s)


# ---------------------------------------------------------------------------
# prepare and run.
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c, kind = case, case["kind"]
    nx, ny, nz = shape_of(c)
    rng = np.random.default_rng(seed)
    st = {"case": c}
    if kind == "box":
        sim = bh.BirdFlowSimulation(config(c, 0.8))
        sim.write_populations(modes(c, seed))
    elif kind in ("fixed", "response"):
        mask, wall, center = obstacle(c, seed)
        sim = bh.BirdFlowSimulation(config(c, 0.62, accumulate_loads=True, far_velocity=(0.05, 0.01, 0.0),
                                           body_position=tuple(center)))
        sim.set_geometry(mask, wall)
        sim.write_populations(modes(c, seed))
        if kind == "response":
            st["weights"] = np.concatenate([rng.normal(size=(c["steps"], 3)),
                                            0.1 * rng.normal(size=(c["steps"], 3))], 1) / c["steps"]
    elif kind == "sphere":
        r = min(nx, ny, nz) * 3.25 / 24.0
        center = (nx / 3.0 + rng.uniform(-0.5, 0.5), ny / 2.0 + rng.uniform(-0.5, 0.5), nz / 2.0)
        sim = bh.BirdFlowSimulation(config(c, 0.8, accumulate_loads=True, selected_part=1, body_position=center))
        v = 0.001 * rng.uniform(0.5, 1.0)       # slow: the program runs for thousands of steps
        sim.set_translating_sphere((*center, r), (v, 0.0, 0.0), (0.05 * rng.uniform(0.8, 1.0), 0.0, 0.0, 0.0))
        sim.init_equilibrium()
    elif kind in ("plate", "gradient"):
        seq, tan = plate_frames(c, seed)
        s = nx / 256.0
        sim = bh.BirdFlowSimulation(config(c, 0.6, accumulate_loads=True, far_velocity=(0.05, 0.0, 0.0),
                                           body_position=(64.0 * s, ny / 2, nz / 2)))
        sim.upload_mesh(seq.points, seq.times, seq.triangles, seq.parts, seq.half_thickness)
        if kind == "gradient":
            sim.adjoint_set_tangents(tan)
            w = np.zeros((c["steps"], 6))
            w[c["steps"] // 2:, 2] = 1.0 / (c["steps"] - c["steps"] // 2)
            st["weights"] = w
        sim.init_equilibrium()
    elif kind == "bird":
        mesh = bird_mesh(nx, ny, nz)
        mesh = dataclasses.replace(mesh, amplitude_scale=mesh.amplitude_scale * rng.uniform(0.8, 1.0))
        sim = bh.BirdFlowSimulation(config(c, 0.52, accumulate_loads=True,
                                           far_velocity=(0.04 * rng.uniform(0.9, 1.0), 0.0, 0.0),
                                           body_position=tuple(mesh.center)))
        sim.upload_articulated(mesh, time_start=float(int(rng.uniform(0.0, mesh.period))))
        sim.init_equilibrium()
    elif kind == "flight":
        sc = bh.LatticeScaling.make(0.14, max(8, round(35 * nx / 512)), 10.0, 500.0 * nx / 512, 1.225)
        dx = sc.cell_size
        pos = (0.3 * nx * dx, 0.5 * ny * dx, 0.5 * nz * dx)
        sim = bh.BirdFlowSimulation(dataclasses.replace(
            config(c, 1.0), omega_plus=sc.omega_plus, omega_minus=sc.omega_minus, cell_size=dx,
            time_step=sc.time_step, velocity_to_lattice=sc.velocity_to_lattice,
            force_to_physical=sc.force_to_physical, accumulate_loads=True, body_position=pos,
            far_velocity=(-10.0 * rng.uniform(0.9, 1.0) * sc.velocity_to_lattice, 0.0, 0.0)))
        # cruise: the weight is carried (external force), the body answers the flapping loads
        sim.set_body([*pos, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0],
                     bh.BodyParameters(mass=0.42, inertia=(0.0024, 0.0068, 0.0074), gravity=(0.0, 0.0, -9.81),
                                       external_force=(0.0, 0.0, 0.42 * 9.81)))
        sim.set_bird(bh.BirdGeometry.demonstration())
        sim.set_restart_state(0, float(rng.uniform(0.0, 1.0 / 4.5)))
        sim.init_equilibrium()
    elif kind == "wing":
        root = (0.5 * nx, 0.5 * ny, 0.5 * nz)
        chord = nx / 10.0 if nx < 300 else nx / 12.0
        sim = bh.BirdFlowSimulation(config(c, 3.0 * 0.08 * chord / 100.0 + 0.5, accumulate_loads=True,
                                           body_position=root))
        sim.set_flapping_wing(bh.FlappingWing.li_nabawy(chord, root, 256.0 * chord))
        sim.set_restart_state(0, float(int(rng.uniform(0.0, 256.0 * chord))))
        sim.init_equilibrium()
    else:
        raise ValueError(kind)
    st["sim"] = sim
    return st


def run(state):
    c, sim = state["case"], state["sim"]
    kind, steps = c["kind"], c["steps"]
    if kind == "gradient":
        value, grad, _ = sim.adjoint_gradient(steps, state["weights"], 25)
        return {"objective": value, "gradient": grad, "loads": sim.load_history(steps)}
    if kind == "response":
        value, _, _ = sim.adjoint_gradient(steps, state["weights"], 10)
        return {"objective": value, "sensitivity": sim.adjoint_sensitivity(), "loads": sim.load_history(steps)}
    sim.advance(steps)
    out = {}
    if kind == "sphere":
        out["load"] = sim.read_loads()
    elif kind != "box":
        out["loads"] = sim.load_history(steps)
    if kind == "flight":
        out["body"] = sim.body_history(steps)
    out["density"], out["velocity"] = sim.copy_macroscopic_fields()
    return out


def work(case):
    """Populations once in and once out per step, the fields and histories once; for the gradients the forward
    pass, the recomputed steps, and per reverse step the state and the adjoint in and the adjoint out.  Operations of
    one collision: about 250 for TRT, 600 for the others; its adjoint about twice that."""
    c = case
    n, k = c["nx"] * c["ny"] * c["nz"], c["steps"]
    elem = 4 if c["storage"] == "fp32" else 2
    ops = 250 if c["collision"] in ("trt", "limited") else 600
    move = 38 * elem * n
    if c["kind"] in ("gradient", "response"):
        reverse = 19 * elem * n + 2 * 19 * 4 * n
        out = 19 * 4 * n if c["kind"] == "response" else 0
        return {"bytes": k * (2 * move + reverse) + out, "flops": k * 4 * ops * n}
    return {"bytes": k * move + 16 * n, "flops": k * ops * n}


# ---------------------------------------------------------------------------
# The same step in 64 bits, written from the equations in plain torch:
# pull stream with face rules, bounce-back at fixed walls, collision, sponge,
# momentum-exchange load.  Moving geometry has no 64-bit value: whether a cell
# is solid is a comparison of FP32 distances, and a cell within rounding of the
# surface decides differently in 64 bits.
# ---------------------------------------------------------------------------
C = np.array([[0, 0, 0], [1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1], [1, 1, 0], [-1, -1, 0],
              [1, -1, 0], [-1, 1, 0], [1, 0, 1], [-1, 0, -1], [1, 0, -1], [-1, 0, 1], [0, 1, 1], [0, -1, -1],
              [0, 1, -1], [0, -1, 1]])
OPP = [0, 2, 1, 4, 3, 6, 5, 8, 7, 10, 9, 12, 11, 14, 13, 16, 15, 18, 17]
W = [1.0 / 3.0] + [1.0 / 18.0] * 6 + [1.0 / 36.0] * 12


def along(q, u):
    return sum(float(C[q, a]) * u[a] for a in range(3))


def equilibria(rho, u):
    """[19, ...] second-order equilibrium of density rho and velocity u [3, ...]."""
    u2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
    out = []
    for q in range(19):
        cu = along(q, u)
        out.append(W[q] * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * u2))
    return torch.stack(out)


class Exact:
    """One FP64 step of a configuration with fixed walls (mask [N], wall [N, 4])."""

    def __init__(self, cfg, mask, wall, dev):
        self.cfg, self.dev = cfg, dev
        nx, ny, nz = cfg.shape
        self.shape = (nz, ny, nx)
        f32 = lambda v: float(np.float32(v))  # noqa: E731  (what the solver is given)
        self.op, self.om = f32(cfg.omega_plus), f32(cfg.omega_minus)
        self.far_u = torch.tensor([f32(v) for v in cfg.far_velocity], dtype=torch.float64, device=dev)
        self.far = equilibria(torch.tensor(f32(cfg.far_density), dtype=torch.float64, device=dev), self.far_u)
        self.solid = torch.as_tensor(mask, device=dev).reshape(self.shape) != 0
        wl = torch.as_tensor(wall, device=dev).double().reshape(*self.shape, 4)
        self.wu, self.wd = wl[..., :3].movedim(-1, 0), wl[..., 3]
        d = [torch.arange(n, device=dev) for n in self.shape]
        edge = torch.minimum(torch.minimum(d[0], nz - 1 - d[0])[:, None, None],
                             torch.minimum(torch.minimum(d[1], ny - 1 - d[1])[None, :, None],
                                           torch.minimum(d[2], nx - 1 - d[2])[None, None, :])).double()
        width = f32(cfg.sponge_width)
        ramp = ((width - edge) / max(width, 1.0)).clamp(0.0, 1.0)
        self.sponge = torch.where(edge >= width, 0.0, f32(cfg.sponge_strength) * ramp * ramp)
        body = [f32(v) for v in cfg.body_position]
        self.arm = [(d[2 - a].double() + 0.5 - body[a]).reshape([-1 if i == 2 - a else 1 for i in range(3)])
                    .expand(self.shape) for a in range(3)]
        self.any_solid = bool(self.solid.any())
        self.src = [self.index(q, -1) for q in range(19)]
        self.ahead = [self.index(q, +1) for q in range(19)]

    def index(self, q, sign):
        """Cells at x + sign c_q: per-axis indices (z, y, x), whether a far-field face lies between, whether a face does."""
        idx, far, out = [], torch.zeros(1, 1, 1, dtype=torch.bool, device=self.dev), None
        out = far
        for i, a in enumerate((2, 1, 0)):
            n = self.shape[i]
            v = torch.arange(n, device=self.dev) + sign * int(C[q, a])
            lo, hi = self.cfg.boundary[a]
            shape = [-1 if j == i else 1 for j in range(3)]
            beyond = ((v < 0) & (lo == bh.BC_FARFIELD)) | ((v >= n) & (hi == bh.BC_FARFIELD))
            far = far | beyond.reshape(shape)
            out = out | ((v < 0) | (v >= n)).reshape(shape)
            idx.append(v % n if lo == bh.BC_PERIODIC else v.clamp(0, n - 1))
        return idx, far.expand(self.shape), out.expand(self.shape)

    @staticmethod
    def at(t, idx):
        return t.index_select(0, idx[0]).index_select(1, idx[1]).index_select(2, idx[2])

    def step(self, f):
        """f [19, z, y, x] -> the next populations and the load [6]."""
        g, load = [], [torch.zeros((), dtype=torch.float64, device=self.dev) for _ in range(6)]
        for q in range(19):
            idx, far, _ = self.src[q]
            v = self.at(f[q], idx)
            if self.any_solid:
                link = self.at(self.solid, idx) & ~far & ~self.solid
                v = self.wall(q, f, v, link, load)
            g.append(torch.where(far, self.far[q], v))
        g = torch.stack(g)
        rho = g.sum(0)
        u = torch.stack([sum(float(C[q, a]) * g[q] for q in range(19) if C[q, a]) / rho for a in range(3)])
        post, act, restr = self.collide(g, equilibria(rho, u), u)
        if self.cfg.sponge_strength > 0.0:
            post = post + (self.far.reshape(19, 1, 1, 1) - post) * self.sponge
        if self.any_solid:
            post = torch.where(self.solid, equilibria(torch.ones_like(rho), self.wu), post)
            act, restr = torch.where(self.solid, 0.0, act), torch.where(self.solid, 0.0, restr)
        return post, torch.stack(load + [act.sum(), restr.max()])

    def wall(self, q, f, v, link, load):
        idx, _, _ = self.src[q]
        reflected = f[OPP[q]]
        ws, ds = torch.stack([self.at(self.wu[a], idx) for a in range(3)]), self.at(self.wd, idx)
        lf, wv, interp = torch.full_like(v, 0.5), ws, torch.zeros_like(link)
        if self.cfg.wall_rule == bh.WALL_INTERPOLATED_SDF:
            df, dn = self.wd.clamp(min=0.0), ds.clamp(max=0.0)
            lf = (df / (df - dn).clamp(min=1e-6)).clamp(1e-4, 1.0)
            aidx, _, out = self.ahead[q]
            blocked = (lf <= 0.5) & (out | self.at(self.solid, aidx))
            interp = ~blocked
            wv = torch.where(blocked, ws, self.wu + (ws - self.wu) * lf)
            lf = torch.where(blocked, 0.5, lf)
        corr = 6.0 * W[q] * float(np.float32(self.cfg.far_density)) * along(q, wv)
        value = reflected + corr
        if self.cfg.wall_rule == bh.WALL_INTERPOLATED_SDF:
            ahead = self.at(f[OPP[q]], self.ahead[q][0])
            near = 2.0 * lf * reflected + (1.0 - 2.0 * lf) * ahead + corr
            beyond = (reflected + corr) / (2.0 * lf) + (2.0 * lf - 1.0) * f[q] / (2.0 * lf)
            value = torch.where(interp, torch.where(lf <= 0.5, near, beyond), value)
        s = torch.where(link, -(value + reflected), 0.0)
        fo = [s * float(C[q, a]) for a in range(3)]
        arm = [self.arm[a] - lf * float(C[q, a]) for a in range(3)]
        for a in range(3):
            load[a] = load[a] + fo[a].sum()
            b, d = (a + 1) % 3, (a + 2) % 3
            load[3 + a] = load[3 + a] + (arm[b] * fo[d] - arm[d] * fo[b]).sum()
        return torch.where(link, value, v)

    def collide(self, g, eq, u):
        zero = torch.zeros_like(g[0])
        if self.cfg.collision in (bh.COLLISION_TRT, bh.COLLISION_TRT_SYMMETRIC_LIMITER):
            go, eo = g[OPP], eq[OPP]
            sym, anti = -self.op * 0.5 * ((g + go) - (eq + eo)), -self.om * 0.5 * ((g - go) - (eq - eo))
            if self.cfg.collision == bh.COLLISION_TRT:
                return g + sym + anti, zero, zero
            floor = (1e-6 * eq.clamp(min=0.0)).clamp(min=1e-12)
            room = ((g + anti - floor) / (-sym).clamp(min=1e-30)).clamp(0.0, 1.0)
            scale = torch.where((sym < 0.0) & (g + anti + sym < floor), room, 1.0).amin(0)
            return g + scale * sym + anti, (scale < 1.0).double(), 1.0 - scale
        neq = g - eq
        h = lambda q, a, b: float(C[q, a] * C[q, b]) - (1.0 / 3.0 if a == b else 0.0)  # noqa: E731
        P = [[sum(h(q, a, b) * neq[q] for q in range(19)) for b in range(3)] for a in range(3)]
        cand = []
        for q in range(19):
            reg = 4.5 * sum(h(q, a, b) * P[a][b] for a in range(3) for b in range(3))
            if self.cfg.collision == bh.COLLISION_RR3:
                # the six third-order terms c_b (c_a c_a - 1/3) with a != b, recursive closure
                reg = reg + 13.5 * sum(float(C[q, b]) * h(q, a, a) * (2.0 * u[a] * P[a][b] + u[b] * P[a][a])
                                       for a in range(3) for b in range(3) if a != b and C[q, b])
            cand.append(eq[q] + (1.0 - self.op) * W[q] * reg)
        cand = torch.stack(cand)
        floor = (1e-6 * eq.clamp(min=0.0)).clamp(min=1e-12)
        room = ((eq - floor) / (eq - cand).clamp(min=1e-30)).clamp(0.0, 1.0)
        scale = torch.where(cand < floor, room, 1.0).amin(0)
        return eq + scale * (cand - eq), (scale < 1.0).double(), 1.0 - scale


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind not in ("box", "fixed", "response"):
        return None
    n, steps = c["nx"] * c["ny"] * c["nz"], c["steps"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "box":
        cfg = config(c, 0.8)
        mask, wall = np.zeros(n, np.uint8), np.zeros((n, 4), np.float32)
    else:
        mask, wall, center = obstacle(c, seed)
        cfg = config(c, 0.62, accumulate_loads=True, far_velocity=(0.05, 0.01, 0.0), body_position=tuple(center))
    ex = Exact(cfg, mask, wall, dev)
    f = torch.as_tensor(modes(c, seed), device=dev).double().reshape(19, *ex.shape)
    if kind == "response":
        rng = np.random.default_rng(seed)
        w = torch.as_tensor(np.concatenate([rng.normal(size=(steps, 3)), 0.1 * rng.normal(size=(steps, 3))], 1) / steps,
                            device=dev)
        start = f.requires_grad_(True)
        loads, value = [], 0.0
        for s in range(steps):
            f, load = torch.utils.checkpoint.checkpoint(ex.step, f, use_reentrant=False)
            value = value + (w[s] * load[:6]).sum()
            loads.append(load.detach())
        value.backward()
        return {"objective": value.detach(), "sensitivity": start.grad.reshape(-1), "loads": torch.stack(loads)}
    loads = []
    with torch.no_grad():
        for _ in range(steps):
            f, load = ex.step(f)
            loads.append(load)
        rho = f.sum(0)
        u = torch.stack([sum(float(C[q, a]) * f[q] for q in range(19) if C[q, a]) / rho for a in range(3)], -1)
    out = {"density": rho.reshape(-1), "velocity": u.reshape(-1, 3)}
    if kind == "fixed":
        out["loads"] = torch.stack(loads)
    return out
