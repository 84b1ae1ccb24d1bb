"""The work that users of this framework have it do, as cases that can be timed.

A case is one call, or the few calls that belong together, through the public
entry points (`fluide_engine_amd.capi` over include/fluide_hip.h), from input
in the caller's hands to output in the caller's hands:

  frames    a simulation advanced by a few frames and its particles read back
            (the loop that every program around the simulators runs)
  batch     many independent scenes advanced together by host workers
  transfer  particles to the face grid and back: binning, P2G, the fluid SDF
            and markers, extrapolation, G2P (the stage entry points)
  project   the pressure projection of a given velocity field
  diffuse   the implicit viscosity step of a given velocity field
  mesh_sdf  the distance field of a triangle mesh (colliders, emitters, sources)
  surface   the triangle surface of a given distance field
  learn     loss, gradients and prediction of the warm-start network

Host buffers that a program allocates once are pinned here, as a program that
cares about its frame rate has them.
"""
import math

import numpy as np
import torch

from fluide_engine_amd import capi

METHODS = {"pic": capi.PIC, "flip": capi.FLIP, "apic": capi.APIC}
SOLVERS = {"jacobi": capi.SOLVER_JACOBI, "cg": capi.SOLVER_CG, "pcg": capi.SOLVER_PCG_JACOBI,
           "mgpcg": capi.SOLVER_MGPCG}
MAX_CFL = 3.0
_ctx = None


def context():
    """One context for the process, as a program has."""
    global _ctx
    if _ctx is None:
        _ctx = capi.Context(0)
    return _ctx


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a preview scene, where the latency of the launches is the cost
        dict(name="frames_flip_32", kind="frames", nx=32, ny=32, nz=32, method="flip", solver="mgpcg", tol=1e-6,
             fill=0.45, frames=4, dt=1 / 240, viscosity=0.0, collider=False),
        # a scene of ordinary size in a domain that is no cube and no power of two, with the reference's own solver
        dict(name="frames_apic_80x56x68", kind="frames", nx=80, ny=56, nz=68, method="apic", solver="cg", tol=1e-6,
             fill=0.4, frames=4, dt=1 / 240, viscosity=0.0, collider=False),
        # the benchmark's grid and method
        dict(name="frames_flip_128", kind="frames", nx=128, ny=128, nz=128, method="flip", solver="mgpcg", tol=1e-6,
             fill=0.24, frames=4, dt=1 / 240, viscosity=0.0, collider=False),
        # honey round an obstacle: the viscous substep and the collider branches of the boundary condition
        dict(name="frames_viscous_collider_48", kind="frames", nx=48, ny=64, nz=40, method="flip", solver="mgpcg",
             tol=1e-6, fill=0.5, frames=1, dt=1 / 240, viscosity=0.05, collider=True),
        # a batch of small scenes of mixed sizes, for data generation
        dict(name="batch_16_scenes", kind="batch", scenes=16, smallest=24, largest=64, workers=4, frames=2,
             dt=1 / 480),
        # the particle-grid transfers alone, through the stage entry points
        dict(name="transfer_flip_104", kind="transfer", nx=104, ny=104, nz=104, method="flip", fill=0.3),
        # the pressure projection of a field that the caller has, with the reference's solver and a tight tolerance
        dict(name="project_cg_72x60x44", kind="project", nx=72, ny=60, nz=44, solver="cg", tol=1e-10, fill=0.5),
        # and on a large grid with the multigrid solver
        dict(name="project_mgpcg_128", kind="project", nx=128, ny=128, nz=128, solver="mgpcg", tol=1e-10, fill=0.5),
        # the implicit viscosity step with the scene's default solver
        dict(name="diffuse_96x80x64", kind="diffuse", nx=96, ny=80, nz=64, fill=0.5, viscosity=0.02, dt=1 / 240),
        # a collider's mesh at the resolution of a scene
        dict(name="mesh_sdf_64", kind="mesh_sdf", nx=64, ny=64, nz=64, rings=24, segments=32),
        # the surface that is written for each frame
        dict(name="surface_128x96x112", kind="surface", nx=128, ny=96, nz=112, fill=0.4, mode="reference"),
        # one training evaluation of the warm-start network
        dict(name="learn_64x96x80", kind="learn", nx=64, ny=96, nz=80, loss="energy"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frames", "frames", "frames", "batch", "transfer", "project", "project", "diffuse", "mesh_sdf",
                       "surface", "learn"])
    if kind == "frames":
        viscous = rng.random() < 0.25
        collider = rng.random() < 0.25
        top = 64 if viscous or collider else 120
        return dict(kind=kind, nx=size(20, top), ny=size(20, top), nz=size(20, top),
                    method=rng.choice(["pic", "flip", "flip", "apic"]), solver=rng.choice(["cg", "mgpcg", "mgpcg"]),
                    tol=1e-6, fill=round(rng.uniform(0.15, 0.5), 3), frames=1 if viscous else rng.choice([2, 3, 4]),
                    dt=1 / rng.choice([120, 240, 480]), viscosity=round(rng.uniform(0.005, 0.05), 4) if viscous else 0.0,
                    collider=collider)
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(4, 24), smallest=rng.randint(16, 28), largest=rng.randint(40, 72),
                    workers=rng.choice([1, 2, 4, 8]), frames=rng.choice([1, 2, 3]), dt=1 / rng.choice([240, 480]))
    if kind == "transfer":
        return dict(kind=kind, nx=size(16, 112), ny=size(16, 112), nz=size(16, 112),
                    method=rng.choice(["pic", "flip", "apic"]), fill=round(rng.uniform(0.1, 0.4), 3))
    if kind == "project":
        solver = rng.choice(["cg", "pcg", "mgpcg", "mgpcg"])
        top = 128 if solver == "mgpcg" else 88
        return dict(kind=kind, nx=size(16, top), ny=size(16, top), nz=size(16, top), solver=solver, tol=1e-10,
                    fill=round(rng.uniform(0.3, 0.7), 3))
    if kind == "diffuse":
        return dict(kind=kind, nx=size(16, 96), ny=size(16, 96), nz=size(16, 96), fill=round(rng.uniform(0.3, 0.7), 3),
                    viscosity=round(rng.uniform(0.005, 0.05), 4), dt=1 / rng.choice([120, 240, 480]))
    if kind == "mesh_sdf":
        return dict(kind=kind, nx=size(24, 80), ny=size(24, 80), nz=size(24, 80), rings=rng.randint(6, 28),
                    segments=rng.randint(8, 32))
    if kind == "surface":
        return dict(kind=kind, nx=size(24, 128), ny=size(24, 128), nz=size(24, 128), fill=round(rng.uniform(0.2, 0.7), 3),
                    mode=rng.choice(["reference", "closed"]))
    return dict(kind=kind, nx=8 * rng.randint(3, 11), ny=8 * rng.randint(3, 11), nz=8 * rng.randint(3, 11),
                loss=rng.choice(["energy", "mse"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def pinned(shape, dtype):
    """A host array that the device can copy to and from at full rate."""
    t = torch.empty(tuple(int(n) for n in shape), dtype=getattr(torch, np.dtype(dtype).name),
                    pin_memory=torch.cuda.is_available())
    return t.numpy()


def dims(case):
    return case["nx"], case["ny"], case["nz"]


def spacing(case):
    return tuple(1.0 / n for n in dims(case))


def face_shape(case, c):
    n = [case["nx"], case["ny"], case["nz"]]
    n[c] += 1
    return n[2], n[1], n[0]


def waves(rng, count=3):
    """Wave numbers, phases and weights of a smooth field."""
    return [(rng.integers(1, 4, 3), rng.uniform(0, 2 * np.pi, 3), rng.normal()) for _ in range(count)]


def smooth(ws, x, y, z):
    """The field's values at broadcastable coordinates in the unit cube."""
    out = 0.0
    for k, p, a in ws:
        out = out + a * (np.cos(k[0] * np.pi * x + p[0]) * np.cos(k[1] * np.pi * y + p[1])
                         * np.cos(k[2] * np.pi * z + p[2]))
    return out / math.sqrt(len(ws))


def particle_velocities(rng, x, speed=0.6):
    """Swirls with some noise between neighbours, as a moving fluid's particles have."""
    v = np.empty_like(x)
    for a in range(3):
        v[:, a] = speed * smooth(waves(rng), x[:, 0], x[:, 1], x[:, 2])
    v += rng.standard_normal(x.shape, dtype=np.float32) * np.float32(0.05 * speed)
    return v


def tank(n, method, seed, fill, viscosity=0.0):
    """A tank filled to `fill` of its height, with a column above that at one side: x and v."""
    rng = np.random.default_rng(seed)
    desc = capi.scene_desc(n, method=method, blend=0.03, max_cfl=MAX_CFL, viscosity=viscosity,
                           max_particles=8 * n[0] * n[1] * n[2])
    boxes = [capi.box((-1, -1, -1), (2, 0.8 * fill, 2)), capi.box((-1, -1, -1), (0.3, 1.5 * fill, 2))]
    x = capi.seed_particles(desc, boxes, seed=int(rng.integers(1 << 40)))
    desc.max_particles = max(1, x.shape[0])
    return desc, x, particle_velocities(rng, x)


def cell_sdf(case, seed):
    """A distance-like field at the cell centres: a liquid with a wavy top and a drop above it.  Its sign is the
    case's own; the seed sets the values, as two fluids of one extent have them."""
    nx, ny, nz = dims(case)
    x = ((np.arange(nx) + 0.5) / nx)[None, None, :]
    y = ((np.arange(ny) + 0.5) / ny)[None, :, None]
    z = ((np.arange(nz) + 0.5) / nz)[:, None, None]
    top = case["fill"] + 0.06 * np.cos(2 * np.pi * x + 0.3) * np.cos(3 * np.pi * z + 0.7)
    drop = np.sqrt((x - 0.55) ** 2 + (y - 0.5 * (1 + case["fill"])) ** 2 + (z - 0.45) ** 2) - 0.3 * (1 - case["fill"])
    phi = np.minimum(y - top, drop)
    rng = np.random.default_rng(seed)
    return np.ascontiguousarray(phi * (1.0 + 0.2 * np.tanh(smooth(waves(rng), x, y, z))))


def face_field(case, seed):
    """The three face arrays of a velocity field: swirls, some noise, and walls that let nothing through."""
    rng = np.random.default_rng(seed + 7)
    n = dims(case)
    out = []
    for c in range(3):
        at = [(np.arange(n[a] + (a == c)) + (0.0 if a == c else 0.5)) / n[a] for a in range(3)]
        f = smooth(waves(rng), at[0][None, None, :], at[1][None, :, None], at[2][:, None, None])
        f = (f + 0.05 * rng.standard_normal(f.shape)).astype(np.float32)
        wall = [slice(None)] * 3
        for end in (0, -1):
            wall[2 - c] = end
            f[tuple(wall)] = 0.0
        p = pinned(f.shape, np.float32)
        p[...] = f
        out.append(p)
    return out


def lathe(rings, segments, lo, hi, rng):
    """A closed mesh: a ball in the box lo..hi with bumps, from pole to pole."""
    lo, hi = np.asarray(lo, float), np.asarray(hi, float)
    ws = waves(rng)
    v = [(0.0, 1.0, 0.0)]
    for r in range(1, rings):
        a = math.pi * r / rings
        for s in range(segments):
            b = 2 * math.pi * s / segments
            v.append((math.sin(a) * math.cos(b), math.cos(a), math.sin(a) * math.sin(b)))
    v.append((0.0, -1.0, 0.0))
    v = np.array(v)
    v = v * (0.85 + 0.1 * np.tanh(smooth(ws, v[:, :1], v[:, 1:2], v[:, 2:])))
    t = []
    at = lambda r, s: 1 + (r - 1) * segments + s % segments  # noqa: E731
    last = v.shape[0] - 1
    for s in range(segments):
        t.append((0, at(1, s + 1), at(1, s)))
        for r in range(1, rings - 1):
            t += [(at(r, s), at(r, s + 1), at(r + 1, s)), (at(r, s + 1), at(r + 1, s + 1), at(r + 1, s))]
        t.append((last, at(rings - 1, s), at(rings - 1, s + 1)))
    return lo + (hi - lo) * (0.5 + 0.5 * v), np.array(t, dtype=np.int32)


def system(case, seed):
    """A pressure system for the network: right-hand side, markers and solution on a liquid's cells."""
    nx, ny, nz = dims(case)
    rng = np.random.default_rng(seed)
    x = ((np.arange(nx) + 0.5) / nx)[None, None, :]
    y = ((np.arange(ny) + 0.5) / ny)[None, :, None]
    z = ((np.arange(nz) + 0.5) / nz)[:, None, None]
    top = 0.5 + 0.1 * smooth(waves(rng), x, 0.0, z)
    flags = np.where(np.broadcast_to(y < top, (nz, ny, nx)), 1, 0).astype(np.uint8)
    p = np.where(flags == 1, np.maximum(top - y, 0) * (1 + 0.3 * smooth(waves(rng), x, y, z)), 0.0)
    p = p + np.where(flags == 1, 0.02 * rng.standard_normal(flags.shape), 0.0)
    target = p.astype(np.float32)
    b = apply_matrix(torch.from_numpy(flags), torch.from_numpy(target).double(), spacing(case)).numpy()
    return np.ascontiguousarray(b, dtype=np.float32), flags, target


def network_parameters(seed):
    rng = np.random.default_rng(seed + 1)
    p = {}
    for name, ci, co in capi.NET_LAYERS:
        p[name] = ((rng.standard_normal((27, ci, co)) * math.sqrt(2.0 / (27 * ci))).astype(np.float32),
                   (rng.standard_normal(co) * 0.05).astype(np.float32))
    p["head"] = ((rng.standard_normal(16) * 0.25).astype(np.float32), np.float32(0.01))
    return p


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def download(scene, field, out):
    scene.ctx.check(scene.L.fe_grid_download(scene._h, field, out.ctypes.data, out.nbytes), "fe_grid_download")
    return out


def upload(scene, field, a):
    scene.ctx.check(scene.L.fe_grid_upload(scene._h, field, a.ctypes.data, a.nbytes), "fe_grid_upload")


class Particles:
    """A program's buffers for a scene's particles."""

    def __init__(self, count, apic):
        self.x = pinned((count, 3), np.float32)
        self.v = pinned((count, 3), np.float32)
        self.c = pinned((count, 9), np.float32) if apic else None

    def read(self, scene, positions=True):
        """What the scene's particles are now; without their positions where the call has not moved them."""
        x = self.x if positions else None
        scene.ctx.check(scene.L.fe_particles_download(scene._h, capi._fptr(x), capi._fptr(self.v),
                                                      capi._fptr(self.c), self.v.shape[0]), "fe_particles_download")
        return [a for a in (x, self.v, self.c) if a is not None]


def prepare(case, seed):
    ctx = context()
    kind = case["kind"]
    if kind == "frames":
        n = dims(case)
        desc, x, v = tank(n, METHODS[case["method"]], seed, case["fill"], case["viscosity"])
        scene = capi.Scene(ctx, desc)
        scene.upload_particles(x, v)
        if case["collider"]:  # a ball on the tank's floor, its mesh on the scene's nodes
            verts, tris = lathe(8, 12, (0.45, 0.05, 0.35), (0.75, 0.35, 0.65), np.random.default_rng(3))
            scene.add_mesh_collider(n, (0, 0, 0), spacing(case), verts, tris)
        return dict(kind=kind, scene=scene, out=Particles(x.shape[0], case["method"] == "apic"), dt=case["dt"],
                    frames=case["frames"],
                    solver=capi.solver(SOLVERS[case["solver"]], 2000, 0, case["tol"], relative=True, warm_start=True))
    if kind == "batch":
        scenes, outs = [], []
        for i in range(case["scenes"]):
            m = case["smallest"] + (case["largest"] - case["smallest"]) * (i * 5 % case["scenes"]) // max(1, case["scenes"] - 1)
            desc, x, v = tank((m, m, m), capi.FLIP, seed * 1009 + i, 0.2 + 0.25 * (i % 4) / 3)
            scene = capi.Scene(ctx, desc)
            scene.upload_particles(x, v)
            scenes.append(scene)
            outs.append(Particles(x.shape[0], False))
        return dict(kind=kind, scenes=scenes, outs=outs, batch=capi.Batch(ctx, scenes, case["workers"]), dt=case["dt"],
                    frames=case["frames"],
                    solver=capi.solver(capi.SOLVER_MGPCG, 2000, 0, 1e-6, relative=True, warm_start=True))
    if kind == "transfer":
        desc, x, v = tank(dims(case), METHODS[case["method"]], seed, case["fill"])
        scene = capi.Scene(ctx, desc)
        c = affine(case, seed, x) if case["method"] == "apic" else None
        scene.upload_particles(x, v, c)
        return dict(kind=kind, scene=scene, grid=[pinned(face_shape(case, a), np.float32) for a in range(3)],
                    flags=pinned((case["nz"], case["ny"], case["nx"]), np.uint8),
                    out=Particles(x.shape[0], case["method"] == "apic"))
    if kind in ("project", "diffuse"):
        n = dims(case)
        scene = capi.Scene(ctx, capi.scene_desc(n, method=capi.FLIP, max_cfl=MAX_CFL, max_particles=64,
                                                viscosity=case.get("viscosity", 0.0)))
        scene.set(capi.GRID_SDF, cell_sdf(case, 0))
        state = dict(kind=kind, scene=scene, field=face_field(case, seed),
                     grid=[pinned(face_shape(case, a), np.float32) for a in range(3)], dt=case.get("dt", 0.0))
        if kind == "project":
            state["p"] = pinned((n[2], n[1], n[0]), np.float64)
            state["solver"] = capi.solver(SOLVERS[case["solver"]], 5000, 0, case["tol"], relative=True,
                                          warm_start=False)
        return state
    if kind == "mesh_sdf":
        verts, tris = lathe(case["rings"], case["segments"], (0.1, 0.1, 0.1), (0.9, 0.9, 0.9),
                            np.random.default_rng(seed))
        return dict(kind=kind, ctx=ctx, n=dims(case), h=spacing(case), verts=verts, tris=tris)
    if kind == "surface":
        scene = capi.Scene(ctx, capi.scene_desc(dims(case), method=capi.FLIP, max_particles=64))
        scene.set_surface_mode(capi.SURFACE_CLOSED if case["mode"] == "closed" else capi.SURFACE_REFERENCE)
        sdf = cell_sdf(case, seed)
        held = pinned(sdf.shape, np.float64)
        held[...] = sdf
        return dict(kind=kind, scene=scene, sdf=held)
    if kind == "learn":
        b, flags, target = system(case, seed)
        net = capi.Net(ctx, seed=1)
        net.set_loss(capi.NET_LOSS_MSE if case["loss"] == "mse" else capi.NET_LOSS_ENERGY)
        net.set_params(capi.net_flatten(network_parameters(seed)))
        return dict(kind=kind, net=net, b=b, flags=flags, target=target, h=spacing(case))
    raise ValueError(kind)


def affine(case, seed, x):
    """The particles' affine matrices: the velocity field's gradients."""
    rng = np.random.default_rng(seed + 13)
    c = np.empty((x.shape[0], 9), np.float32)
    for q in range(9):
        c[:, q] = 2.0 * smooth(waves(rng, 2), x[:, 0], x[:, 1], x[:, 2])
    return c


def run(state):
    kind = state["kind"]
    if kind == "frames":
        for _ in range(state["frames"]):
            state["scene"].advance_frame(state["dt"], state["solver"])
        return state["out"].read(state["scene"])
    if kind == "batch":
        for _ in range(state["frames"]):
            state["batch"].advance_frame(state["dt"], state["solver"])
        return [o.read(s) for o, s in zip(state["outs"], state["scenes"])]
    if kind == "transfer":
        scene = state["scene"]
        for stage in (capi.STAGE_SORT, capi.STAGE_P2G, capi.STAGE_SDF, capi.STAGE_EXTRAPOLATE, capi.STAGE_G2P):
            scene.run_stage(stage)
        for c in range(3):
            download(scene, capi.GRID_U + c, state["grid"][c])
        download(scene, capi.GRID_FLAGS, state["flags"])
        return {"grid": state["grid"], "flags": state["flags"], "particles": state["out"].read(scene, positions=False)}
    if kind in ("project", "diffuse"):
        scene = state["scene"]
        for c in range(3):
            upload(scene, capi.GRID_U + c, state["field"][c])
        if kind == "project":
            scene.run_stage(capi.STAGE_PRESSURE, state["dt"], state["solver"])
        else:
            scene.run_stage(capi.STAGE_DIFFUSION, state["dt"])
        out = {"grid": [download(scene, capi.GRID_U + c, state["grid"][c]) for c in range(3)]}
        if kind == "project":
            out["pressure"] = download(scene, capi.GRID_PRESSURE, state["p"])
        return out
    if kind == "mesh_sdf":
        return capi.mesh_sdf(state["ctx"], state["n"], (0.0, 0.0, 0.0), state["h"], state["verts"], state["tris"])
    if kind == "surface":
        upload(state["scene"], capi.GRID_SDF, state["sdf"])
        return list(state["scene"].surface())
    loss, grads, prediction = state["net"].loss_and_grads(state["b"], state["flags"], state["target"], state["h"])
    return [loss, grads, prediction]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact its outputs are
# ---------------------------------------------------------------------------
def tank_particles(n, fill):
    """The particles of tank(), to a layer of cells."""
    return 8 * n[0] * n[1] * n[2] * min(1.0, 0.8 * fill + 0.3 * 0.7 * fill)


def work(case):
    kind = case["kind"]
    if kind == "frames":  # each frame reads and writes the particles and the pressure; the last goes to the caller
        n = dims(case)
        state = 60 if case["method"] == "apic" else 24
        return {"bytes": case["frames"] * (2 * state * tank_particles(n, case["fill"]) + 16 * n[0] * n[1] * n[2])
                + state * tank_particles(n, case["fill"]), "flops": 0}
    if kind == "batch":
        total = 0.0
        for i in range(case["scenes"]):
            m = case["smallest"] + (case["largest"] - case["smallest"]) * (i * 5 % case["scenes"]) // max(1, case["scenes"] - 1)
            total += (48 * case["frames"] + 24) * tank_particles((m, m, m), 0.2 + 0.25 * (i % 4) / 3)
            total += 16 * case["frames"] * m ** 3
        return {"bytes": total, "flops": 0}
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "transfer":  # particles in and their velocities out, face arrays and markers out
        state = 60 if case["method"] == "apic" else 24
        return {"bytes": (2 * state - 12) * tank_particles(dims(case), case["fill"]) + 13 * cells, "flops": 0}
    if kind == "project":
        return {"bytes": (12 + 1 + 12 + 8) * cells, "flops": 0}
    if kind == "diffuse":
        return {"bytes": (12 + 3 + 12) * cells, "flops": 0}
    if kind == "mesh_sdf":  # the sign is a sum over every triangle: some 60 operations for each node and triangle
        triangles = 2 * case["segments"] * (case["rings"] - 1)
        return {"bytes": 8 * cells + 36 * triangles, "flops": 60.0 * cells * triangles}
    if kind == "surface":  # two cells of the three at a crossing are new vertices of 48 bytes, with their triangles
        area = 1.3 * case["nx"] * case["nz"]
        return {"bytes": 8 * cells + area * (2 * 48 + 4 * 12), "flops": 0}
    flops = 0.0
    for (_, ci, co), level in zip(capi.NET_LAYERS, (0, 1, 2, 3, 2, 1, 0)):
        flops += 3 * 2 * 27 * ci * co * cells / 8 ** level  # forward, and both gradients
    return {"bytes": (4 + 1 + 4 + 4) * cells, "flops": flops}


def tolerance(case):
    if case.get("method") == "apic":
        return TOLERANCE["apic"]
    return TOLERANCE[case["kind"]]


# About four times what was seen: the split V-cycle and another solver against the default for whole frames and the
# projection, exact() for the others.
TOLERANCE = {
    # 2e-7 as a rule (largest 3e-5); but the particle that decides a cell's marker may land on the other side of the
    # threshold by rounding, and then the dozens of particles round that cell move otherwise from there on
    "frames": {"rel": 1e-3, "max": 0.5},
    "batch": {"rel": 1e-3, "max": 0.5},
    # the affine matrix jumps where a particle crosses from cell to cell: of 15 million entries some dozens lie so near
    # to a crossing that 32-bit positions put them on the other side, which is 1.3e-3 in all
    "apic": {"rel": 5e-3, "max": 0.9},
    "transfer": {"rel": 1e-6, "max": 2e-5},
    "project": {"rel": 2e-7, "max": 2e-6},
    "diffuse": {"rel": 1e-7, "max": 2e-6},
    # 64 bits throughout
    "mesh_sdf": {"rel": 1e-13, "max": 1e-12},
    "surface": {"rel": 1e-13, "max": 1e-12},
    # activations and their gradients are bfloat16 between the layers
    "learn": {"rel": 3e-2},
}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def shift(a, axis, step, fill=0):
    """a[i + step] along an axis, `fill` outside."""
    out = torch.full_like(a, fill)
    n = a.shape[axis]
    if step > 0:
        out.narrow(axis, 0, n - step).copy_(a.narrow(axis, step, n - step))
    else:
        out.narrow(axis, -step, n + step).copy_(a.narrow(axis, 0, n + step))
    return out


def apply_matrix(flags, p, h):
    """The pressure matrix on fluid cells: 1/h^2 for each neighbour inside the domain, fluid neighbours couple."""
    fluid = flags == 1
    p = torch.where(fluid, p, torch.zeros((), dtype=p.dtype, device=p.device))
    out = torch.zeros_like(p)
    inside = torch.ones_like(p)
    for axis, ha in ((2, h[0]), (1, h[1]), (0, h[2])):
        for step in (1, -1):
            out += (shift(inside, axis, step) * p - shift(p, axis, step)) / (ha * ha)
    return torch.where(fluid, out, torch.zeros_like(out))


def conjugate_gradients(apply, b, diag, tol=1e-14, most=6000):
    x = torch.zeros_like(b)
    r = b.clone()
    z = r / diag
    d = z.clone()
    rz = (r * z).sum()
    stop = tol * float(b.norm())
    for it in range(most):
        q = apply(d)
        alpha = rz / (d * q).sum()
        x += alpha * d
        if it % 50 == 49:
            r = b - apply(x)
        else:
            r -= alpha * q
        if it % 10 == 9 and float(r.norm()) <= stop:
            break
        z = r / diag
        new = (r * z).sum()
        d = z + (new / rz) * d
        rz = new
    return x


def stencil(x, n, origin, h):
    """Corner indices (8 of i, j, k) and fractions of positions on a grid of n nodes, clamped at its ends."""
    base, frac = [], []
    for a in range(3):
        s = (x[:, a] - origin[a]) / h[a]
        i = torch.floor(s)
        f = s - i
        f = torch.where(i < 0, torch.zeros_like(f), torch.where(i > n[a] - 2, torch.ones_like(f), f))
        base.append(i.clamp(0, n[a] - 2).long())
        frac.append(f)
    return base, frac


def corners(base, frac):
    for q in range(8):
        o = (q & 1, q >> 1 & 1, q >> 2)
        w = 1.0
        for a in range(3):
            w = w * (frac[a] if o[a] else 1 - frac[a])
        yield [base[a] + o[a] for a in range(3)], o, w


def face_origin(c, h):
    return [0.0 if a == c else 0.5 * h[a] for a in range(3)]


def inner(x, c, h):
    """Positions with the axes across component c kept half a cell from the walls."""
    p = x.clone()
    for a in range(3):
        if a != c:
            p[:, a] = x[:, a].clamp(0.5 * h[a], 1.0 - 0.5 * h[a])
    return p


def exact_transfer(case, seed):
    dev, h, n = device(), spacing(case), dims(case)
    _, x, v = tank(n, METHODS[case["method"]], seed, case["fill"])
    apic, flip = case["method"] == "apic", case["method"] == "flip"
    cm = torch.from_numpy(affine(case, seed, x)).double().to(dev) if apic else None
    x = torch.from_numpy(x).double().to(dev)
    v = torch.from_numpy(v).double().to(dev)
    grids, new_v, new_c = [], torch.empty_like(v), torch.zeros_like(cm) if apic else None
    for c in range(3):
        own = [n[a] + (a == c) for a in range(3)]
        size = own[0] * own[1] * own[2]
        o = face_origin(c, h)
        at = lambda ijk: ijk[0] + own[0] * (ijk[1] + own[1] * ijk[2])  # noqa: E731, B023
        top = torch.zeros(size, dtype=torch.float64, device=dev)
        wsum, mark = torch.zeros_like(top), torch.zeros(size, dtype=torch.bool, device=dev)
        px = inner(x, c, h)
        for ijk, _, w in corners(*stencil(x, own if flip else n, o, h)):
            value = v[:, c]
            if apic:
                for a in range(3):
                    value = value + cm[:, 3 * c + a] * (o[a] + h[a] * ijk[a] - px[:, a])
            top.index_add_(0, at(ijk), value * w)
            wsum.index_add_(0, at(ijk), w)
            mark[at(ijk)] = True
        top = torch.where(wsum > 0, top / torch.where(wsum > 0, wsum, torch.ones_like(wsum)), top)
        u = top.reshape(own[2], own[1], own[0]).clone()
        ok = mark.reshape(u.shape)
        for _ in range(int(math.ceil(MAX_CFL))):
            total, count = torch.zeros_like(u), torch.zeros_like(u)
            for axis in range(3):
                for step in (1, -1):
                    k = shift(ok, axis, step, False)
                    total += torch.where(k, shift(u, axis, step), torch.zeros_like(u))
                    count += k
            write = ~ok & (count > 0)
            u = torch.where(write, total / count.clamp(min=1), u)
            ok = ok | write
        grids.append(u)
        flat, change = u.reshape(-1), (u.reshape(-1) - top)
        pic = torch.zeros_like(v[:, c])
        delta = torch.zeros_like(pic)
        for ijk, _, w in corners(*stencil(x, own, o, h)):
            pic += w * flat[at(ijk)]
            if flip:
                delta += w * change[at(ijk)]
        new_v[:, c] = 0.97 * (v[:, c] + delta) + 0.03 * pic if flip else pic
        if apic:
            base, frac = stencil(px, n, o, h)
            for ijk, off, _ in corners(base, frac):
                val = flat[at(ijk)]
                for a in range(3):
                    g = (1.0 if off[a] else -1.0) / h[a]
                    for e in range(3):
                        if e != a:
                            g = g * (frac[e] if off[e] else 1 - frac[e])
                    new_c[:, 3 * c + a] += g * val
    parts = [new_v] + ([new_c] if apic else [])
    return {"grid": [g.cpu().numpy() for g in grids], "flags": None, "particles": [p.cpu().numpy() for p in parts]}


def exact_project(case, seed):
    dev, h = device(), spacing(case)
    u = [torch.from_numpy(f).double().to(dev) for f in face_field(case, seed)]
    flags = (torch.from_numpy(cell_sdf(case, 0)).to(dev) < 0).to(torch.uint8)
    fluid = flags == 1
    b = sum((u[c].narrow(2 - c, 1, dims(case)[c]) - u[c].narrow(2 - c, 0, dims(case)[c])) / h[c] for c in range(3))
    b = torch.where(fluid, b, torch.zeros_like(b))
    diag = torch.zeros_like(b)
    for axis, ha in ((2, h[0]), (1, h[1]), (0, h[2])):
        for step in (1, -1):
            diag += shift(torch.ones_like(b), axis, step) / (ha * ha)
    p = conjugate_gradients(lambda d: apply_matrix(flags, d, h), b, diag)
    out = []
    for c in range(3):
        axis, n = 2 - c, dims(case)[c]
        f = u[c].clone()
        # a fluid cell corrects its face towards the next cell
        grad = (p.narrow(axis, 1, n - 1) - p.narrow(axis, 0, n - 1)) / h[c]
        f.narrow(axis, 1, n - 1).add_(torch.where(fluid.narrow(axis, 0, n - 1), grad, torch.zeros_like(grad)))
        out.append(f.cpu().numpy())
    return {"grid": out, "pressure": p.cpu().numpy()}


def exact_diffuse(case, seed):
    dev, h, n = device(), spacing(case), dims(case)
    phi = torch.from_numpy(cell_sdf(case, 0)).to(dev)
    out = []
    for c, f in enumerate(face_field(case, seed)):
        axis = 2 - c
        u = torch.from_numpy(f).double().to(dev)
        ends = phi.narrow(axis, 0, 1), phi.narrow(axis, n[c] - 1, 1)
        mid = 0.5 * (phi.narrow(axis, 0, n[c] - 1) + phi.narrow(axis, 1, n[c] - 1))
        fluid = torch.cat([ends[0], mid, ends[1]], axis) < 0
        coef = [case["dt"] * case["viscosity"] / (ha * ha) for ha in h]
        diag = torch.ones_like(u)
        links = []
        for a in range(3):
            for step in (1, -1):
                k = (shift(fluid, 2 - a, step, False) & fluid).double() * coef[a]
                diag += k
                links.append((2 - a, step, k))

        def apply(d, links=links, diag=diag):
            q = diag * d
            for ax, step, k in links:
                q -= k * shift(d, ax, step)
            return q

        out.append(conjugate_gradients(apply, u, diag).cpu().numpy())
    return {"grid": out}


def exact_mesh_sdf(case, seed):
    """Distances to the triangles that a node is near, and the sign from the summed solid angles."""
    dev, h, n = device(), spacing(case), dims(case)
    if dev.type == "cpu" and n[0] * n[1] * n[2] * case["rings"] * case["segments"] > 3e7:
        return None
    verts, tris = lathe(case["rings"], case["segments"], (0.1, 0.1, 0.1), (0.9, 0.9, 0.9), np.random.default_rng(seed))
    ax = [torch.arange(n[a], dtype=torch.float64, device=dev) * h[a] for a in range(3)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    node = torch.stack([x, y, z], -1).reshape(-1, 3)
    angle = torch.zeros(node.shape[0], dtype=torch.float64, device=dev)
    dist = torch.full((n[2], n[1], n[0]), max(h) * sum(n), dtype=torch.float64, device=dev)
    for tri in verts[tris]:
        A, B, C = (torch.from_numpy(p).to(dev) - node for p in tri)
        na, nb, nc = (p.norm(dim=1) for p in (A, B, C))
        det = (A * torch.linalg.cross(B, C)).sum(1)
        k = na * nb * nc + nc * (A * B).sum(1) + na * (B * C).sum(1) + nb * (C * A).sum(1)
        angle += torch.atan2(det, k)
        # the node box of a triangle: its coordinates over the x spacing, one below and two above
        t = tri / h[0]
        lo = [min(max(int(t[:, a].min()) - 1, 0), n[a] - 1) for a in range(3)]
        hi = [min(max(int(t[:, a].max()) + 2, 0), n[a] - 1) for a in range(3)]
        box = tuple(slice(lo[a], hi[a] + 1) for a in (2, 1, 0))
        q = torch.stack([x[box], y[box], z[box]], -1)
        dist[box] = torch.minimum(dist[box], triangle_distance(q, tri))
    inside = angle.abs().reshape(dist.shape) >= 2 * math.pi - 0.001
    return torch.where(inside, -dist, dist).cpu().numpy()


def triangle_distance(q, tri):
    """The least of the distances to the three edges and, where it falls inside, to the plane."""
    dev = q.device
    p = [torch.from_numpy(a).to(dev) for a in tri]
    best = None
    for a, b in ((0, 1), (1, 2), (2, 0)):
        e = p[b] - p[a]
        s = (((q - p[a]) * e).sum(-1) / (e * e).sum()).clamp(0, 1)
        d = (q - p[a] - s[..., None] * e).norm(dim=-1)
        best = d if best is None else torch.minimum(best, d)
    nrm = torch.linalg.cross(p[1] - p[0], p[2] - p[0])
    nrm = nrm / nrm.norm()
    off = ((q - p[0]) * nrm).sum(-1)
    foot = q - off[..., None] * nrm
    side = [(torch.linalg.cross((p[b] - p[a]).expand_as(q), foot - p[a]) * nrm).sum(-1) >= 0
            for a, b in ((0, 1), (1, 2), (2, 0))]
    return torch.where(side[0] & side[1] & side[2], off.abs(), best)


def exact_learn(case, seed):
    dev = device()
    b, flags, target = system(case, seed)
    nz, ny, nx = b.shape
    if dev.type == "cpu" and b.size > 40000:
        return None
    params = {}
    for name, value in network_parameters(seed).items():
        params[name] = tuple(torch.from_numpy(np.asarray(p, np.float64)).to(dev).requires_grad_(True) for p in value)
    flags = torch.from_numpy(flags).to(dev)
    b = torch.from_numpy(b).double().to(dev)
    target = torch.from_numpy(target).double().to(dev)

    def conv(name, a):
        w, bias = params[name]
        Z, Y, X, _ = a.shape
        pad = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
        out = bias
        for t in range(27):
            dx, dy, dz = t % 3, t // 3 % 3, t // 9
            part = pad[dz:dz + Z, dy:dy + Y, dx:dx + X].reshape(Z * Y * X, -1)
            out = out + part @ w[t]
        return torch.relu(out).reshape(Z, Y, X, -1)

    def pool(a):
        Z, Y, X, C = a.shape
        return a.reshape(Z // 2, 2, Y // 2, 2, X // 2, 2, C).mean((1, 3, 5))

    def up(a):
        for axis in range(3):
            a = a.repeat_interleave(2, axis)
        return a

    x0 = torch.zeros((nz, ny, nx, 16), dtype=torch.float64, device=dev)
    x0[..., 0] = b / b.square().mean().sqrt()
    x0[..., 1] = flags == 1
    x0[..., 2] = flags == 0
    e0 = conv("enc0", x0)
    e1 = conv("enc1", pool(e0))
    e2 = conv("enc2", pool(e1))
    e3 = conv("enc3", pool(e2))
    d2 = conv("dec2", torch.cat([up(e3), e2], 3))
    d1 = conv("dec1", torch.cat([up(d2), e1], 3))
    d0 = conv("dec0", torch.cat([up(d1), e0], 3))
    out = (d0 * params["head"][0]).sum(3) + params["head"][1]
    fluid = flags == 1
    p = torch.where(fluid, out, torch.zeros_like(out))
    if case["loss"] == "mse":
        loss = torch.where(fluid, out - target, torch.zeros_like(out)).square().sum() / fluid.sum()
    else:
        q = apply_matrix(flags, p, spacing(case))
        s = (b * p).sum()
        loss = 1 - s * s / ((p * q).sum() * (b * target)[fluid].sum())
    loss.backward()
    grads = [params[name][i].grad.reshape(-1) for name in [layer[0] for layer in capi.NET_LAYERS] + ["head"]
             for i in (0, 1)]
    return [float(loss.detach()), torch.cat(grads).cpu().numpy(), out.detach().cpu().numpy()]


def exact(case, seed):
    """None for whole simulations, where 32-bit positions move a cell's marker and the trajectory with it, and for the
    surface, whose vertex order is the framework's own."""
    return {"transfer": exact_transfer, "project": exact_project, "diffuse": exact_diffuse,
            "mesh_sdf": exact_mesh_sdf, "learn": exact_learn}.get(case["kind"], lambda c, s: None)(case, seed)
