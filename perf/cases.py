"""The work a simulation program has the coupled solver do, as cases to be timed.

A pass is one output interval of such a program: a number of time steps, then the
frame it takes off the device.  The runs with platelets take the frame the host
driver writes (positions, velocities and forces of the markers, the bonds held);
those with many platelets or 16-bit storage keep positions and velocities of it
(the forces follow from the positions, and there some pair always lies within
rounding of the hard Morse cutoff).  The flow runs take density and velocity; the
channel's frames and the 128^3 box's hold both.

The trajectories are chaotic through that cutoff, so the intervals are short.

Three kinds of case:
  markers  one lattice with platelets (and fibrin, ligands) in it: the channel,
           the single platelet in shear, the tube, the large Couette lattice and
           its 128^3 box, as the scene generators build them
  batch    many small lattices stepped together
  flow     one lattice without markers

Sizes are those of the configurations in bench.py and tests/, or generic odd ones.
Everything random comes from the seed of a case.
"""
import math

import numpy as np
import torch

import platelet_fiber_gpu_amd as pfg

STORES = {"f32": pfg.STORE_F32, "f16": pfg.STORE_F16, "bf16": pfg.STORE_BF16}
VALUE_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
WALLS = {"periodic": pfg.WALL_PERIODIC, "bounce": pfg.WALL_BOUNCE, "velocity": pfg.WALL_VELOCITY}
SCENES = {"channel": pfg.SCENE_CHANNEL, "shear": pfg.SCENE_SHEAR,
          "thrombus": pfg.SCENE_THROMBUS, "large": pfg.SCENE_LARGE}


def markers(name, scene, nx, ny, nz, store, steps, platelets=1, elements=0, receptors=-1,
            ligands=-1, fibrin=-1, physics="morse", flow_frame=False, forces=True):
    return {"name": name, "kind": "markers", "scene": scene, "nx": nx, "ny": ny, "nz": nz,
            "store": store, "steps": steps, "platelets": platelets, "elements": elements,
            "receptors": receptors, "ligands": ligands, "fibrin": fibrin, "physics": physics,
            "flow_frame": flow_frame, "forces": forces}


def flow(name, nx, ny, nz, store, steps, wall_y, wall_z, tube=False):
    return {"name": name, "kind": "flow", "nx": nx, "ny": ny, "nz": nz, "store": store,
            "steps": steps, "wall_y": wall_y, "wall_z": wall_z, "tube": tube}


def batch(name, lattices, store, steps, receptors=-1):
    return {"name": name, "kind": "batch", "lattices": lattices, "store": store, "steps": steps,
            "receptors": receptors}


def listed():
    return [
        # the channel with one platelet, watched step by step: a program that
        # decides after every step (a detach test, a coupled outer solver)
        markers("channel step", "channel", 64, 32, 32, "f32", 1, elements=256),
        # the same run with a frame every 16 steps
        markers("channel interval", "channel", 64, 32, 32, "f32", 16, elements=256,
                flow_frame=True),
        # one platelet over the ligand wall in shear, full resolution
        markers("shear f32", "shear", 256, 128, 128, "f32", 8, elements=2048, receptors=512,
                ligands=4096),
        # the same platelet without its receptors (how it tumbles and deforms), FP16
        markers("shear f16", "shear", 256, 128, 128, "f16", 4, elements=2048, forces=False),
        # the physics of the parameter file (springs, area and volume, bending, the
        # force-dependent bond rates) on an odd lattice, several platelets
        markers("membrane", "shear", 150, 75, 67, "f32", 6, platelets=3, elements=958,
                receptors=256, ligands=1024, physics="membrane"),
        # the 128^3 box of the large configuration with its platelets and fibrin, FP16,
        # flow written too
        markers("box 128", "large", 128, 128, 128, "f16", 8, platelets=16, elements=1000,
                fibrin=625, flow_frame=True, forces=False),
        # a thrombus in a tube: solid flags, fibrin, 520 000 markers
        markers("tube", "thrombus", 512, 256, 256, "f32", 8, platelets=500, elements=1000,
                receptors=64, ligands=16384, fibrin=20000, forces=False),
        # the largest single-GPU run: 268 M cells, 2.08 M markers
        markers("large f16", "large", 1024, 512, 512, "f16", 8, platelets=2000, elements=1000,
                receptors=64, ligands=65536, fibrin=80000, forces=False),
        # 256 uneven vessel segments stepped together, one run per seed and shear rate
        batch("batch 256", 256, "f32", 8, receptors=32),
        # a few segments in FP16, platelets without receptors
        batch("batch 24", 24, "f16", 8),
        # flow alone: a duct of odd sizes with velocity inlet and outlet, and a
        # tube in bfloat16 storage developing under a body force
        flow("duct", 201, 99, 75, "f32", 32, "bounce", "velocity"),
        flow("tube flow", 320, 128, 128, "bf16", 32, "bounce", "bounce", tube=True),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    c = _draw(rng)
    del c["name"]
    return c


def _draw(rng):
    kind = rng.choice(["channel", "shear", "membrane", "suspension", "thrombus", "batch", "flow",
                       "flow"])
    steps = rng.choice([1, 2, 4, 6, 8])
    store = rng.choice(["f32", "f32", "f16", "f16", "bf16"])
    bonds = store == "f32"
    if kind == "channel":
        return markers("", "channel", log_int(rng, 48, 300), log_int(rng, 30, 140),
                       log_int(rng, 30, 140), store, steps if bonds else min(steps, 4),
                       elements=log_int(rng, 100, 600), forces=bonds)
    if kind == "shear":
        return markers("", "shear", log_int(rng, 64, 400), log_int(rng, 64, 200),
                       log_int(rng, 64, 200), store, steps if bonds else min(steps, 4),
                       elements=log_int(rng, 200, 2048),
                       receptors=log_int(rng, 32, 512) if bonds else -1,
                       ligands=log_int(rng, 256, 4096) if bonds else -1, forces=bonds)
    if kind == "membrane":
        return markers("", "shear", log_int(rng, 90, 300), log_int(rng, 64, 150),
                       log_int(rng, 64, 150), "f32", min(steps, 6), platelets=rng.randint(1, 3),
                       elements=log_int(rng, 200, 1000), receptors=log_int(rng, 32, 512),
                       ligands=log_int(rng, 256, 4096), physics="membrane")
    if kind in ("suspension", "thrombus"):
        nx, ny, nz = log_int(rng, 128, 512), log_int(rng, 128, 300), log_int(rng, 128, 300)
        elements = log_int(rng, 500, 1000)
        # at most the densities of the tube and of the large lattice
        room = nx * ny * nz / (90e3 if kind == "thrombus" else 134e3)
        platelets = max(2, log_int(rng, 0.25 * room, 0.9 * room))
        fibrin = max(64, int(40 * platelets * rng.uniform(0.5, 1.0)))
        scene = "thrombus" if kind == "thrombus" else "large"
        return markers("", scene, nx, ny, nz, store, steps, platelets=platelets,
                       elements=elements, receptors=64 if bonds else -1,
                       ligands=log_int(rng, 1024, 16384) if bonds else -1, fibrin=fibrin,
                       flow_frame=nx * ny * nz < 3e6, forces=False)
    if kind == "batch":
        store = rng.choice(["f32", "f16"])
        return batch("", log_int(rng, 8, 200), store, steps,
                     receptors=32 if store == "f32" else -1)
    wall_z = rng.choice(["bounce", "velocity", "periodic"])
    return flow("", log_int(rng, 32, 512), log_int(rng, 24, 200), log_int(rng, 24, 200), store,
                4 * steps, rng.choice(["periodic", "bounce"]), wall_z,
                tube=wall_z == "bounce" and rng.random() < 0.5)


# ---------------- inputs ----------------

def poiseuille_force(u_max, tau, height):
    """Body force of plane Poiseuille flow with peak u_max between walls `height` apart."""
    return 8.0 * u_max * (tau - 0.5) / 3.0 / height ** 2


def marker_scene(case, seed):
    c = case
    kw = dict(seed=seed + 1, nx=c["nx"], ny=c["ny"], nz=c["nz"], n_platelets=c["platelets"],
              elements=c["elements"], receptors=c["receptors"], ligands=c["ligands"],
              store=STORES[c["store"]], fibrin_nodes=c["fibrin"])
    if c["fibrin"] > 0:
        kw["fibrin_links"] = c["fibrin"] * 3 // 2
    if c["scene"] == "thrombus":  # the scene's own radius, inside a box of any shape
        kw["tube_radius"] = 0.47 * min(c["ny"], c["nz"])
    sc = pfg.Scene(SCENES[c["scene"]], **kw)
    p = sc.params
    if c["scene"] == "channel":
        z = (np.arange(p.nz) + 0.5) / p.nz
        p.body_force[0] = poiseuille_force(0.02, p.tau, p.nz)
        sc.u0_z[0][:] = 0.08 * z * (1.0 - z)
    if c["scene"] == "large":  # the shear rate of a 0.05 wall velocity over 512 cells
        p.wall_u_hi[2][0] = 0.05 * p.nz / 512
        p.detach_rate = 0.05 / 512
        sc.u0_z[0][:] = p.wall_u_hi[2][0] * (np.arange(p.nz) + 0.5) / p.nz
    if c["physics"] == "membrane":
        p.morse_u0 = 0.0
        p.k_spring, p.ks, p.kv, p.kbend = 0.3, 0.5, 0.4, 0.5
        p.wall_rep_a = 1e-3
        p.bond_law = pfg.BOND_REFERENCE
    return sc


def batch_scenes(case, seed):
    """Vessel segments: each axis 32 to 96 cells, 1 to 8 platelets of 256 elements as
    they fit (the batch's own, whatever the seed), wall shear log-uniform over two
    decades."""
    sizes = np.random.default_rng(case["lattices"])
    rng = np.random.default_rng(seed)
    scenes = []
    for k in range(case["lattices"]):
        nx, ny, nz = (int(v) for v in sizes.integers(32, 97, size=3))
        room = nx * (ny - 14) * (nz - 14) // 10000  # centres stay off the walls
        n = min(int(sizes.integers(1, 9)), max(1, room))
        for again in range(100):  # a placement that does not fit is drawn again
            try:
                sc = pfg.Scene(pfg.SCENE_BATCH, nx=nx, ny=ny, nz=nz, n_platelets=n, elements=256,
                               receptors=case["receptors"],
                               ligands=512 if case["receptors"] > 0 else -1,
                               store=STORES[case["store"]],
                               seed=int(rng.integers(1, 2 ** 31)))
                break
            except pfg.PfgError:
                if again == 99:
                    raise
        u = 0.05 * math.exp(rng.uniform(math.log(0.01), 0.0)) * nz / 96.0
        sc.params.wall_u_hi[2][0] = u
        sc.u0_z[0][:] = u * (np.arange(nz) + 0.5) / nz
        scenes.append(sc)
    return scenes


def flow_inputs(case, seed):
    """Parameters, solid flags (or None) and the initial density and velocity: the
    developed profile with long waves of a tenth of its peak on it."""
    c = case
    p = pfg.default_params(nx=c["nx"], ny=c["ny"], nz=c["nz"], tau=0.8,
                           store=STORES[c["store"]])
    p.wall[1], p.wall[2] = WALLS[c["wall_y"]], WALLS[c["wall_z"]]
    p.use_flags = int(c["tube"])
    rng = np.random.default_rng(seed)
    x, y, z = (np.arange(n, dtype=np.float32) for n in (c["nx"], c["ny"], c["nz"]))
    shape = np.ones((c["nz"], c["ny"], 1), np.float32)
    flags = None
    if c["tube"]:
        r2 = ((y[None, :] - 0.5 * (c["ny"] - 1)) ** 2 + (z[:, None] - 0.5 * (c["nz"] - 1)) ** 2)
        radius = 0.47 * min(c["ny"], c["nz"])
        flags = np.broadcast_to((r2 > radius ** 2)[:, :, None],
                                (c["nz"], c["ny"], c["nx"])).astype(np.uint8)
        shape = np.maximum(0.0, 1.0 - r2 / radius ** 2)[:, :, None].astype(np.float32)
    else:
        if c["wall_y"] == "bounce":
            s = (y + 0.5) / c["ny"]
            shape = shape * (4 * s * (1 - s))[None, :, None]
        if c["wall_z"] == "bounce":
            s = (z + 0.5) / c["nz"]
            shape = shape * (4 * s * (1 - s))[:, None, None]
    phase = rng.uniform(0, 2 * np.pi, 6).astype(np.float32)
    wave = [np.sin(2 * np.pi * (x / c["nx"])[None, None, :] + phase[0])
            * np.cos(2 * np.pi * (y / c["ny"])[None, :, None] + phase[1])
            * np.cos(2 * np.pi * (z / c["nz"])[:, None, None] + phase[k]) for k in (2, 3, 4, 5)]
    amp = rng.uniform(0.5, 1.0, 4).astype(np.float32)
    rho = 1.0 + 1e-3 * amp[0] * wave[0]
    u = [8e-3 * a * w for a, w in zip(amp[1:], wave[1:])]
    along = 2 if c["wall_z"] == "velocity" else 0
    u[along] = u[along] + 0.05 * shape
    if along == 2:
        p.wall_u_lo[2][2] = p.wall_u_hi[2][2] = 0.05
    else:
        p.body_force[0] = poiseuille_force(0.05, p.tau, min(c["ny"], c["nz"]))
    return p, flags, [np.ascontiguousarray(a, np.float32) for a in (rho, *u)]


class Run:
    """A run under way: the solver and what its frames hold."""

    def __init__(self, solver, case):
        self.solver, self.steps, self.kind = solver, case["steps"], case["kind"]
        self.flow_frame = case["kind"] == "flow" or case.get("flow_frame", False)
        self.bonds = solver.n_rec > 0
        self.frame = ("x", "y", "z", "vx", "vy", "vz")
        if case.get("forces", False):
            self.frame += ("fx", "fy", "fz")


def prepare(case, seed):
    if case["kind"] == "flow":
        p, flags, start = flow_inputs(case, seed)
        s = pfg.Solver(p)
        if flags is not None:
            s.upload_flags(flags)
        s.init_equilibrium(*start)
    elif case["kind"] == "batch":
        scenes = batch_scenes(case, seed)
        s = pfg.Batch([sc.params for sc in scenes])
        s.load_scenes(scenes)
    else:
        sc = marker_scene(case, seed)
        s = pfg.Solver(sc.params)
        s.load(sc)
    return Run(s, case)


def run(state):
    s = state.solver
    info = s.step(state.steps)
    out = {}
    if state.kind != "flow":
        m = s.markers()
        out.update((k, m[k]) for k in state.frame)
        out["total_bonds"] = info["total_bonds"]
    if state.bonds:
        out["rec_bond"] = s.bonds()[0]
    if state.flow_frame:
        out["rho"], out["ux"], out["uy"], out["uz"] = s.fields()
    return out


def work(case):
    """Each step reads and writes the 19 populations of every cell that is not solid
    once, and of every marker the position and what moves it; the frame is written
    once.  A cell takes about 250 operations, a marker's two stencils 64 nodes each
    and its neighbours about 40 pairs."""
    c = case
    if c["kind"] == "batch":
        cells = c["lattices"] * 64.0 ** 3
        n = c["lattices"] * 4.5 * 256
    else:
        cells = float(c["nx"] * c["ny"] * c["nz"])
        if c.get("tube") or c.get("scene") == "thrombus":
            cells = c["nx"] * math.pi * (0.47 * min(c["ny"], c["nz"])) ** 2
        n = 0
        if c["kind"] == "markers":
            n = c["platelets"] * c["elements"] + max(0, c["fibrin"])
    frame = (36.0 if c.get("forces") else 24.0) * n + (16.0 * cells if c["kind"] == "flow" or c.get("flow_frame") else 0.0)
    per_step = cells * 2 * 19 * VALUE_BYTES[c["store"]] + n * 2 * 24.0
    return {"bytes": c["steps"] * per_step + frame,
            "flops": c["steps"] * (250.0 * cells + n * (2 * 64 * 9 + 40 * 20))}


# ---------------- the same in 64 bits ----------------

CX = (0, 1, -1, 0, 0, 0, 0, 1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0)
CY = (0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1)
CZ = (0, 0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 1, -1)
OPP = (0, 2, 1, 4, 3, 6, 5, 12, 11, 14, 13, 8, 7, 10, 9, 18, 17, 16, 15)
W = (1 / 3,) + (1 / 18,) * 6 + (1 / 36,) * 12


class Lattice64:
    """D3Q19 BGK with Guo forcing on [nz][ny][nx] in 64 bits: pull streaming, halfway
    bounce-back at walls (moving ones too) and solid cells, velocity faces on z."""

    def __init__(self, p, solid, rho, u):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.n = (p.nz, p.ny, p.nx)
        self.periodic = [p.wall[a] == pfg.WALL_PERIODIC for a in range(3)]
        self.faces = p.wall[2] == pfg.WALL_VELOCITY
        self.u_wall = [[[float(v[a][k]) for k in range(3)] for v in (p.wall_u_lo, p.wall_u_hi)]
                       for a in range(3)]
        self.omega, self.g = 1.0 / float(p.tau), [float(p.body_force[k]) for k in range(3)]
        self.solid = None
        if solid is not None:
            self.solid = torch.as_tensor(solid.astype(bool), device=self.dev).reshape(self.n)
        rho, *u = (self.tensor(a) for a in (rho, *u))
        self.f = torch.stack([self.equilibrium(d, rho, u) for d in range(19)])

    def tensor(self, a):
        return torch.as_tensor(np.asarray(a, np.float64), device=self.dev).expand(self.n)

    @staticmethod
    def equilibrium(d, rho, u):
        cu = CX[d] * u[0] + CY[d] * u[1] + CZ[d] * u[2]
        usq = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
        return W[d] * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * usq)

    def pulled(self):
        """The populations after streaming."""
        f = self.f
        out = torch.empty_like(f)
        for d in range(19):
            c = (CX[d], CY[d], CZ[d])
            g = torch.roll(f[d], (c[2], c[1], c[0]), (0, 1, 2))
            if self.solid is not None and d:
                up = torch.roll(self.solid, (c[2], c[1], c[0]), (0, 1, 2))
                g = torch.where(up, f[OPP[d]], g)
            for axis in range(3):  # the z walls last: they win at an edge
                if c[axis] == 0 or self.periodic[axis]:
                    continue
                lower = c[axis] > 0
                at = [slice(None)] * 3
                at[2 - axis] = 0 if lower else -1
                v = self.u_wall[axis][0 if lower else 1]
                g[tuple(at)] = f[OPP[d]][tuple(at)] + 6.0 * W[d] * sum(
                    c[k] * v[k] for k in range(3))
            out[d] = g
        if self.faces:
            for s in (1, -1):
                self.velocity_face(out, s)
        return out

    def velocity_face(self, f, s):
        at = 0 if s > 0 else -1
        q = torch.ones(self.n[1], self.n[2], dtype=torch.float64, device=self.dev)
        rim = torch.zeros_like(q, dtype=torch.bool)
        for axis, dim in ((0, 1), (1, 0)):
            if self.periodic[axis]:
                continue
            n = q.shape[dim]
            t = torch.arange(n, dtype=torch.float64, device=self.dev) + 0.5
            line = 4.0 * t * (n - t) / n ** 2
            q = q * (line[None, :] if dim else line[:, None])
            edge = torch.zeros(n, dtype=torch.bool, device=self.dev)
            edge[0] = edge[-1] = True
            rim |= edge[None, :] if dim else edge[:, None]
        u = [v * q for v in self.u_wall[2][0 if s > 0 else 1]]
        face = [f[d][at].clone() for d in range(19)]
        level = sum(face[d] for d in range(19) if CZ[d] == 0)
        leaving = sum(face[d] for d in range(19) if CZ[d] == -s)
        rho = (level + 2.0 * leaving) / (1.0 - s * u[2])
        nx = 0.5 * sum(CX[d] * face[d] for d in range(19) if CZ[d] == 0) - rho * u[0] / 3.0
        ny = 0.5 * sum(CY[d] * face[d] for d in range(19) if CZ[d] == 0) - rho * u[1] / 3.0
        for d in range(19):
            new = face[d]
            if CZ[d] == s:
                if CX[d]:
                    t = rho * (s * u[2] + CX[d] * u[0]) / 6.0 - CX[d] * nx
                elif CY[d]:
                    t = rho * (s * u[2] + CY[d] * u[1]) / 6.0 - CY[d] * ny
                else:
                    t = s * rho * u[2] / 3.0
                new = face[OPP[d]] + t
            f[d][at] = torch.where(rim, self.equilibrium(d, torch.ones_like(q), u), new)

    def moments(self, f, force):
        rho = f.sum(0)
        j = [sum(c[d] * f[d] for d in range(19) if c[d]) for c in (CX, CY, CZ)]
        return rho, [(j[k] + 0.5 * force[k]) / rho for k in range(3)]

    def step(self, extra=None):
        """One step; `extra`: a force per cell beside the uniform one. The velocity."""
        f = self.pulled()
        force = [self.g[k] + (0.0 if extra is None else extra[k]) for k in range(3)]
        rho, u = self.moments(f, force)
        u_f = sum(u[k] * force[k] for k in range(3))
        for d in range(19):
            c = (CX[d], CY[d], CZ[d])
            cu = sum(c[k] * u[k] for k in range(3) if c[k]) if d else 0.0
            cf = sum(c[k] * force[k] for k in range(3) if c[k]) if d else 0.0
            new = f[d] + self.omega * (self.equilibrium(d, rho, u) - f[d])
            new += (1.0 - 0.5 * self.omega) * W[d] * (3.0 * (cf - u_f) + 9.0 * cu * cf)
            f[d] = new if self.solid is None else torch.where(self.solid, self.f[d], new)
        self.f = f
        return u

    def fields(self):
        rho, u = self.moments(self.pulled(), self.g)
        if self.solid is not None:
            rho, u = rho.masked_fill(self.solid, 0.0), [v.masked_fill(self.solid, 0.0) for v in u]
        return {k: v.reshape(-1).cpu().numpy() for k, v in zip(("rho", "ux", "uy", "uz"),
                                                               (rho, *u))}


def morse64(p, x, body):
    """Morse forces between the elements of each platelet within the cutoff."""
    out = torch.zeros_like(x)
    for b in torch.unique(body[body >= 0]):
        at = torch.nonzero(body == b).reshape(-1)
        d = x[at][None, :, :] - x[at][:, None, :]
        r = d.square().sum(-1).sqrt()
        near = (r < float(p.morse_cutoff)) & (r > 0)
        e = torch.exp(-float(p.morse_rho) * (r - float(p.morse_req)))
        c = 2.0 * float(p.morse_rho) * float(p.morse_u0) * (e - e * e)
        c = torch.where(near, c / r.clamp_min(1e-30), torch.zeros_like(c))
        out[at] = (c[:, :, None] * d).sum(1)
    return out


def links64(p, x, link, l0):
    """Worm-like-chain forces of the fibrin links."""
    i, j = link[0::2], link[1::2]
    d = x[j] - x[i]
    length = d.square().sum(-1).sqrt()
    s = ((length - l0) / l0).clamp_max(float(p.fiber_xmax))
    pull = float(p.fiber_k) / l0 * (0.25 / (1.0 - s) ** 2 - 0.25 + s) / length
    out = torch.zeros_like(x)
    out.index_add_(0, i, pull[:, None] * d)
    out.index_add_(0, j, -pull[:, None] * d)
    return out


def stencil64(lat, x):
    """Cell indices and weights [markers][64] of the 4-point cosine kernel."""
    idx = torch.zeros(len(x), 1, dtype=torch.int64, device=x.device)
    w = torch.ones(len(x), 1, dtype=torch.float64, device=x.device)
    for axis in (2, 1, 0):
        n = lat.n[2 - axis]
        v = x[:, axis]
        if lat.periodic[axis]:
            v = v - n * torch.floor(v / n)
        node = torch.floor(v)[:, None] - 1 + torch.arange(4, device=x.device)
        phi = 0.25 * (1.0 + torch.cos(0.5 * math.pi * (v[:, None] - node)))
        if lat.periodic[axis]:
            node = node % n
        else:
            phi = torch.where((node < 0) | (node >= n), torch.zeros_like(phi), phi)
            node = node.clamp(0, n - 1)
        idx = (idx[:, :, None] * n + node.long()[:, None, :]).reshape(len(x), -1)
        w = (w[:, :, None] * phi[:, None, :]).reshape(len(x), -1)
    return idx, w


def platelets64(sc, steps, flow_frame):
    """`steps` coupled steps of a scene whose platelets have Morse forces and no
    receptors: the frame's positions, velocities and forces, and the flow."""
    p = sc.params
    lat = Lattice64(p, sc.flags, 1.0, [v[:, None, None] for v in sc.u0_z])
    cells = p.nx * p.ny * p.nz
    x = torch.as_tensor(np.stack([sc.x, sc.y, sc.z], 1).astype(np.float64), device=lat.dev)
    body = torch.as_tensor(sc.body, device=lat.dev)
    link = torch.as_tensor(sc.link.astype(np.int64), device=lat.dev)
    l0 = torch.as_tensor(sc.link_l0.astype(np.float64), device=lat.dev)
    moves = torch.as_tensor(sc.kind != pfg.MARKER_FIXED, device=lat.dev)[:, None]
    for _ in range(steps):
        force = morse64(p, x, body)
        if len(l0):
            force = force + links64(p, x, link, l0)
        idx, w = stencil64(lat, x)
        w = w * moves  # an anchored node neither spreads nor moves
        extra = []
        for k in range(3):
            a = torch.zeros(cells, dtype=torch.float64, device=lat.dev)
            a.index_add_(0, idx.reshape(-1),
                         (w * force[:, k:k + 1] * float(p.ib_force_scale)).reshape(-1))
            extra.append(a.reshape(lat.n))
        u = lat.step(extra)
        v = torch.stack([(w * u[k].reshape(-1)[idx]).sum(1) for k in range(3)], 1)
        x = x + float(p.marker_dt) * v
    out = {}
    for names, a in (("xyz", x), (("vx", "vy", "vz"), v), (("fx", "fy", "fz"), force)):
        out.update({k: a[:, i].cpu().numpy() for i, k in enumerate(names)})
    if flow_frame:
        out.update(lat.fields())
    return out


def exact(case, seed):
    """Flow runs, and runs whose platelets have Morse forces and no receptors."""
    if case["kind"] == "flow":
        p, flags, (rho, *u) = flow_inputs(case, seed)
        lat = Lattice64(p, flags, rho, u)
        for _ in range(case["steps"]):
            lat.step()
        return lat.fields()
    if case["receptors"] > 0 or case.get("physics") == "membrane":
        return None
    if case["kind"] == "batch":
        runs = [platelets64(sc, case["steps"], False) for sc in batch_scenes(case, seed)]
        out = {k: np.concatenate([r[k] for r in runs]) for k in runs[0]}
    else:
        out = platelets64(marker_scene(case, seed), case["steps"], case["flow_frame"])
    if not case.get("forces", False):
        out = {k: v for k, v in out.items() if k not in ("fx", "fy", "fz")}
    return out
