"""The work that programs built on biblbm_amd have it do, as timed cases.

Every case is one stretch of simulation through the public entry points: a
number of coupled time steps (or lattice-only steps), then the velocity field
and the vertices read back, as a program does between two outputs.  Programs
keep their output buffers, so the field goes into page-locked memory that
belongs to the state.

Families
  box       one deformable cell in a shear box (velocity walls at the two y
            faces): the shear set-ups of the progs and of the benchmark
  pipe      one red cell in a body-force driven pipe along x, bounce-back on
            the cells outside or the curved (Guo) wall the pipe prog defaults to
  channel   many red cells and platelets between bounce-back planes: the
            suspension
  vortex    a fully periodic vortex lattice with a few capsules, far larger
            than any cache: the Taylor-Green box of the benchmark
  ensemble  independent shear boxes of several sizes advanced together
  lattice   a driven channel without particles, odd sizes

`graph` says how steps are issued: true hands a run of steps to
coupled_steps, false calls the immersed-boundary step and collideAndStream one
after the other from the program, which is what a program written against the
reference's class names does.  `lam` is the viscosity ratio of the cells'
inside to the outside; other than 1 it needs the inside voxelised each step.

exact() is the same physics in plain torch, FP64, on the same inputs.
"""
import math

import numpy as np
import torch

SKALAK_CAPSULE, SKALAK_RBC = 0, 3  # membrane models, as bl_particle_add numbers them


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest call: a 24-cell box stepped stage by stage, as a prog's
        # own loop does it; launches and latency are all of it.
        dict(name="box_24_stages", family="box", nx=24, ny=24, nz=24, storage="f64", kernel="roma", level=2,
             model="capsule", lam=1.0, graph=False, steps=20),
        # The capsule-in-shear prog's set-up at the benchmark's size.
        dict(name="box_64", family="box", nx=64, ny=64, nz=64, storage="f64", kernel="peskin", level=3,
             model="capsule", lam=1.0, graph=True, steps=100),
        # A red cell with a viscous inside (ratio 5) in a sheared box of odd sides.
        dict(name="box_75_viscous", family="box", nx=75, ny=61, nz=83, storage="f64", kernel="peskin", level=4,
             model="rbc", lam=5.0, graph=True, steps=50),
        # The pipe of the benchmark (257 x 67 x 67), bounce-back.
        dict(name="pipe_257", family="pipe", nx=257, R=32.0, wall="bounce", storage="f64", kernel="peskin", level=4,
             model="rbc", lam=1.0, graph=True, steps=100),
        # The same pipe with the curved wall, the pipe prog's default, in FP32.
        dict(name="pipe_257_guo", family="pipe", nx=257, R=31.6, wall="guo", storage="f32", kernel="peskin", level=4,
             model="rbc", lam=1.0, graph=True, steps=60),
        # A short, narrow pipe stepped from the program: a small flow cell, FP32.
        dict(name="pipe_91_stages", family="pipe", nx=91, R=14.0, wall="bounce", storage="f32", kernel="peskin",
             level=2, model="rbc", lam=1.0, graph=False, steps=40),
        # The 400-cell suspension of the benchmark in its two reduced storages.
        dict(name="channel_512_f32", family="channel", nx=512, ny=128, nz=128, storage="f32", kernel="peskin",
             lam=1.0, graph=True, steps=50),
        dict(name="channel_512_f16s", family="channel", nx=512, ny=128, nz=128, storage="f16s", kernel="peskin",
             lam=1.0, graph=True, steps=50),
        # A suspension that fills a smaller channel of odd sides, FP64.
        dict(name="channel_171", family="channel", nx=171, ny=70, nz=101, storage="f64", kernel="peskin", lam=1.0,
             graph=True, steps=50),
        # The benchmark's headline: 384^3 FP64, out of every cache.
        dict(name="vortex_384", family="vortex", nx=384, ny=384, nz=384, storage="f64", kernel="peskin", caps=16,
             level=3, lam=1.0, graph=True, steps=40),
        # Sixty-four shear boxes in one batch.
        dict(name="ensemble_64", family="ensemble", boxes=64, side_min=32, side_max=64, storage="f64", kernel="peskin",
             level=3, graph=True, steps=60),
        # No particles: a driven channel of odd sides, FP32.
        dict(name="lattice_301", family="lattice", nx=301, ny=129, nz=181, storage="f32", graph=True, steps=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["box", "box", "pipe", "pipe", "channel", "channel", "vortex", "ensemble", "lattice"])
    storage = rng.choice(["f64", "f64", "f32", "f16s"])
    if family == "box":
        n = _log_int(rng, 24, 100)
        lam = rng.choice([1.0, 1.0, 5.0])
        return dict(family="box", nx=n, ny=max(24, n + rng.randint(-9, 9)), nz=max(24, n + rng.randint(-9, 9)),
                    storage="f64" if lam != 1.0 else storage, kernel=rng.choice(["roma", "peskin"]),
                    level=2 if n < 48 else (3 if n < 76 else 4), model=rng.choice(["capsule", "rbc"]), lam=lam,
                    graph=rng.random() < 0.7, steps=rng.randint(10, 100))
    if family == "pipe":
        R = float(_log_int(rng, 15, 34))  # the cell is 3/8 of it; the explicit step cannot take finer meshes on it
        return dict(family="pipe", nx=_log_int(rng, 48, 300), R=R - 0.4, wall=rng.choice(["bounce", "guo"]),
                    storage=storage, kernel="peskin", level=2 if R < 20 else 3 if R < 30 else 4, model="rbc", lam=1.0,
                    graph=rng.random() < 0.7, steps=rng.randint(10, 100))
    if family == "channel":
        return dict(family="channel", nx=_log_int(rng, 96, 512), ny=rng.randint(66, 128), nz=rng.randint(64, 128),
                    storage=storage, kernel="peskin", lam=1.0, graph=True, steps=rng.randint(10, 50))
    if family == "vortex":
        n = _log_int(rng, 96, 320)
        return dict(family="vortex", nx=n, ny=n + rng.randint(-20, 20), nz=n + rng.randint(-20, 20), storage=storage,
                    kernel=rng.choice(["roma", "peskin"]), caps=rng.randint(2, 16), level=3, lam=1.0, graph=True,
                    steps=rng.randint(10, 40))
    if family == "ensemble":
        return dict(family="ensemble", boxes=_log_int(rng, 4, 64), side_min=32, side_max=rng.choice([40, 48, 56, 64]),
                    storage=rng.choice(["f64", "f32"]), kernel="peskin", level=3, graph=True, steps=rng.randint(10, 60))
    return dict(family="lattice", nx=_log_int(rng, 40, 400), ny=rng.randint(33, 160), nz=rng.randint(33, 260),
                storage=storage, graph=True, steps=rng.randint(10, 100))


# ----------------------------------------------------------------- the inputs
def _sphere(level):
    """Unit icosphere: vertices and outward triangles."""
    g = (1 + 5 ** 0.5) / 2
    v = np.array([[s * a, t * b, 0.0] for s in (1, -1) for t in (1, -1) for a, b in ((1, g),)])
    v = np.concatenate([v, v[:, [2, 0, 1]], v[:, [1, 2, 0]]])
    d = np.linalg.norm(v[:, None] - v[None], axis=2)
    near = np.abs(d - 2) < 1e-9
    tri = np.array([(i, j, k) for i in range(12) for j in range(i + 1, 12) for k in range(j + 1, 12)
                    if near[i, j] and near[j, k] and near[i, k]])
    v = v / np.linalg.norm(v, axis=1, keepdims=True)
    for _ in range(level):
        e = np.sort(np.concatenate([tri[:, [0, 1]], tri[:, [1, 2]], tri[:, [2, 0]]]), axis=1)
        e, back = np.unique(e, axis=0, return_inverse=True)
        mid = v[e].sum(1)
        ab, bc, ca = (back.reshape(3, -1) + len(v))
        v = np.concatenate([v, mid / np.linalg.norm(mid, axis=1, keepdims=True)])
        a, b, c = tri.T
        tri = np.concatenate([np.stack(t, 1) for t in ((a, ab, ca), (ab, b, bc), (ca, bc, c), (ab, bc, ca))])
    p, q, r = v[tri[:, 0]], v[tri[:, 1]], v[tri[:, 2]]
    flip = (p * np.cross(q, r)).sum(1) < 0
    tri[flip] = tri[flip][:, [0, 2, 1]]
    return v, tri.astype(np.int32)


def _disc(level, radius):
    """Evans and Fung's biconcave red cell (Microvasc. Res. 4 (1972) 335), axis z."""
    v, t = _sphere(level)
    r2 = np.clip(v[:, 0] ** 2 + v[:, 1] ** 2, 0, 1)
    z = 0.5 * np.sqrt(1 - r2) * (0.207 + 2.003 * r2 - 1.123 * r2 * r2)
    return np.stack([v[:, 0], v[:, 1], np.sign(v[:, 2]) * z], 1) * radius, t


def _volume(v, t):
    return float((v[t[:, 0]] * np.cross(v[t[:, 1]], v[t[:, 2]])).sum() / 6)


def _rotation(axis, angle):
    a = np.asarray(axis, float)
    a = a / np.linalg.norm(a)
    k = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
    return np.eye(3) + np.sin(angle) * k + (1 - np.cos(angle)) * (k @ k)


def _rbc_params(G, C, R, volume, kb):
    extra = 18 * G  # area modulus 20 G less the 2 G of the in-plane law
    return [G, C, 0.8 * extra, 0.2 * extra, 1000 * G / R, volume, 2 * kb / math.sqrt(3)]


def _shear(nx, ny, nz, level, model, rng, tau, Ca, radius=None, kernel="peskin", lam=1.0):
    """One cell in a box between moving walls: the description both prepare and exact start from."""
    R = radius or (8.0 if model == "capsule" else 12.0) * min(ny, nx, nz) / 64.0
    mu = (tau - 0.5) / 3
    if model == "capsule":
        wall = 0.01 * (ny - 1) / 63.0
        G = mu * 2 * wall / (ny - 1) * R / Ca
        v, t = _sphere(level)
        v = v * R
        kind, params = SKALAK_CAPSULE, [G, 10.0]
        rot = np.eye(3)
    else:
        G = 0.002
        wall = Ca * G / (mu * R) * (ny - 1) / 2
        v, t = _disc(level, R)
        kind, params = SKALAK_RBC, _rbc_params(G, 10.0, R, _volume(v, t), 0.02 * G * R * R)
        rot = _rotation(rng.normal(size=3), rng.uniform(0, np.pi))
    centre = np.array([nx / 2, (ny - 1) / 2, nz / 2]) + rng.uniform(-0.5, 0.5, 3)
    prof = np.zeros((1, ny, 1, 3))
    prof[..., 0] = (wall * (2 * np.arange(ny) / (ny - 1) - 1))[None, :, None]
    mask = np.zeros((nx, ny, nz), np.uint8)
    mask[:, [0, -1]] = 3
    return dict(shape=(nx, ny, nz), periodic=(1, 0, 1), omega=1 / tau, lam=lam, tau=tau, mask=mask, wall_u=wall,
                g=np.zeros(3), u0=("profile", prof), kernel=kernel, meshes=[(v, t)],
                particles=[(0, kind, params, v @ rot.T + centre)], guo=None)


def _setup(case, seed):
    """A case's physical description from its seed, in plain numpy (a list of them for an ensemble)."""
    rng = np.random.default_rng([int(seed) & 0x7fffffff, 77])
    family, kernel, lam = case["family"], case.get("kernel"), case.get("lam", 1.0)
    if family == "box":
        return _shear(case["nx"], case["ny"], case["nz"], case["level"], case["model"], rng,
                      1.0 if case["model"] == "capsule" else rng.uniform(0.8, 1.1), rng.uniform(0.08, 0.2), None,
                      kernel, lam)
    if family == "ensemble":
        sides = [s for s in (32, 40, 48, 56, 64) if case["side_min"] <= s <= case["side_max"]]
        # the same sides for every seed, so that every state has the same work
        return [_shear(s, s, s, case["level"], "rbc", rng, rng.uniform(0.7, 1.2),
                       math.exp(rng.uniform(math.log(0.05), math.log(0.5))), 0.16 * s, kernel)
                for s in np.random.default_rng(11).choice(sides, case["boxes"]).tolist()]
    if family == "pipe":
        R, nx, tau, uc = case["R"], case["nx"], 0.9, 0.02 * rng.uniform(0.9, 1.1)
        n = 2 * int(math.ceil(R)) + 3
        c = (n - 1) / 2
        yy, zz = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
        r = np.sqrt((yy - c) ** 2 + (zz - c) ** 2)
        solid = np.where(r > R, 1, 0) if case["wall"] == "bounce" else np.where(r > R + 1, 2, 0)
        nu = (tau - 0.5) / 3
        prof = np.zeros((1, n, n, 3))
        prof[..., 0] = np.where(r <= R, uc * (1 - (r / R) ** 2), 0)[None]
        a = 0.375 * R
        G = nu * uc / R * a / 0.1
        v, t = _disc(case["level"], a)
        rot = _rotation([0, 1, 0], np.pi / 2) @ _rotation([1, 0, 0], rng.uniform(0, np.pi))
        centre = np.array([nx / 2, c, c]) + rng.uniform(-1, 1, 3)
        return dict(shape=(nx, n, n), periodic=(1, 0, 0), omega=1 / tau, lam=lam, tau=tau,
                    mask=np.broadcast_to(solid.astype(np.uint8), (nx, n, n)).copy(), wall_u=None,
                    g=np.array([4 * nu * uc / (R * R), 0, 0]), u0=("profile", prof), kernel=kernel, meshes=[(v, t)],
                    particles=[(0, SKALAK_RBC, _rbc_params(G, 10.0, a, _volume(v, t), 0.02 * G * a * a),
                                v @ rot.T + centre)],
                    guo=(c, R) if case["wall"] == "guo" else None)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if family in ("channel", "lattice"):
        tau, uc = 1.0, 0.02 * rng.uniform(0.9, 1.1)
        nu, H = (tau - 0.5) / 3, (ny - 2) / 2
        prof = np.zeros((1, ny, 1, 3))
        prof[0, :, 0, 0] = np.clip(uc * (1 - ((np.arange(ny) - (ny - 1) / 2) / H) ** 2), 0, None)
        mask = np.zeros((nx, ny, nz), np.uint8)
        mask[:, [0, -1]] = 1
        d = dict(shape=(nx, ny, nz), periodic=(1, 0, 1), omega=1 / tau, lam=lam, tau=tau, mask=mask, wall_u=None,
                 g=np.array([2 * nu * uc / (H * H), 0, 0]), u0=("profile", prof, 0.002, rng.uniform(0, 6, 6)),
                 kernel=kernel, meshes=[], particles=[], guo=None)
        if family == "lattice":
            return d
        # discs whose axes lie within 20 degrees of the flow, on a jittered grid that keeps them apart, and
        # platelets in the place of some: about 18 % of the volume
        a = 13.5
        G = nu * uc / H * a / 0.1
        small, large, plate = _disc(3, a), _disc(4, a), _sphere(2)
        plate = (plate[0] * [3.0, 3.0, 1.2], plate[1])
        d["meshes"] = [small, large, plate]
        kx, ky, kz = nx // 20, int((ny - 4) // 30.5), int(nz // 30.5)
        sites = [((i + 0.5) * nx / kx, 1.5 + (j + 0.5) * (ny - 4) / ky, (k + 0.5) * nz / kz)
                 for i in range(kx) for j in range(ky) for k in range(kz)]
        # one site in five a large mesh, one in twenty a platelet: the same counts for every seed
        kinds = [1 if s % 5 == 2 else (2 if s % 20 == 4 else 0) for s in range(len(sites))]
        for kind, site in zip(rng.permutation(kinds).tolist(), sites):
            v, t = d["meshes"][kind]
            az = rng.uniform(0, 2 * np.pi)
            rot = _rotation([0, np.cos(az), np.sin(az)], rng.uniform(0, np.pi / 9)) @ _rotation([0, 1, 0], np.pi / 2)
            pos = v @ rot.T + np.array(site) + rng.uniform(-0.4, 0.4, 3)
            if kind == 2:
                d["particles"].append((kind, SKALAK_CAPSULE, [20 * G, 10.0], pos))
            else:
                d["particles"].append((kind, SKALAK_RBC, _rbc_params(G, 10.0, a, _volume(v, t), 0.02 * G * a * a),
                                       pos))
        return d
    # vortex
    tau, a = 0.8, 8.0
    nu, k = (tau - 0.5) / 3, 2 * np.pi / nx
    G = nu * 0.03 * k * a / 0.1
    v, t = _sphere(case["level"])
    v = v * a
    cells = [(i, j, l) for i in range(nx // 24) for j in range(ny // 24) for l in range(nz // 24)]
    at = rng.choice(len(cells), case["caps"], replace=False)
    return dict(shape=(nx, ny, nz), periodic=(1, 1, 1), omega=1 / tau, lam=lam, tau=tau, mask=None, wall_u=None,
                g=np.zeros(3), u0=("vortex", 0.03, rng.uniform(0, 2 * np.pi, 3)), kernel=kernel, meshes=[(v, t)],
                particles=[(0, SKALAK_CAPSULE, [G, 10.0],
                            v + 24.0 * np.array(cells[i]) + 12 + rng.uniform(-3, 3, 3)) for i in at], guo=None)


def _velocity(d):
    """The starting velocity field (nx, ny, nz, 3), FP64 on the GPU."""
    nx, ny, nz = d["shape"]
    kind = d["u0"]
    u = torch.zeros(nx, ny, nz, 3, dtype=torch.float64, device="cuda")
    ax = [torch.arange(n, dtype=torch.float64, device="cuda") * (2 * math.pi / n) for n in d["shape"]]
    x, y, z = ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]
    if kind[0] == "vortex":
        px, py, pz = kind[2]
        u[..., 0] = kind[1] * torch.sin(x + px) * torch.cos(y + py) * torch.cos(z + pz)
        u[..., 1] = -kind[1] * torch.cos(x + px) * torch.sin(y + py) * torch.cos(z + pz)
        return u
    u += torch.from_numpy(kind[1]).cuda()
    if len(kind) > 2:  # a few percent of cross flow, zero at the walls
        p = kind[3]
        wall = torch.sin(torch.arange(ny, dtype=torch.float64, device="cuda") * (math.pi / (ny - 1)))[None, :, None]
        for a in range(3):
            u[..., a] += kind[2] * wall * torch.sin(2 * x + p[a]) * torch.cos(3 * z + p[3 + a])
    return u


# ------------------------------------------------------- prepare, run, checks
def _build(d, storage, u):
    """Lattice and immersed boundary of one description through the Python layer; u: page-locked field buffer."""
    from biblbm_amd.ibm import ImmersedBoundary
    from biblbm_amd.lattice import Lattice
    from biblbm_amd.walls import Boundary, GuoWall
    nx, ny, nz = d["shape"]
    w = d["omega"]
    # the inside's viscosity is lam times the outside's
    w_in = w if d["lam"] == 1 else 1 / (0.5 + d["lam"] * (d["tau"] - 0.5))
    L = Lattice(nx, ny, nz, periodic=d["periodic"], storage=storage, omega=w, omega_in=w_in)
    guo = None
    if d["wall_u"] is not None:
        L.set_velocity_walls(1, [-d["wall_u"], 0, 0], [d["wall_u"], 0, 0])
    if d["guo"] is not None:
        c, R = d["guo"]
        guo = GuoWall(L, Boundary.pipe(c, c, R, float(nx)))
        guo.insert()
    if d["mask"] is not None:
        L.set_mask(d["mask"])
    if d["g"].any():
        L.set_body_force(d["g"])
    u.copy_(_velocity(d))
    L.init_equilibrium(None, u.numpy())
    if d["wall_u"] is not None or guo is not None:
        L.initialize()
    ib = None
    if d["particles"]:
        ib = ImmersedBoundary(L, d["kernel"])
        ids = [ib.add_shape(v, t) for v, t in d["meshes"]]
        for mesh, model, params, pos in d["particles"]:
            ib.add_particle(ids[mesh], model, params, pos)
        ib.init()
    return L, ib, guo


def prepare(case, seed):
    d = _setup(case, seed)
    many = d if isinstance(d, list) else [d]
    cells = [int(np.prod(b["shape"])) for b in many]
    field = torch.empty(sum(cells), 3, dtype=torch.float64, pin_memory=True)
    views = [v.view(*b["shape"], 3) for v, b in zip(field.split(cells), many)]
    boxes = [_build(b, case["storage"], v) for b, v in zip(many, views)]
    ens = None
    if isinstance(d, list):
        from biblbm_amd.ensemble import Ensemble
        ens = Ensemble([(L, ib) for L, ib, _ in boxes])
    return dict(case=case, boxes=boxes, ens=ens, field=field if ens else views[0],
                ptrs=[v.data_ptr() for v in views])


def run(state):
    from biblbm_amd import capi
    case, boxes = state["case"], state["boxes"]
    n = case["steps"]
    L, ib, _ = boxes[0]
    if state["ens"] is not None:
        state["ens"].steps(n)
    elif ib is None:
        L.collide_and_stream(n)
    elif case["graph"]:
        ib.coupled_steps(n)
    else:
        for _ in range(n):
            ib.step()
            L.collide_and_stream(1)
    for (L, _, _), p in zip(boxes, state["ptrs"]):
        capi.call("bl_lattice_get_moments", L.handle, None, p)
    out = {"u": state["field"]}
    if ib is not None:
        out["pos"] = np.concatenate([b.positions() for _, b, _ in boxes])
        out["vel"] = np.concatenate([b.velocities() for _, b, _ in boxes])
    return out


def work(case):
    """Per step: each population read and written once, and for each vertex its stencil's velocities read and forces
    added once and its state and mesh; then the velocity field written once.  Flops: about 250 a cell, and a stencil's
    weights and sums and a membrane's forces a vertex."""
    s = {"f64": 8, "f32": 4, "f16s": 2}[case["storage"]]
    r = max(s, 4)
    d = _setup(case, 0)
    cells = verts = 0
    for b in d if isinstance(d, list) else [d]:
        cells += int(np.prod(b["shape"])) if b["mask"] is None else int(np.isin(b["mask"], (0, 3)).sum())
        verts += sum(len(p[3]) for p in b["particles"])
    support = {"roma": 27, "peskin": 64}.get(case.get("kernel"), 0)
    field = 3 * 8 * cells
    # velocities and forces of the nodes under the membranes: neighbouring stencils share nodes, one vertex has about
    # eight of its own
    per_vertex = 8 * 2 * 3 * r + 9 * r + 2 * 3 * 12 + 2 * 9 * r
    return {"bytes": case["steps"] * (2 * 19 * s * cells + verts * per_vertex) + field,
            "flops": case["steps"] * (250 * cells + verts * (support * 14 + 1500))}


def tolerance(case):
    # about four times the largest error against exact() that these ranges show; a step's rounding grows over the
    # steps, most where fine membranes are stiff
    return {"rel": {"f64": 4e-11, "f32": 2e-4, "f16s": 1e-3}[case["storage"]]}


# ------------------------------------------------- the same physics in FP64
_C = torch.tensor([(0, 0, 0)] + [(a, b, e) for a in (-1, 0, 1) for b in (-1, 0, 1) for e in (-1, 0, 1)
                                 if 0 < a * a + b * b + e * e < 3])
_W = [1 / 3 if not any(c) else (1 / 18 if sum(map(abs, c)) == 1 else 1 / 36) for c in _C.tolist()]
_OPP = [(_C == -c).all(1).nonzero().item() for c in _C]


class _Fluid:
    """D3Q19 lattice Boltzmann with Guo forcing; populations are f_i - w_i, a tensor (19, nx, ny, nz)."""

    def __init__(self, d):
        self.d, self.shape = d, d["shape"]
        self.mask = None if d["mask"] is None else torch.from_numpy(d["mask"]).cuda()
        self.g = torch.tensor(d["g"], device="cuda").view(3, 1, 1, 1)
        self.F = self.g.expand(3, *self.shape).clone()
        u = _velocity(d).permute(3, 0, 1, 2)
        self.f = torch.stack([self.equilibrium(i, torch.zeros_like(u[0]), u) for i in range(19)])
        self.phase = None
        self.guo = None if d["guo"] is None else self._guo_nodes()
        if d["wall_u"] is not None or d["guo"] is not None:
            self.F.zero_()  # the start's own boundary pass runs before any force is set
            self.F += self.g
            self.boundaries()

    @staticmethod
    def equilibrium(i, rb, j):
        c = _C[i].tolist()
        cj = sum(c[a] * j[a] for a in range(3) if c[a]) if any(c) else torch.zeros_like(rb)
        return _W[i] * (rb + 3 * cj + (4.5 * cj * cj - 1.5 * (j * j).sum(0)) / (1 + rb))

    @staticmethod
    def moments(f):
        c = _C.to(f)
        return f.sum(0), torch.stack([sum(f[i] * c[i, a].item() for i in range(19) if _C[i, a]) for a in range(3)])

    def velocity(self):
        rb, j = self.moments(self.f)
        u = j / (1 + rb) + self.F / 2
        if self.mask is not None:
            u = u * ((self.mask == 0) | (self.mask == 3))
        if self.d["wall_u"] is not None:
            for y, s in ((0, -1), (-1, 1)):
                u[:, :, y] = 0
                u[0, :, y] = s * self.d["wall_u"]
        return u

    def step(self):
        f, F, w = self.f, self.F, self.d["omega"]
        rb, j = self.moments(f)
        u = j / (1 + rb) + F / 2
        if self.phase is not None:
            wi = 1 / (0.5 + self.d["lam"] * (self.d["tau"] - 0.5))
            w = w * wi / (self.phase * w + (1 - self.phase) * wi)
        j = (1 + rb) * u
        uF = (u * F).sum(0)
        live = None if self.mask is None else (self.mask == 0) | (self.mask == 3)
        wall = None if self.mask is None else self.mask == 1
        new = torch.empty_like(f)
        for i in range(19):
            c = _C[i].tolist()
            cu = sum((c[a] * u[a] for a in range(3) if c[a]), torch.zeros_like(rb))
            cF = sum((c[a] * F[a] for a in range(3) if c[a]), torch.zeros_like(rb))
            g = (1 - w) * f[i] + w * self.equilibrium(i, rb, j) + (1 - w / 2) * _W[i] * (3 * (cF - uF) + 9 * cu * cF)
            if live is not None:
                g = torch.where(live, g, torch.where(wall, f[_OPP[i]], f[i]))
            new[i] = g
        for i in range(19):
            c = _C[i].tolist()
            g = torch.roll(new[i], c, (0, 1, 2))
            for a in range(3):  # what would come from beyond a closed face is what went out there
                if c[a] and not self.d["periodic"][a]:
                    at = [slice(None)] * 3
                    at[a] = 0 if c[a] > 0 else -1
                    g[tuple(at)] = new[_OPP[i]][tuple(at)]
            f[i] = g
        self.boundaries()

    def boundaries(self):
        f, F = self.f, self.F
        if self.d["wall_u"] is not None:  # regularised velocity walls, gradients by one-sided differences
            planes = []
            for y, s in ((0, -1), (-1, 1)):
                uw = torch.tensor([s * self.d["wall_u"], 0.0, 0.0], device="cuda", dtype=torch.float64).view(3, 1, 1)
                p, q = f[:, :, y], (1 if y == 0 else -2)
                on = sum(p[i] for i in range(19) if _C[i, 1] == 0)
                out = sum(p[i] for i in range(19) if _C[i, 1] == s)
                vn = s * (uw[1] - F[1, :, y] / 2)
                rb = (2 * out + on - vn) / (1 + vn)
                rb1, j1 = self.moments(f[:, :, q])
                du = -s * (j1 / (1 + rb1) + F[:, :, q] / 2 - uw)
                k = -(1 + rb) / 3 / self.d["omega"]
                pxy, pyy, pyz = du[0] * k, 2 * du[1] * k, du[2] * k
                j = (1 + rb) * uw
                rows = []
                for i in range(19):
                    c = _C[i].tolist()
                    neq = 4.5 * _W[i] * (2 * c[0] * c[1] * pxy + 2 * c[1] * c[2] * pyz + (c[1] * c[1] - 1 / 3) * pyy)
                    rows.append(self.equilibrium(i, rb, j) + neq)
                planes.append((y, torch.stack(rows)))
            for y, p in planes:
                f[:, :, y] = p
        if self.guo is not None:  # Guo's extrapolation onto the first cells outside the pipe
            yz, step, delta, live = self.guo
            f1 = f[:, :, yz[0] + step[0], yz[1] + step[1]]
            f2 = f[:, :, yz[0] + 2 * step[0], yz[1] + 2 * step[1]]
            (r1, j1), (r2, j2) = self.moments(f1), self.moments(f2)
            near = delta < 0.75
            jw = torch.where(near, (delta - 1) * j1 + (1 - delta) / (1 + delta) * (delta - 1) * j2,
                             (delta - 1) * j1 / delta)
            rows = []
            for i in range(19):
                n1 = f1[i] - self.equilibrium(i, r1, j1)
                n2 = f2[i] - self.equilibrium(i, r2, j2)
                rows.append(torch.where(near, delta * n1 + (1 - delta) * n2, n1) +
                            live * self.equilibrium(i, r1, jw))
            f[:, :, yz[0], yz[1]] = torch.stack(rows)

    def _guo_nodes(self):
        """Cells outside the circle with a lattice link across it: the link most opposed to the normal there, and the
        share of it outside.  The pipe is the same at every x, and a link with an x part is never the most opposed."""
        c0, R = self.d["guo"]
        n = self.shape[1]
        best, link, delta = np.full((n, n), 2.0), np.zeros((n, n, 2), np.int64), np.zeros((n, n))
        y, z = np.meshgrid(np.arange(n) - c0, np.arange(n) - c0, indexing="ij")
        for dy, dz in [(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1) if a or b]:
            a, b, c = dy * dy + dz * dz, y * dy + z * dz, y * y + z * z - R * R
            with np.errstate(invalid="ignore"):
                t = (-b - np.sqrt(b * b - a * c)) / a
                t2 = (-b + np.sqrt(b * b - a * c)) / a
            t = np.where((t >= 0) & (t <= 1), t, t2)
            ok = (t >= 0) & (t <= 1) & (c >= 0)
            wy, wz = y + dy / math.sqrt(a) * t, z + dz / math.sqrt(a) * t
            cos = (wy * dy + wz * dz) / math.sqrt(a) / np.sqrt(wy * wy + wz * wz)
            ok &= cos < best
            best[ok], delta[ok] = cos[ok], 1 - t[ok]
            link[ok] = (dy, dz)
        at = np.nonzero(best < 2)
        live = torch.from_numpy((self.d["mask"][0][at] == 0).astype(float)).cuda()
        return ([torch.from_numpy(a).cuda() for a in at],
                [torch.from_numpy(link[at][:, k].copy()).cuda() for k in (0, 1)],
                torch.from_numpy(delta[at]).cuda(), live)


class _Cells:
    """The membranes: Skalak triangles, and for red cells area, volume and bending terms."""

    def __init__(self, d):
        self.d = d
        pos, tri, rest, par, hinge, owner, off = [], [], [], [], [], [], 0
        for mesh, model, params, p in d["particles"]:
            v, t = d["meshes"][mesh]
            k = len(owner)
            pos.append(p)
            tri.append(t.astype(np.int64) + off)
            rest.append(v)
            owner.append(len(t))
            par.append(list(params) + [0.0] * (7 - len(params)) if model == SKALAK_RBC
                       else list(params) + [0, 0, 0, 1.0, 0])
            e = np.concatenate([np.concatenate([t[:, [a, b]], t[:, [c]], np.full((len(t), 1), k)], 1)
                                for a, b, c in ((0, 1, 2), (1, 2, 0), (2, 0, 1))]).astype(np.int64)
            up, down = e[e[:, 0] < e[:, 1]], e[e[:, 0] > e[:, 1]]
            up = up[np.lexsort((up[:, 1], up[:, 0]))]
            down = down[np.lexsort((down[:, 0], down[:, 1]))]
            if model == SKALAK_RBC:
                hinge.append(np.stack([up[:, 1] + off, up[:, 2] + off, up[:, 0] + off, down[:, 2] + off, up[:, 3]], 1))
            off += len(v)
        cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        self.pos, self.tri, self.rest = cu(np.concatenate(pos)), cu(np.concatenate(tri)), cu(np.concatenate(rest))
        self.owner = cu(np.repeat(np.arange(len(owner)), owner))
        self.vowner = cu(np.repeat(np.arange(len(pos)), [len(p) for p in pos]))
        self.par = cu(np.array(par, float))
        self.hinge = cu(np.concatenate(hinge)) if hinge else None
        self.vel = torch.zeros_like(self.pos)
        self.count = len(owner)
        with torch.no_grad():
            self.A0 = self._areas(self.rest)
            self.A0t = self._sum(self.A0)
            if self.hinge is not None:
                self.cs0 = self._angles(self.rest)

    def _sum(self, x):
        return torch.zeros(self.count, *x.shape[1:], dtype=x.dtype, device=x.device).index_add(0, self.owner, x)

    def _areas(self, p):
        a, b, c = (p[self.tri[:, k]] for k in range(3))
        return 0.5 * torch.linalg.cross(b - a, c - a).norm(dim=1)

    def _angles(self, p):
        v0, v1, v2, v3 = (p[self.hinge[:, k]] for k in range(4))
        e = v2 - v0
        n1, n2 = torch.linalg.cross(v1 - v0, e), torch.linalg.cross(e, v3 - v0)
        n1, n2, e = (n / n.norm(dim=1, keepdim=True) for n in (n1, n2, e))
        return (n1 * n2).sum(1), -(torch.linalg.cross(n1, n2) * e).sum(1)

    def forces(self):
        """Minus the gradient of the membrane energy; the coefficients the library's law takes as they stand are
        detached (its strain c is the ratio of the sines alone, the reference's own form)."""
        p = self.pos.detach().requires_grad_(True)
        G, C, kag, kal, kv, v_des, kb = (self.par[self.owner, k] for k in range(7))
        t = self.tri
        e0, e1 = p[t[:, 1]] - p[t[:, 0]], p[t[:, 2]] - p[t[:, 0]]
        r0, r1 = self.rest[t[:, 1]] - self.rest[t[:, 0]], self.rest[t[:, 2]] - self.rest[t[:, 0]]
        l0, l1 = r0.norm(dim=1), r1.norm(dim=1)
        c0 = (r0 * r1).sum(1) / (l0 * l1)
        s0 = torch.linalg.cross(r0, r1).norm(dim=1) / (l0 * l1)
        q00, q11, q01 = (e0 * e0).sum(1) / l0 ** 2, (e1 * e1).sum(1) / l1 ** 2, (e0 * e1).sum(1) / (l0 * l1)
        D11 = (q00 - 1) / 2
        D22 = ((q11 + q00 * c0 ** 2 - 2 * q01 * c0) / s0 ** 2 - 1) / 2
        D12 = (q01 - q00 * c0) / (2 * s0)
        with torch.no_grad():
            sin = torch.linalg.cross(e0, e1).norm(dim=1) / (e0.norm(dim=1) * e1.norm(dim=1))
            b = 2 * D12 / q00.sqrt()
            H22 = (b * b + (sin / s0) ** 2 - 1) / 2
            I1 = 2 * (D11 + H22)
            I2 = I1 + 4 * (D11 * H22 - D12 * D12)
            k11 = 2 * (I1 + 1) + (C * I2 - 1) * (2 + 4 * H22)
            k22 = 2 * (I1 + 1) + (C * I2 - 1) * (2 + 4 * D11)
            k12 = -8 * D12 * (C * I2 - 1) * l0 / l1  # the law's own factor: its shear gradient is over the other edge
        E = (G / 2 * self.A0 * (k11 * D11 + k22 * D22 + k12 * D12)).sum()
        if self.hinge is not None:
            A = self._areas(p)
            V = (p[t[:, 0]] * torch.linalg.cross(p[t[:, 1]], p[t[:, 2]])).sum(1) / 6
            with torch.no_grad():
                dA = kag * ((self.A0t - self._sum(A)) / self.A0t)[self.owner] + kal * (self.A0 - A) / self.A0
                dV = kv * (v_des - self._sum(V)[self.owner]) / v_des
            cs, sn = self._angles(p)
            E = E - (dA * A).sum() - (dV * V).sum()
            E = E - (self.par[self.hinge[:, 4], 6] * (cs * self.cs0[0] + sn * self.cs0[1])).sum()
        return -torch.autograd.grad(E, p)[0]

    def stencil(self, shape):
        """Flat node indices (n, S^3) of every vertex's support and its weights."""
        S, half = {"roma": (3, 1.5), "peskin": (4, 2.0)}[self.d["kernel"]]
        idx, wts = [], []
        for a in range(3):
            x = self.pos[:, a, None]
            k = torch.ceil(x - half) + torch.arange(S, device="cuda")
            r = (k - x).abs()
            if S == 3:
                w = torch.where(r > 0.5, (5 - 3 * r - (1 - 3 * (1 - r) ** 2).clamp(min=0).sqrt()) / 6,
                                (1 + (1 - 3 * r * r).clamp(min=0).sqrt()) / 3)
            else:
                w = torch.where(r <= 1, (3 - 2 * r + (1 + 4 * r - 4 * r * r).clamp(min=0).sqrt()) / 8,
                                (5 - 2 * r - (12 * r - 7 - 4 * r * r).clamp(min=0).sqrt()) / 8)
            k = k.long()
            if self.d["periodic"][a]:
                k = k % shape[a]
            else:
                w = w * ((k >= 0) & (k < shape[a]))
                k = k.clamp(0, shape[a] - 1)
            idx.append(k)
            wts.append(w)
        n = len(self.pos)
        i = (idx[0][:, :, None, None] * shape[1] + idx[1][:, None, :, None]) * shape[2] + idx[2][:, None, None, :]
        w = wts[0][:, :, None, None] * wts[1][:, None, :, None] * wts[2][:, None, None, :]
        return i.reshape(n, -1), w.reshape(n, -1)

    def couple(self, fluid):
        """Velocities at the vertices, forces onto the nodes, then the vertices move."""
        u = fluid.velocity().reshape(3, -1)
        i, w = self.stencil(fluid.shape)
        F = self.forces()
        fluid.F = fluid.g.expand(3, *fluid.shape).clone()
        for a in range(3):
            self.vel[:, a] = (u[a][i] * w).sum(1)
            fluid.F[a].view(-1).index_add_(0, i.reshape(-1), (w * F[:, a, None]).reshape(-1))
        self.pos += self.vel
        p, t = self.pos, self.tri
        A = self._areas(p)
        com = self._sum((p[t[:, 0]] + p[t[:, 1]] + p[t[:, 2]]) / 3 * A[:, None]) / self._sum(A)[:, None]
        for a in range(3):  # a centre of mass that left the periodic box re-enters it
            if self.d["periodic"][a]:
                n = fluid.shape[a]
                p[:, a] += (-n * torch.floor((com[:, a] + 0.5) / n))[self.vowner]
        if self.d["lam"] != 1:
            fluid.phase = self.inside(fluid.shape)

    def inside(self, shape):
        """1 on the nodes inside a membrane: the parity of the surface crossings below them along z."""
        t, p = self.tri, self.pos
        a, e, h = p[t[:, 0]], p[t[:, 1]] - p[t[:, 0]], p[t[:, 2]] - p[t[:, 0]]
        lo = torch.ceil(torch.minimum(a, torch.minimum(p[t[:, 1]], p[t[:, 2]])))
        hi = torch.floor(torch.maximum(a, torch.maximum(p[t[:, 1]], p[t[:, 2]])))
        m = int((hi - lo)[:, :2].max().item()) + 1
        cross = torch.zeros(*shape, dtype=torch.int64, device="cuda")
        det = e[:, 0] * h[:, 1] - e[:, 1] * h[:, 0]
        for i in range(max(m, 0)):
            for j in range(max(m, 0)):
                x, y = lo[:, 0] + i, lo[:, 1] + j
                dx, dy = x - a[:, 0], y - a[:, 1]
                s, r = (dx * h[:, 1] - dy * h[:, 0]) / det, (e[:, 0] * dy - e[:, 1] * dx) / det
                ok = (x <= hi[:, 0]) & (y <= hi[:, 1]) & (s >= 0) & (r >= 0) & (s + r <= 1) & (det.abs() > 2e-16)
                z = a[:, 2] + s * e[:, 2] + r * h[:, 2]
                k = [x.long(), y.long(), None]
                for b in (0, 1):
                    if self.d["periodic"][b]:
                        k[b] = k[b] % shape[b]
                    else:
                        ok &= (k[b] >= 0) & (k[b] < shape[b])
                if self.d["periodic"][2]:
                    z = z - shape[2] * torch.floor((z + 0.5) / shape[2])
                z = torch.ceil(z).clamp(min=0)
                ok &= z < shape[2]
                cross.index_put_((k[0][ok], k[1][ok], z[ok].long()), torch.ones_like(k[0][ok]), accumulate=True)
        return (cross.cumsum(2) % 2).double()


def exact(case, seed):
    d = _setup(case, seed)
    many = d if isinstance(d, list) else [d]
    cells = sum(int(np.prod(b["shape"])) for b in many)
    if cells * case["steps"] > 1.5e9:
        return None  # over about twenty seconds
    field, pos, vel = [], [], []
    for b in many:
        fluid = _Fluid(b)
        membranes = _Cells(b) if b["particles"] else None
        for _ in range(case["steps"]):
            if membranes is not None:
                membranes.couple(fluid)
            fluid.step()
        u = fluid.velocity().permute(1, 2, 3, 0).contiguous()
        field.append(u.reshape(-1, 3) if len(many) > 1 or isinstance(d, list) else u)
        if membranes is not None:
            pos.append(membranes.pos)
            vel.append(membranes.vel)
    out = {"u": torch.cat(field) if isinstance(d, list) else field[0]}
    if pos:
        out["pos"], out["vel"] = torch.cat(pos), torch.cat(vel)
    return out
