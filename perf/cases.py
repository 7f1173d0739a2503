"""The engine's work as its users run it, for timing: stretches of time steps
of the four kinds of model (with the fields that an output interval reads at
the end), and training and inference of the closure network.

A step case advances the model by `steps` steps through the captured step,
as the integration header's time loop does between two outputs, and then
reads the node fields.  The simulation goes on from pass to pass.  Engines
run at their default launch shape.  Fields of a mixed-precision model, whose
bond arithmetic is FP32, are kept as float32; fields of an FP64 model as
float64.
"""
from __future__ import annotations

import copy
import math

import numpy as np
import torch

from peridem_amd import capi, closure, configs

MM = 1.0e-3


def listed():
    return [
        # the two-particle collision, the smallest model there is: a step is a chain of launches
        dict(name="two_particle_fp64", model="two", nodes=367, steps=500),
        # a small bed of circles and hexagons, odd sizes, velocity Verlet
        dict(name="bed_37_verlet_fp64", model="bed", particles=37, nodes=151, steps=400, verlet=True),
        # the compressive test's size: 500 particles of about 400 nodes in contact, a wall pressing on them
        dict(name="bed_500_fp64", model="bed", particles=500, nodes=400, steps=1000, verlet=False),
        # a small state-based packing in the FP64 parity mode
        dict(name="packing_60_fp64", model="packing", particles=60, nodes=1000, steps=200, mixed=False, verlet=False),
        # a small state-based packing in mixed precision, particles of uneven size
        dict(name="packing_27_mixed", model="packing", particles=27, nodes=333, steps=500, mixed=True, verlet=False),
        # the 3D packing of the benchmark: 2000 spheres, 2.08M nodes
        dict(name="packing_2000_mixed", model="packing", particles=2000, nodes=1000, steps=300, mixed=True,
             verlet=False),
        # a few collisions batched in one model, plain and with the learned contact closure
        dict(name="ensemble_16_mixed", model="ensemble", instances=16, steps=500, closure=False),
        dict(name="ensemble_48_closure", model="ensemble", instances=48, steps=500, closure=True),
        # the batched ensemble of the benchmark: 512 independent collisions, 4.2M nodes
        dict(name="ensemble_512_mixed", model="ensemble", instances=512, steps=300, closure=False),
        # the closure network: minibatch training on logged pair rows, at the benchmark's batch
        dict(name="mlp_train_1024", model="mlp_train", rows=20000, batch=1024, iters=200),
        # the closure network: inference on one pair's worth of rows, and on a logged set
        dict(name="mlp_forward_17", model="mlp_forward", rows=17),
        dict(name="mlp_forward_100000", model="mlp_forward", rows=100000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["two", "bed", "packing", "packing", "ensemble", "mlp_train", "mlp_forward"])
    if kind == "two":
        return dict(model="two", nodes=_log(rng, 60, 2000), steps=_log(rng, 100, 700))
    if kind == "bed":
        return dict(model="bed", particles=_log(rng, 9, 500), nodes=_log(rng, 40, 500), steps=_log(rng, 200, 700),
                    verlet=rng.random() < 0.3)
    if kind == "packing":
        mixed = rng.random() < 0.6
        return dict(model="packing", particles=_log(rng, 6, 1500 if mixed else 100), nodes=_log(rng, 100, 1000),
                    steps=_log(rng, 100, 400), mixed=mixed, verlet=rng.random() < 0.3)
    if kind == "ensemble":
        return dict(model="ensemble", instances=_log(rng, 3, 400), steps=_log(rng, 100, 300),
                    closure=rng.random() < 0.25)
    if kind == "mlp_train":
        return dict(model="mlp_train", rows=_log(rng, 500, 100000), batch=_log(rng, 64, 4096), iters=_log(rng, 50, 300))
    return dict(model="mlp_forward", rows=_log(rng, 1, 200000))


# ------------------------------------------------------------------ models

_specs = {}


def _geometry(c):
    """The deck's model of a case: meshes, particles, walls, contact table
    (the same for every seed, kept while the case is measured)."""
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "steps", "verlet")))
    if key not in _specs:
        if len(_specs) >= 2:
            _specs.clear()
        if c["model"] == "two":
            # disks of about `nodes` nodes each, a gap just inside contact distance
            h = MM * math.sqrt(math.pi / (c["nodes"] * math.sqrt(3.0) / 2.0))
            s = configs.two_particle(R=MM, h=h, gap=0.94 * h)
        elif c["model"] == "bed":
            # neighbours touch from the start: gaps below the contact radius
            s = configs.compressive_2d(n_particles=c["particles"], nodes_per_particle=c["nodes"], R_lo=1.0 * MM,
                                       R_hi=1.02 * MM, pitch_factor=1.01, seed=1)
        elif c["model"] == "packing":
            n = c["particles"]
            s = configs.packing_3d(n_spheres=n, nodes_per_sphere=c["nodes"], seed=1,
                                   L=30.0 * MM if n > 800 else 1.25 * MM * (16.0 * n) ** (1.0 / 3.0))
        else:
            s = configs.ensemble_2d(n_instances=c["instances"], seed=1)
        _specs[key] = s
    return _specs[key]


#: largest speed of a particle at the start [m/s]
SPEED = {"two": 0.1, "bed": 0.1, "packing": 0.5, "ensemble": 1.0}
#: peak strain of the particles at the start
STRAIN = {"two": 1e-4, "bed": 1e-4, "packing": 1e-3, "ensemble": 1e-3}


def _model(c, seed):
    """The model with the seed's state: every particle moves as a rigid body
    at its own velocity and carries a smooth displacement."""
    g = _geometry(c)
    rng = np.random.default_rng(seed)
    s = copy.copy(g)
    d = s.dim
    free = np.array([p["type_index"] == 0 for p in s.particles])
    n_p = len(s.particles)
    vp = rng.normal(size=(n_p, 3))
    vp[:, d:] = 0.0
    if c["model"] == "two":  # toward each other
        vp[:] = 0.0
        vp[0, 1], vp[1, 1] = 0.5, -1.0
    vp *= (SPEED[c["model"]] * rng.uniform(0.05, 1.0, n_p) / np.linalg.norm(vp, axis=1))[:, None] * free[:, None]
    s.v = vp[s.pt_id]
    length = 0.5 * MM  # of the waves, over 2 pi
    phase = rng.uniform(0.0, 2.0 * math.pi, (n_p, 3))
    amp = STRAIN[c["model"]] * length * free
    s.u = np.zeros_like(s.x_ref)
    for k in range(d):
        s.u[:, k] = amp[s.pt_id] * np.sin(s.x_ref[:, (k + 1) % d] / length + phase[s.pt_id, k])
    return s


def _rows(c, seed):
    """Normalised pair features and targets of a smooth law of them."""
    r = np.random.default_rng(seed)
    x = r.normal(size=(c["rows"], capi.Mlp.NIN)).astype(np.float32)
    w = r.normal(size=(capi.Mlp.NIN, capi.Mlp.NOUT)).astype(np.float32) / 4.0
    t = np.tanh(x @ w) + 0.1 * (x @ w) ** 2
    return x, t.astype(np.float32)


def _net(seed):
    """An untrained network with an output layer of the size that training ends with."""
    net = capi.Mlp(seed=seed % 65521)
    p = net.params()
    p[-(128 * 4 + 4):] *= 10.0
    net.set_params(p)
    return net


def prepare(case, seed):
    c = dict(case)
    if c["model"].startswith("mlp"):
        x, t = _rows(c, seed)
        net = _net(seed)
        net.set_normalization(np.zeros(16), np.ones(16), np.ones(4), (1.0, 1.0, 1.0, 0.1))
        return dict(case=c, net=net, x=x, t=t, seed=int(seed))
    s = _model(c, seed)
    mixed = c.get("mixed", c["model"] == "ensemble")
    eng = capi.GpuEngine(s, capi.PREC_MIXED if mixed else capi.PREC_FP64)
    net = None
    if c.get("closure"):
        # corrections of some hundredths of the contact force's unit
        net = _net(seed)
        net.set_normalization(np.zeros(16), np.ones(16), np.full(4, 50.0), (1.0, 1.0, 1.0, 0.1))
        eng.closure_setup(closure.particle_codes(s))
        eng.closure_enable(net, pen_max_h=0.05, dz_max=0.5, check_every=100)
    eng.integrate_begin()
    return dict(case=c, eng=eng, mixed=mixed, net=net)


def run(state):
    c = state["case"]
    if c["model"] == "mlp_forward":
        return state["net"].forward(state["x"])
    if c["model"] == "mlp_train":
        loss = state["net"].train(state["x"], state["t"], iters=c["iters"], batch=c["batch"], lr=1e-3,
                                  seed=state["seed"] % 1000003)
        return dict(loss=loss, params=state["net"].params())
    eng = state["eng"]
    if c.get("verlet"):
        eng.integrate_verlet_graph(c["steps"])
    else:
        eng.integrate_cd_graph(c["steps"])
    out = {n: eng.field(f) for n, f in (("u", capi.FIELD_U), ("v", capi.FIELD_V), ("f", capi.FIELD_F),
                                        ("Z", capi.FIELD_Z))}
    if state["mixed"]:
        out = {n: a.astype(np.float32) for n, a in out.items()}
    return out


# ------------------------------------------------------- what a pass needs

def _mesh_bonds(x, horizon):
    """Nodes and directed bonds of one particle's mesh."""
    t = torch.from_numpy(np.ascontiguousarray(x))
    near = sum(int((((a[:, None, :] - t[None, :, :]) ** 2).sum(-1) < horizon ** 2).sum()) for a in t.split(512))
    return len(x), near - len(x)


def work(case):
    """Bytes that a step cannot do without, times the steps, and the read of
    the fields: per force-computing node the bond passes' 24 d + 20 + 4.25 N
    bytes (N bonds: 4-byte ids, a bit each; FP64 state; theta on chip) and the
    node update's 56 d + 13.  Operations: about 45 per bond (a dilation and a
    force term, or the RNP law from one end), 12 d per node."""
    c = dict(case)
    if c["model"].startswith("mlp"):
        n, mac = c["rows"], 16 * 128 + 2 * 128 * 128 + 128 * 4
        params = mac + 3 * 128 + 4
        if c["model"] == "mlp_forward":
            return {"bytes": n * 80.0 + 4 * params, "flops": 2.0 * mac * n}
        # parameters and both Adam moments read and written, in each iteration
        return {"bytes": n * 80.0 + c["iters"] * (24.0 * params + 80 * c["batch"]),
                "flops": 6.0 * mac * c["batch"] * c["iters"]}
    g = _geometry(c)
    d = g.dim
    meshes, nodes, bonds = {}, 0, 0
    for p in g.particles:
        if not p["compute_force"]:
            continue
        lo, hi = p["glob_start"], p["glob_end"]
        key = (hi - lo, p["zone"])
        if key not in meshes:
            meshes[key] = _mesh_bonds(g.x_ref[lo:hi], p["horizon"])
        nodes += meshes[key][0]
        bonds += meshes[key][1]
    step = nodes * (24.0 * d + 20 + 56 * d + 13) + 4.25 * bonds
    return {"bytes": c["steps"] * step + g.n_nodes * (24.0 * d + 4),
            "flops": c["steps"] * (45.0 * bonds + 12.0 * d * nodes)}


# ------------------------------------------------------------ 64-bit values

def exact(case, seed):
    """What run() returns in 64 bits: the network's outputs, and the steps of
    a 3D packing whose particles are out of each other's contact reach (bond
    forces, gravity, centre damping, the wall's motion).  None for the others:
    beds, ensembles and small packings have node contacts, and the trained
    weights follow the rounding of every step."""
    c = dict(case)
    if c["model"] == "mlp_forward":
        st = prepare(c, seed)
        return _forward64(st["net"].params().astype(np.float64), st["x"].astype(np.float64)).numpy()
    if c["model"] == "packing" and c["particles"] > 800 and not c["verlet"]:
        return _packing64(c, seed)
    return None


def _forward64(p, x):
    p, h, at = torch.from_numpy(p), torch.from_numpy(x), 0
    for k, (a, b) in enumerate(((16, 128), (128, 128), (128, 128), (128, 4))):
        w = p[at:at + a * b].reshape(a, b)
        at += a * b
        h = h @ w + p[at:at + b]
        at += b
        if k < 3:
            h = torch.relu(h)
    return h


def _packing64(c, seed):
    """The packing's steps in FP64 torch on the GPU; None where a node contact
    or a breaking bond comes into reach (they are not worked out here)."""
    s = _model(c, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def up(a, dtype=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=dev)

    parts = s.particles
    n_p = len(parts)
    pid = up(s.pt_id, torch.int64)
    per = {k: up([float(p[k]) for p in parts]) for k in ("horizon", "mesh_size", "density", "bounding_radius")}
    mat = up([p["mat"] for p in parts])
    on = up([p["compute_force"] for p in parts], torch.bool)
    wall = up([p["type_index"] for p in parts], torch.bool)
    xr, vol = up(s.x_ref), up(s.vol)
    p0, p1 = s.influence_fn_params
    rc = s.max_contact_r
    gravity = up(s.gravity)[None, :]
    # bonds and their reference data, particle by particle, node lists padded to the
    # longest (with the node itself at weight 0); sums run over chunks of whole particles
    m = torch.zeros_like(vol)
    bonds, part, size = [], [], 0
    for k, p in enumerate(parts):
        lo, hi = p["glob_start"], p["glob_end"]
        if p["compute_force"]:
            x = xr[lo:hi]
            ij = []
            for a in range(0, hi - lo, 2048):
                hit = (((x[a:a + 2048, None, :] - x[None, :, :]) ** 2).sum(-1) < p["horizon"] ** 2).nonzero()
                hit[:, 0] += a
                ij.append(hit[hit[:, 0] != hit[:, 1]])
            part.append((lo, hi, torch.cat(ij) + lo))
            size += len(part[-1][2])
        if part and (size > 8_000_000 or k == n_p - 1):
            first, last = part[0][0], part[-1][1]
            ij = torch.cat([t for _, _, t in part])
            i = ij[:, 0] - first
            deg = torch.bincount(i, minlength=last - first)
            place = torch.arange(len(ij), device=dev) - (torch.cumsum(deg, 0) - deg)[i]
            j = torch.arange(first, last, device=dev)[:, None].repeat(1, int(deg.max()))
            j[i, place] = ij[:, 1]
            own = slice(first, last)
            dx = xr[j] - xr[own, None, :]
            r = dx.norm(dim=2)
            de, h = per["horizon"][pid[own], None], per["mesh_size"][pid[own], None]
            low = de - 0.5 * h
            vc = torch.where((r - low) > 1e-5 * torch.maximum(r, low), vol[j] * (de + 0.5 * h - r) / h, vol[j])
            jv = torch.where(r > 0, (p0 + p1 * r / de) * vc, torch.zeros_like(r))
            m[own] = (r * r * jv).sum(1)
            bonds.append((own, j, dx, torch.where(r > 0, r, torch.ones_like(r)), jv))
            part, size = [], 0
    m = torch.where(m > 0, m, torch.ones_like(m))
    kk, gg, s0 = mat[pid, 0], mat[pid, 1], float(mat[:, 2].min())
    alpha = 15.0 * gg / m
    beta = 3.0 * kk / m - alpha / 3.0
    # damping of the particles' centres
    body = (~wall).nonzero()[:, 0]
    centre = up([p["center_node"] for p in parts], torch.int64)[body]
    rad, rho = per["bounding_radius"][body], per["density"][body]
    ct = s.contact[0][0]
    area = math.pi * rad * rad
    mass = rho * area
    meq = 2.0 * mass[:, None] * mass[None, :] / (mass[:, None] + mass[None, :])
    bn = ct["betan"] * torch.sqrt(ct["kappa"] * ct["contact_r"] * meq)
    reach = rad[:, None] + rad[None, :] + 1.01 * ct["contact_r"]

    def forces(u, v):
        th = torch.zeros_like(vol)
        far = torch.zeros((), dtype=u.dtype, device=dev)
        for own, j, dx, r, jv in bonds:
            du = u[j] - u[own, None, :]
            t2 = (du * (2.0 * dx + du)).sum(2)
            cl = t2 / (torch.sqrt(r * r + t2) + r)
            far = torch.maximum(far, (cl.abs() / r).max())
            th[own] = (r * cl * jv).sum(1)
        b = (3.0 * th / m) * beta
        f = torch.zeros_like(u)
        for own, j, dx, r, jv in bonds:
            y = dx + (u[j] - u[own, None, :])
            ly = y.norm(dim=2)
            ly = torch.where(ly > 0, ly, torch.ones_like(ly))
            cl = ((y - dx) * (y + dx)).sum(2) / (ly + r)
            sf = jv * (r * (b[own, None] + b[j]) + cl * (alpha[own, None] + alpha[j])) / ly
            f[own] = (sf[:, :, None] * y).sum(1)
        xc = (xr + u)[centre]
        dc = xc[None, :, :] - xc[:, None, :]
        dist = dc.norm(dim=2)
        near = (dist < reach * (1.0 - 1e-5))
        near.fill_diagonal_(False)
        hat = dc / torch.where(dist > 0, dist, torch.ones_like(dist))[:, :, None]
        vn = ((v[centre][None, :, :] - v[centre][:, None, :]) * hat).sum(2).clamp(max=0.0)
        fd = torch.zeros((n_p, 3), dtype=u.dtype, device=dev)
        fd[body] = (torch.where(near, bn * vn, torch.zeros_like(bn))[:, :, None] * hat).sum(1) / area[:, None]
        return f + fd[pid] + per["density"][pid][:, None] * gravity, far

    # no two nodes of different particles may come within contact distance: particles keep
    # their shape to far less than a mesh size, so the rigid motion bounds the approach
    u, v = up(s.u), up(s.v)
    clear = rc * 1.01 + 2.4 * c["steps"] * s.dt * SPEED["packing"]
    x = xr + u
    xc = x[centre]
    close = ((xc[None, :, :] - xc[:, None, :]).norm(dim=2) - rad[:, None] - rad[None, :] < clear).triu(1).nonzero()
    ends = [(parts[int(k)]["glob_start"], parts[int(k)]["glob_end"]) for k in body]
    for a, b in close.tolist():
        if float((x[ends[a][0]:ends[a][1], None, :] - x[None, ends[b][0]:ends[b][1], :]).norm(dim=2).min()) < clear:
            return None
    inside = x[~wall[pid], 2]
    if float((inside.min() - x[wall[pid], 2][:, None]).abs().min()) < clear or \
            float((inside.max() - x[wall[pid], 2][:, None]).abs().min()) < clear:
        return None
    top = up([k == s.wall_id for k in range(n_p)], torch.bool)[pid]
    dof = up(s.fix[:, None] >> np.arange(3)[None, :] & 1, torch.bool)
    move = (on[pid][:, None] & ~dof).to(u.dtype)
    speed = [b for b in s.ubc if not b["is_zero"]][0]["amp"][0]
    t = 0.0
    f, far = forces(u, v)
    for _ in range(c["steps"]):
        v = v + move * (s.dt / per["density"][pid])[:, None] * f
        u = u + move * s.dt * v
        t += s.dt
        u[:, 2] = torch.where(top, speed * t, u[:, 2])
        v[:, 2] = torch.where(top, speed, v[:, 2])
        f, more = forces(u, v)
        far = torch.maximum(far, more)
    return None if float(far) > 0.99 * s0 else dict(u=u.cpu().numpy(), v=v.cpu().numpy(), f=f.cpu().numpy(), Z=None)
