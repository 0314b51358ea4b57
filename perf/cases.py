"""Workloads that stand for the framework's use, each one pass of a user's
program through the package's public entry points (xpbdfem.Scene).

listed() are the named cases, draw(rng) gives further ones of the same
ranges, prepare(case, seed) builds what a program holds before the call (the
scenes), run(state) is one pass, work(case) the bytes and operations of a
pass that no implementation can do without, and exact(case, seed) the result
in FP64 from plain torch where the case has one that does not depend on a
schedule of the library's own.

Sizes: the 12x4x4, 16x4x4 and 96x24x24 beams, the random boxes of 3 to 24
cells a side and the fitting beams of 4 to 16 cells a side are the
workloads of workloads.py and bench.py; the others lie between them.
"""
import math
import os
import sys

import numpy as np
import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
_PKG = os.path.join(os.path.dirname(_HERE), "xpbd-fem_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import xpbdfem as xf  # noqa: E402  (after torch, whose HIP runtime the library then shares)

_CTX = None

# The Yeoh constants of the benchmark beam in the skin normalisation
# (C10 = 5e4, C20 = 5e3, C30 = 5e2 Pa).
_YEOH = (0.1095, 0.01095, 0.001095)


def _context():
    global _CTX
    if _CTX is None:
        _CTX = xf.Context(0)
    return _CTX


# ------------------------------------------------------------------- meshes

# The six tets of a cell: paths of unit steps from corner 000 to corner 111,
# positively oriented (corner index x + 2 y + 4 z).
_PATHS = ((0, 1, 2), (1, 2, 0), (2, 0, 1), (1, 0, 2), (0, 2, 1), (2, 1, 0))


def _block(W, H, D, h, mirrored=False):
    """(positions [n, 3] float64, tets [t, 4], cell sum and split of each tet)
    of a W x H x D block of cells of edge h, x from 0, centred in y and z.
    mirrored: the cells' diagonals alternate along every axis."""
    zz, yy, xx = np.meshgrid(np.arange(D + 1), np.arange(H + 1), np.arange(W + 1), indexing="ij")
    pos = np.stack([xx.ravel() * h, (yy.ravel() - 0.5 * H) * h, (zz.ravel() - 0.5 * D) * h], axis=1)
    cz, cy, cx = (a.ravel() for a in np.meshgrid(np.arange(D), np.arange(H), np.arange(W), indexing="ij"))
    cell = np.stack([cx, cy, cz], axis=1)
    flip = (cell & 1) if mirrored else np.zeros_like(cell)
    odd = flip.sum(axis=1) & 1
    stride = np.array([1, W + 1, (W + 1) * (H + 1)])
    tets = np.zeros((len(cell), 6, 4), np.int64)
    for s, path in enumerate(_PATHS):
        corner = np.zeros(3, np.int64)
        nodes = []
        for step in (None,) + path:
            if step is not None:
                corner[step] = 1
            nodes.append((cell + (corner ^ flip)) @ stride)
        even = s < 3  # even axis permutations give positive volume in this node order
        n = [nodes[1], nodes[2], nodes[3], nodes[0]]
        swap = odd == (1 if even else 0)
        tets[:, s, 0] = np.where(swap, n[1], n[0])
        tets[:, s, 1] = np.where(swap, n[0], n[1])
        tets[:, s, 2] = n[2]
        tets[:, s, 3] = n[3]
    split = np.tile(np.arange(6), len(cell))
    return pos, tets.reshape(-1, 4), np.repeat(cell.sum(axis=1), 6), split


def _volumes(pos, tets):
    d = pos[tets[:, :3]] - pos[tets[:, 3:]]
    return np.einsum("ij,ij->i", d[:, 0], np.cross(d[:, 1], d[:, 2])) / 6.0


def _sizes(case):
    """Cell counts of the case's bodies: (W, H, D) once, or `bodies` boxes
    with counts per axis uniform in [lo, hi], fixed by the case's mesh number."""
    if case.get("bodies", 1) == 1:
        return [(case["W"], case["H"], case["D"])]
    r = np.random.RandomState(case["mesh"])
    return [tuple(int(v) for v in r.randint(case["lo"], case["hi"] + 1, 3)) for _ in range(case["bodies"])]


def _inputs(case, seed):
    """The bodies of a case as plain arrays."""
    r = np.random.RandomState(seed % (1 << 32))
    fit = case["kind"] == "adjoint"
    h = 0.08 if fit and case.get("bodies", 1) > 1 else 0.1
    out = []
    for b, (W, H, D) in enumerate(_sizes(case)):
        pos, tets, cell_sum, split = _block(W, H, D, h, case.get("mirrored", False))
        if case.get("jitter"):  # an unstructured mesh's uneven elements
            inner = (pos[:, 0] > 0) & (pos[:, 0] < W * h)
            pos[inner] += r.uniform(-0.12 * h, 0.12 * h, (int(inner.sum()), 3))
        boxes = case.get("bodies", 1) > 1 and not fit
        if boxes:  # each dropped on its own ground plane, turned about z and x
            a, c = r.uniform(0, 2 * np.pi, 2)
            R = np.array([[np.cos(a), -np.sin(a), 0], [np.sin(a), np.cos(a), 0], [0, 0, 1]]) @ \
                np.array([[1, 0, 0], [0, np.cos(c), -np.sin(c)], [0, np.sin(c), np.cos(c)]])
            pos = pos @ R.T
            pos[:, 1] += 0.2 + 0.8 * r.rand() - pos[:, 1].min()
        pos[:, 2] += 5.0 * b
        xyz = pos.astype(np.float32)
        body = dict(xyz=xyz, tets=tets, cell_sum=cell_sum, split=split,
                    density=float(r.uniform(500.0, 2000.0)) if boxes else 1000.0,
                    pinned=None if boxes else (pos[:, 0] == 0.0).astype(np.uint8),
                    velocity=r.normal(0.0, 0.05, xyz.shape).astype(np.float32), mu=None)
        yeoh = case["energy"] == "yeoh" or (case["energy"] == "mixed" and b % 2 == 1)
        mod = float(10.0 ** r.uniform(4.0, 6.0)) if boxes else 5e4 if yeoh else 1e5
        nu = case.get("nu", 0.5)
        body["settings"] = dict(
            energy=xf.ENERGY_CONTINUOUS_SKIN if case["energy"] == "ring" else
            xf.ENERGY_YEOH_SKIN_FAST if yeoh else xf.ENERGY_MIXED_SEL,
            simultaneous=0 if case.get("serial") else 1,
            compliance=0.1095 / mod if yeoh or case["energy"] == "ring" else 1.0 / mod,
            poissons_ratio=0.45 if case["energy"] == "ring" else nu, gravity=(0.0, -9.81), yeoh=_YEOH,
            collide=xf.COLLIDE_GROUND | (xf.COLLIDE_SPHERE if case.get("sphere") else 0),
            ground_y=0.0 if boxes else -0.5 * H * h - 0.3, friction=0.5,
            sphere_c0=(0.0, -0.5 * H * h - 0.3, 0.0), sphere_v=(1.0, 0.0, 0.0), sphere_r=0.3,
            damping=case.get("damping", 0.0), rayleigh_type=case.get("rayleigh", 0),
            pbd_damping=case.get("pbd", 0.0), pbd_damping_amortized=8.0 * case.get("pbd", 0.0),
            volume_passes=case.get("volume_passes", 0))
        if fit:  # the optimiser's present estimate: smooth in space, within a decade
            cen = pos[tets].mean(axis=1) / h
            k = r.uniform(-0.5, 0.5, 3)
            lg = 0.8 * np.sin(cen @ k + r.uniform(0, 6.28)) + 0.2 * r.normal(size=len(tets))
            base = (1e5 / 0.1095) if yeoh else 1e5
            body["mu"] = (base * np.exp(lg)).astype(np.float32)
        out.append(body)
    return out


def _dt(case):
    return float(np.float32(1.0) / np.float32(60 * case["substeps"]))


# -------------------------------------------------------------------- cases

def listed():
    return [
        # The C++ drop-in's call pattern on the smallest body: settings and
        # one substep per call, the positions read for drawing. The smallest
        # call; latency is everything.
        dict(name="substep_beam12x4x4", kind="substep", W=12, H=4, D=4, energy="neo", schedule="colour", substeps=20,
             frames=1),
        # An interactive frame of the same body with the default options.
        dict(name="frame_beam12x4x4", kind="frame", W=12, H=4, D=4, energy="neo", schedule="colour", substeps=20,
             frames=1),
        # A mid-size body with the reference's damping passes and one volume
        # pass, compressible: all per-substep passes that settings can add.
        dict(name="frame_damped21x9x7", kind="frame", W=21, H=9, D=7, energy="neo", schedule="colour", substeps=20,
             frames=1, nu=0.45, damping=0.01, rayleigh=2, pbd=0.002, volume_passes=1),
        # An uneven mesh with alternating diagonals (no short colouring), as
        # meshes from files have; greedy colours.
        dict(name="frame_uneven17x11x10", kind="frame", W=17, H=11, D=10, energy="yeoh", schedule="colour",
             substeps=20, frames=1, mirrored=True, jitter=True),
        # A beam with the caller's own 24-colouring, one launch per colour.
        dict(name="frame_slabs64x16x16", kind="frame", W=64, H=16, D=16, energy="yeoh", schedule="slabs",
             substeps=30, frames=1),
        # The benchmark beam with the sweep-block schedule and both contacts.
        dict(name="frame_beam96x24x24", kind="frame", W=96, H=24, D=24, energy="yeoh", schedule="blocks",
             substeps=30, frames=1, sphere=True, block_size=256),
        # A large beam, written out every fourth frame: bound by throughput.
        dict(name="frames_beam192x48x48", kind="frame", W=192, H=48, D=48, energy="yeoh", schedule="blocks",
             substeps=30, frames=4, sphere=True, block_size=256),
        # A batch of uneven free boxes with mixed materials.
        dict(name="frame_boxes64", kind="frame", bodies=64, lo=3, hi=24, mesh=2, energy="mixed", schedule="blocks",
             substeps=20, frames=2, block_size=128, block_lanes=128),
        # The vertex-ring energy, one launch per ring colour.
        dict(name="frame_rings48x12x12", kind="frame", W=48, H=12, D=12, energy="ring", schedule="slabs",
             substeps=30, frames=1),
        # Gradients of a trajectory loss for one body, in both element models.
        dict(name="adjoint_beam16x4x4", kind="adjoint", W=16, H=4, D=4, energy="neo", schedule="colour", substeps=20,
             frames=10, loss_every=5),
        dict(name="adjoint64_beam16x4x4", kind="adjoint", W=16, H=4, D=4, energy="neo", schedule="colour",
             substeps=20, frames=5, loss_every=5, fp64=True),
        # One optimiser iteration of batched fitting: new moduli, the state
        # reset, loss at every frame, gradients for every tet.
        dict(name="adjoint_fit24", kind="adjoint", bodies=24, lo=4, hi=16, mesh=4, energy="yeoh", schedule="colour",
             substeps=40, frames=5, loss_every=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["substep", "frame", "frame", "frame", "damped", "slabs", "blocks", "boxes", "ring", "adjoint",
                       "adjoint", "fit"])
    energy = rng.choice(["neo", "yeoh"])
    dims = lambda lo, hi: dict(W=_log_int(rng, lo, 4 * hi), H=_log_int(rng, lo, hi), D=_log_int(rng, lo, hi))  # noqa: E731
    if kind == "substep":
        return dict(kind="substep", **dims(2, 8), energy=energy, schedule="colour", substeps=20, frames=1)
    if kind == "frame":
        return dict(kind="frame", **dims(2, 14), energy=energy, schedule="colour", substeps=rng.choice([10, 20, 30]),
                    frames=1, mirrored=rng.random() < 0.4, jitter=rng.random() < 0.5, serial=rng.random() < 0.15,
                    nu=rng.choice([0.5, 0.5, 0.49, 0.45]))
    if kind == "damped":
        return dict(kind="frame", **dims(2, 10), energy=energy, schedule="colour", substeps=20, frames=1, nu=0.45,
                    damping=rng.choice([0.0, 0.01, 0.02]), rayleigh=rng.randint(0, 3), pbd=rng.choice([0.0, 0.002]),
                    volume_passes=rng.randint(0, 2))
    if kind == "slabs":
        return dict(kind="frame", **dims(6, 20), energy=energy, schedule="slabs", substeps=30, frames=1)
    if kind == "blocks":
        return dict(kind="frame", **dims(6, 36), energy=energy, schedule="blocks", substeps=30, frames=1,
                    sphere=rng.random() < 0.5, block_size=rng.choice([128, 256]))
    if kind == "boxes":
        lo = rng.randint(2, 6)
        return dict(kind="frame", bodies=_log_int(rng, 2, 64), lo=lo, hi=lo + rng.randint(2, 14),
                    mesh=rng.randint(0, 1 << 20), energy="mixed", schedule=rng.choice(["blocks", "colour"]),
                    substeps=20, frames=1, block_size=128)
    if kind == "ring":
        return dict(kind="frame", **dims(3, 12), energy="ring", schedule=rng.choice(["slabs", "colour"]), substeps=30,
                    frames=1)
    if kind == "adjoint":
        return dict(kind="adjoint", **dims(2, 6), energy=energy, schedule="colour", substeps=20,
                    frames=rng.randint(2, 6), loss_every=rng.randint(1, 3), fp64=rng.random() < 0.3)
    return dict(kind="adjoint", bodies=_log_int(rng, 2, 24), lo=4, hi=rng.randint(6, 14), mesh=rng.randint(0, 1 << 20),
                energy="yeoh", schedule="colour", substeps=40, frames=rng.randint(1, 3), loss_every=1)


def _structured(case):
    """Cases whose caller brings the 24-colouring of the block (the fitting
    beams as well); the others leave the colouring to the library."""
    return not case.get("mirrored") and (case["schedule"] == "slabs" or case["kind"] == "adjoint" and
                                         case.get("bodies", 1) > 1)


def _colours(body):
    return (6 * (body["cell_sum"] % 4) + body["split"]).astype(np.uint32)


def prepare(case, seed):
    bodies = _inputs(case, seed)
    sc = xf.Scene(_context())
    for b in bodies:
        sc.add_body(b["xyz"], b["tets"], b["density"], pinned=b["pinned"], velocity=b["velocity"], tet_mu=b["mu"],
                    tet_colour=_colours(b) if _structured(case) else None)
    blocks = case["schedule"] == "blocks"
    sc.finalize(block_size=case.get("block_size", 64), xcd_slabs=case["schedule"] == "slabs", sweep_blocks=blocks,
                launch_mode=xf.LAUNCH_BLOCKS if blocks else xf.LAUNCH_PER_COLOUR,
                block_lanes=case.get("block_lanes", 0))
    settings = [xf.default_settings(**b["settings"]) for b in bodies]
    for i, s in enumerate(settings):
        sc.set_settings(i, s)
    state = dict(scene=sc, settings=settings, dt=_dt(case), substeps=case["substeps"], frames=case["frames"],
                 kind=case["kind"], n=len(bodies))
    if case["kind"] == "adjoint":
        n_loss = case["frames"] // case["loss_every"]
        state["loss_at"] = np.array([(j + 1) * case["loss_every"] * case["substeps"] for j in range(n_loss)], np.uint32)
        # observed positions: a sag that grows with time
        tg = []
        for j in range(n_loss):
            row = []
            for b in bodies:
                p = b["xyz"].astype(np.float64)
                t = (j + 1) * case["loss_every"] / 60.0
                p[:, 1] -= 2.0 * t * t * (p[:, 0] / max(p[:, 0].max(), 0.1)) ** 2
                row.append(p.ravel())
            tg.append(np.concatenate(row))
        state.update(targets=np.array(tg), mu=[b["mu"] for b in bodies], fp64=bool(case.get("fp64")),
                     x0=[(b["xyz"].astype(np.float64), np.zeros(b["xyz"].shape)) for b in bodies])
    return state


def run(state):
    sc = state["scene"]
    if state["kind"] == "adjoint":
        for i in range(state["n"]):
            sc.set_tet_mu(i, state["mu"][i])
            sc.set_state(i, *(a.ravel() for a in state["x0"][i]))
        sc.set_time(0.0)
        loss, grad = sc.adjoint(state["frames"] * state["substeps"], state["dt"], state["loss_at"], state["targets"],
                                window=state["substeps"], fp64=state["fp64"])
        return {"loss": loss, "grad": grad}
    if state["kind"] == "substep":
        sc.set_settings(0, state["settings"][0])
        sc.step(1, state["dt"])
    else:
        for _ in range(state["frames"]):
            sc.step(state["substeps"], state["dt"])
    got = [sc.get_state(i) for i in range(state["n"])]
    if state["n"] == 1:
        return {"x": got[0][0], "v": got[0][1]}
    return {"x": np.concatenate([g[0] for g in got]), "v": np.concatenate([g[1] for g in got])}


def work(case):
    tets = nodes = 0
    for W, H, D in _sizes(case):
        tets += 6 * W * H * D
        nodes += (W + 1) * (H + 1) * (D + 1)
    steps = 1 if case["kind"] == "substep" else case["substeps"] * case["frames"]
    # state in and out (x, v in FP64), inverse masses, tet indices and element constants once
    bytes_ = 2 * 48 * nodes + 4 * nodes + 80 * tets
    # FP32 operations: 503 per tet projection, about 40 per node and substep
    per_tet, per_node = 503, 40
    if case["energy"] == "ring":
        per_tet = 4 * 300 + 4 * 60  # four ring tets per tet, and the ring nodes' sums
    per_tet += 180 * case.get("volume_passes", 0)
    if case.get("damping", 0.0) > 0.0 and case.get("rayleigh", 0) >= 2:
        per_tet += 500
    if case.get("pbd", 0.0) > 0.0:
        per_tet += 350
    if case["kind"] == "adjoint":
        per_tet += 1100  # the reverse of a projection
        bytes_ += 4 * tets + 8 * tets + (case["frames"] // case["loss_every"]) * 24 * nodes
    return {"bytes": bytes_, "flops": steps * (per_tet * tets + per_node * nodes)}


# ---------------------------------------------------------- results in FP64

def _greedy(n_nodes, tets):
    """First colour, in input order, that none of the tet's nodes has yet."""
    used = [0] * n_nodes
    out = []
    for a, b, c, d in tets.tolist():
        m = used[a] | used[b] | used[c] | used[d]
        k = (~m & (m + 1)).bit_length() - 1
        out.append(k)
        bit = 1 << k
        used[a] |= bit
        used[b] |= bit
        used[c] |= bit
        used[d] |= bit
    return np.array(out)


def exact(case, seed):
    """Positions of the rollout in FP64, for the cases whose sweep order
    follows from the mesh alone (the caller's colours, or the first free
    colour in input order) with the simultaneous solve and no damping. None
    where the sweep order or the passes are a schedule of the library's own,
    for gradients, and for velocities (a position difference over one
    substep, which carries the rounding of FP32 elements some hundred times
    enlarged). The order inside a colour does not matter: its tets share no
    node."""
    if case["kind"] == "adjoint" or case["schedule"] == "blocks" or case["energy"] == "ring" or \
            case.get("bodies", 1) > 1 or case.get("serial") or case.get("volume_passes") or case.get("damping") or \
            case.get("pbd") or case.get("sphere"):
        return None
    b = _inputs(case, seed)[0]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = lambda a: torch.tensor(np.asarray(a, np.float64), device=dev)  # noqa: E731
    tets_np = b["tets"]
    if len(tets_np) > 200000:
        return None
    colour = _colours(b) if _structured(case) else _greedy(len(b["xyz"]), tets_np)
    pos = b["xyz"].astype(np.float64)
    vol = _volumes(pos, tets_np)
    mass = np.zeros(len(pos))
    np.add.at(mass, tets_np.ravel(), np.repeat(b["density"] * vol / 4.0, 4))
    s = b["settings"]
    f32 = lambda v: float(np.float32(v))  # noqa: E731
    dt = _dt(case)
    mu = 1.0 / f32(s["compliance"])
    nu = f32(s["poissons_ratio"])
    ratio = (1.0 - 2.0 * nu) / (2.0 * nu)  # mu / lambda
    pinned = torch.tensor(b["pinned"].astype(bool), device=dev)
    w = torch.where(pinned, torch.zeros((), dtype=torch.float64, device=dev), 1.0 / f64(mass))
    x, v = f64(pos), f64(b["velocity"])
    g = f64([f32(s["gravity"][0]) * dt, f32(s["gravity"][1]) * dt, 0.0])
    yeoh = [f32(c) for c in s["yeoh"]]
    is_yeoh = s["energy"] == xf.ENERGY_YEOH_SKIN_FAST
    a = 1.0 + ratio
    groups = []
    for c in range(int(colour.max()) + 1):
        sel = np.flatnonzero(colour == c)
        t = torch.tensor(tets_np[sel], device=dev)
        Dm = (x[t[:, :3]] - x[t[:, 3:]]).transpose(1, 2)
        B = torch.linalg.inv(Dm)
        V = f64(vol[sel])
        groups.append((t, B, w[t], 1.0 / (mu * V) / (dt * dt), ratio / (mu * V) / (dt * dt)))
    ground, fr = f32(s["ground_y"]), f32(s["friction"])
    for _ in range(1 if case["kind"] == "substep" else case["substeps"] * case["frames"]):
        v = v + g
        o = x
        x = x + v * dt
        for t, B, wt, al0, al1 in groups:
            xt = x[t]
            F = (xt[:, :3] - xt[:, 3:]).transpose(1, 2).matmul(B)
            U0 = (F * F).sum(dim=(1, 2))
            G0 = 2.0 * F
            if is_yeoh:
                im = U0 - 3.0
                U0 = torch.clamp(yeoh[0] * im + yeoh[1] * im ** 2 + yeoh[2] * im ** 3, min=1e-4)
                G0 = G0 * (yeoh[0] + 2.0 * yeoh[1] * im + 3.0 * yeoh[2] * im ** 2)[:, None, None]
            cof = torch.stack([torch.linalg.cross(F[:, :, 1], F[:, :, 2]), torch.linalg.cross(F[:, :, 2], F[:, :, 0]),
                               torch.linalg.cross(F[:, :, 0], F[:, :, 1])], dim=2)
            d = (F[:, :, 0] * cof[:, :, 0]).sum(dim=1) - a
            U1 = d * d
            Bt = B.transpose(1, 2).contiguous()
            g0 = G0.matmul(Bt).transpose(1, 2)
            g1 = (cof * (2.0 * d)[:, None, None]).matmul(Bt).transpose(1, 2)
            g0 = torch.cat([g0, -g0.sum(dim=1, keepdim=True)], dim=1)
            g1 = torch.cat([g1, -g1.sum(dim=1, keepdim=True)], dim=1)
            A0 = (wt * (g0 * g0).sum(dim=2)).sum(dim=1) + 1e-22 + 2.0 * U0 * al0
            A1 = (wt * (g0 * g1).sum(dim=2)).sum(dim=1) + 1e-22
            A2 = (wt * (g1 * g1).sum(dim=2)).sum(dim=1) + 1e-22 + 2.0 * U1 * al1
            p, q = A1 / A0, A1 / A2
            be0, be1 = -2.0 * U0 / A0, -2.0 * U1 / A2
            inv = 1.0 / torch.clamp(1.0 - p * q, min=1e-8)
            l0, l1 = inv * (be0 - p * be1), inv * (be1 - be0 * q)
            x[t] = xt + wt[:, :, None] * (l0[:, None, None] * g0 + l1[:, None, None] * g1)
        x = torch.where(pinned[:, None], o, x)
        depth = ground - x[:, 1]
        hit = (depth > 0) & ~pinned
        dx, dz = x[:, 0] - o[:, 0], x[:, 2] - o[:, 2]
        t2 = torch.sqrt(dx * dx + dz * dz)
        keep = torch.where(fr * depth >= t2, torch.zeros_like(t2), 1.0 - fr * depth / torch.clamp(t2, min=1e-300))
        x = torch.where(hit[:, None], torch.stack([o[:, 0] + dx * keep, torch.full_like(dx, ground), o[:, 2] + dz * keep],
                                                  dim=1), x)
        v = (x - o) / dt
    return {"x": x.reshape(-1).cpu().numpy(), "v": None}
