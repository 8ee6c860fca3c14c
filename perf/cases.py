"""Performance cases of the DEM engine and of the learned coarse step, over the sizes and options
users run them with.

``listed()`` names the measured cases, ``draw(rng)`` gives more of the same ranges. ``prepare``
builds what a program has in hand before the call (a loaded context, a trained network), ``run``
is one pass through the public entry points, ``exact`` is the same result from plain torch in 64
bits. The step cases rewind to an in-memory snapshot (Scene.loadTmp) at each pass, so that every
pass does the same work however often it is called.
"""
import math

import numpy as np
import torch

from woo_amd import surrogate
from woo_amd._native import FACET, LAW_HERTZDMT, LAW_IDEALELPL, PHYS_FRICT, PHYS_HERTZ, SPHERE, WALL, Device
from woo_amd.surrogate import A0, COARSE, R0, V0, VERLET, Network

RHO, POISSON, EN = 3000., .25, .6  # the material of the benchmark's workloads
ENGINES = ["Collider", "ContactLoop", "Leapfrog"]
DRUM_ENGINES = ["Collider", "ContactLoop", "IntraForce", "Leapfrog"]
WARM = 10  # steps before the snapshot, so that contacts with history exist

# the largest size of each kind of case (spheres, or nodes of the network's graph)
RANGE = dict(engines=(200, 5000), walls=(500, 100000), periodic=(1500, 1000000), fp32=(1500, 250000),
             drum=(10000, 200000), batch=(4, 64), observe=(2000, 400000), pack=(2000, 150000),
             learned=(2000, 60000), forward=(2000, 120000), train=(1000, 25000))
STEPS = dict(engines=50, walls=100, periodic=150, fp32=150, drum=60, batch=96)
SWEEPS = 48       # relaxation sweeps of a packing pass
COARSE_STEPS = 5  # learned coarse steps of a pass


def listed():
    return [
        # a small box of spheres whose engines a host program calls one by one: latency and launches
        dict(name="engines_300", kind="engines", n=300),
        # the 2000-sphere deposition between walls, friction, plain step loop
        dict(name="walls_2000", kind="walls", n=2000, graph=False),
        # periodic Hertz gas of grains, graph replay: an ordinary size and the benchmark's
        dict(name="periodic_20k", kind="periodic", n=20001, graph=True),
        dict(name="periodic_1m", kind="periodic", n=1000000, graph=True),
        # the FP32 contact form
        dict(name="fp32_250k", kind="fp32", n=250000, graph=True),
        # rotating drum of facets and end walls with the forces on the facet nodes
        dict(name="drum_200k", kind="drum", n=200000, graph=True),
        # parametric study: many deposition scenes in one context
        dict(name="batch_64", kind="batch", n=64, graph=True),
        # what a monitoring program reads from a state: coordination, stress, energy, timestep
        dict(name="observe_400k", kind="observe", n=400000),
        # initial condition: overlapping random spheres pushed apart
        dict(name="pack_150k", kind="pack", n=150000),
        # learned coarse steps of a falling column: graph, network, advance
        dict(name="learned_60k", kind="learned", n=60000),
        # the network's accelerations for a graph in hand
        dict(name="forward_120k", kind="forward", n=120000),
        # one training step on a graph kept on the device: loss, gradients, Adam
        dict(name="train_25k", kind="train", n=25000),
    ]


def draw(rng):
    kind = rng.choice(sorted(RANGE))
    lo, hi = RANGE[kind]
    c = dict(kind=kind, n=int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))
    if kind in ("walls", "periodic", "fp32", "drum", "batch"):
        c["graph"] = rng.random() < .7
    return c


# ---------------------------------------------------------------- inputs
def _block(nb, rmin, rmax, phi, gen, sweeps=200):
    """nb spheres in a periodic cube at solid fraction phi, pushed apart (plain torch)"""
    r = rmin + (rmax - rmin) * torch.rand(nb, generator=gen, device="cuda", dtype=torch.float64)
    L = (float((4 / 3. * math.pi * r ** 3).sum()) / phi) ** (1 / 3.)
    x = (torch.rand(nb, 3, generator=gen, device="cuda", dtype=torch.float64) * L).float()
    rs = ((r[:, None] + r[None, :]) * .999).float()  # some of the pairs touch
    rs.fill_diagonal_(0.)
    for _ in range(sweeps):
        d = x[None, :, :] - x[:, None, :]
        d -= L * torch.round(d / L)
        dist = d.square().sum(-1).sqrt_()
        w = torch.clamp(rs - dist, min=0.) / dist.clamp(min=1e-9)
        x = x - .5 * (w[:, :, None] * d).sum(1)
    x = x.double()
    return torch.remainder(x, L).clamp(max=L * (1 - 1e-9)), r, L


def _packing(n, rmin, rmax, phi, rng, gen, extent=None, block=None):
    """Dense packing by periodic repetition of a relaxed block. Without extent: n spheres filling
    a periodic cube; with extent (lengths): every sphere centre of the box [0, extent]."""
    if extent is None:
        t = [max(1, round((n / 1400.) ** (1 / 3.)))] * 3
        x, r, L = _block(-(-n // t[0] ** 3), rmin, rmax, phi, gen)
    else:
        x, r, L = block or _block(min(1200, max(300, n)), rmin, rmax, phi, gen)
        t = [int(math.ceil(e / L)) for e in extent]
    x, r = x.cpu().numpy(), r.cpu().numpy()
    off = np.stack(np.meshgrid(*[np.arange(k) for k in t], indexing="ij"), -1).reshape(-1, 1, 3) * L
    pos, rad = (x[None] + off).reshape(-1, 3), np.tile(r, len(off))
    if extent is None:  # a few vacancies, so that any n can be asked for
        keep = np.sort(rng.permutation(len(pos))[:n])
        return pos[keep], rad[keep], tuple(k * L for k in t)
    return pos, rad, None


def _lowest(pos, rad, n):
    """the lowest n spheres, without those that overlap another after being set onto a boundary"""
    i = np.argsort(pos[:, 2], kind="stable")[:int(1.25 * n) + 50]
    pos, rad = pos[i], rad[i]
    a, b = _pairs(_t(pos), 2 * float(rad.max()))
    a, b = a.cpu().numpy(), b.cpu().numpy()
    bad = np.linalg.norm(pos[a] - pos[b], axis=1) < .99 * (rad[a] + rad[b])
    keep = np.ones(len(rad), bool)
    keep[b[bad]] = False
    if keep.sum() < n:
        raise RuntimeError("packing: too few spheres")
    return pos[keep][:n], rad[keep][:n]


def _bed(n, r0, r1, rng, gen, phi=.5, aspect=1., block=None):
    """n spheres on the bottom of a box of square cross-section; returns pos, radius, width"""
    v = float(np.mean(4 / 3. * math.pi * np.linspace(r0, r1, 64) ** 3))
    W = max((n * v / phi / aspect) ** (1 / 3.), 6 * r1)
    H = 1.7 * n * v / phi / W ** 2 + 12 * r1
    for _ in range(4):
        pos, rad, _ = _packing(n, r0, r1, phi, rng, gen, (W, W, H), block)
        ok = np.all((pos[:, :2] > rad[:, None]) & (pos[:, :2] < W - rad[:, None]), axis=1) & (pos[:, 2] > rad)
        i = np.flatnonzero(ok)
        if len(i) >= 1.25 * n + 50:
            break
        H *= 1.5
    pos, rad = pos[i], rad[i]
    low = pos[:, 2] < 1.4 * rad
    pos[low, 2] = .998 * rad[low]
    return _lowest(pos, rad, n) + (W,)


def _box_walls(W, H, off=(0., 0., 0.), scene=0):
    out = []
    for sense, c in ((1, (0., 0., 0.)), (-1, (W, W, H))):
        for ax in range(3):
            p = np.array(off, dtype=float)
            p[ax] += c[ax]
            out.append((p, ax, sense, scene))
    return out


def _scene(case, seed):
    """the spheres, boundary bodies, materials and field of a step case, from the seed alone"""
    kind, n = case["kind"], case["n"]
    rng = np.random.default_rng([seed, 77])
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)
    s = dict(walls=[], verts=np.zeros((0, 9)), fake=np.zeros((0, 3)), gravity=(0., 0., 0.), cell=None, damping=0.,
             mat=None, scene=None, dts=None, hertz=True)
    if kind in ("periodic", "fp32", "observe"):
        s["pos"], s["radius"], s["cell"] = _packing(n, 2e-3, 4e-3, .55, rng, gen)
        s["mats"] = [dict(kind=1, density=RHO, young=1e8, ktDivKn=.2, tanPhi=.4, surfEnergy=0., alpha=0.)]
        s["vel"] = rng.normal(0., .1, (n, 3))
        s["dt"] = .3 * 2e-3 / math.sqrt(1e8 / RHO)
    elif kind in ("engines", "walls"):
        s["pos"], s["radius"], W = _bed(n, 5e-3, 5e-3, rng, gen)
        s["walls"] = _box_walls(W, float(np.max(s["pos"][:, 2])) + .1)
        s["mats"] = [dict(kind=0, density=RHO, young=1e7, ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)]
        s.update(vel=rng.normal(0., .05, s["pos"].shape), dt=.5 * 5e-3 / math.sqrt(1e7 / RHO), gravity=(0., 0., -9.81),
                 damping=.2, hertz=False)
    elif kind == "batch":
        size = np.exp(np.random.default_rng(n).uniform(math.log(500), math.log(8000), n)).astype(int)
        young = np.exp(rng.uniform(math.log(1e6), math.log(1e8), n))
        P, R, S, V, x = [], [], [], [], 0.
        block = _block(1200, 5e-3, 5e-3, .4, gen)
        for k in range(n):
            p, r, W = _bed(int(size[k]), 5e-3, 5e-3, rng, gen, phi=.4, block=block)
            P.append(p + np.array([x, 0., 0.]))
            R.append(r)
            S.append(np.full(len(r), k))
            V.append(rng.normal(0., .05, p.shape))
            s["walls"] += _box_walls(W, float(np.max(p[:, 2])) + .1, (x, 0., 0.), k)
            x += W + .05
        s.update(pos=np.concatenate(P), radius=np.concatenate(R), scene=np.concatenate(S), vel=np.concatenate(V))
        s["mat"] = s["scene"]
        s["mats"] = [dict(kind=0, density=RHO, young=float(e), ktDivKn=.2, tanPhi=float(t), surfEnergy=0., alpha=0.)
                     for e, t in zip(young, rng.uniform(.1, .9, n))]
        s["dts"] = .5 * 5e-3 / np.sqrt(young / RHO)
        s.update(dt=float(s["dts"][0]), gravity=(0., 0., -9.81), damping=.2, hertz=False)
    elif kind == "drum":
        rlo, rhi, omega, div = .8e-3, 2.5e-3, 2., 128
        v = float(np.mean(4 / 3. * math.pi * np.linspace(rlo, rhi, 64) ** 3))
        R = (2 * n * v / (.55 * math.pi * .8)) ** (1 / 3.)  # half full, length 0.8 R
        Ln, Rin = .8 * R, R * math.cos(math.pi / div)
        pos, rad, _ = _packing(n, rlo, rhi, .55, rng, gen, (Ln, 2 * R, 1.7 * R))
        pos = pos - np.array([Ln / 2, R, R])
        # the outermost spheres are set onto the mantle
        w = 2 * math.pi / div
        phi = np.arctan2(pos[:, 2], pos[:, 1])
        rho, onto = np.hypot(pos[:, 1], pos[:, 2]), (Rin - .998 * rad) / np.cos(np.mod(phi, w) - w / 2)
        out = (rho < onto) & (rho > onto - .4 * rad)
        pos[out, 1:] *= (onto[out] / rho[out])[:, None]
        i = np.flatnonzero((np.abs(pos[:, 0]) < Ln / 2 - rad) & (out | (rho < Rin - rad)))
        pos, rad = _lowest(pos[i], rad[i], n)
        th = np.linspace(0, 2 * math.pi, div + 1)
        a = np.stack([np.full(div + 1, -Ln / 2), R * np.cos(th), R * np.sin(th)], 1)
        b = a + np.array([Ln, 0., 0.])
        verts = np.stack([np.concatenate([a[:-1], b[:-1], b[1:]], 1), np.concatenate([a[:-1], b[1:], a[1:]], 1)],
                         1).reshape(-1, 9)
        nn = np.cross(verts[:, 3:6] - verts[:, :3], verts[:, 6:] - verts[:, :3])
        nn /= np.linalg.norm(nn, axis=1)[:, None]
        s.update(pos=pos, radius=rad, verts=verts, fake=-R * omega * np.cross(nn, [1., 0., 0.]),
                 vel=rng.normal(0., .1, pos.shape), gravity=(0., 0., -9.81), dt=.3 * rlo / math.sqrt(1e8 / RHO))
        s["walls"] = [(np.array([-Ln / 2, 0., 0.]), 0, 1, 0), (np.array([Ln / 2, 0., 0.]), 0, -1, 0)]
        s["mats"] = [dict(kind=1, density=RHO, young=1e8, ktDivKn=.2, tanPhi=.4, surfEnergy=0., alpha=0.)]
    ns = len(s["pos"])
    s["mat"] = np.zeros(ns, int) if s["mat"] is None else s["mat"]
    s["scene"] = np.zeros(ns, int) if s["scene"] is None else s["scene"]
    s["mass"] = 4 / 3. * math.pi * s["radius"] ** 3 * RHO
    s["inertia"] = .4 * s["mass"] * s["radius"] ** 2
    return s


def _load(dev, s):
    """the scene into a context: walls, then facets, then spheres"""
    nw, nf, ns = len(s["walls"]), len(s["verts"]), len(s["pos"])
    nb = nw + nf
    N = nb + ns

    def full(width, boundary, spheres, dtype=float):
        a = np.zeros((N, width) if width > 1 else N, dtype)
        a[:nb], a[nb:] = boundary, spheres
        return a

    pos = full(3, 0., s["pos"])
    fv, fk = np.zeros((N, 9)), np.zeros((N, 3))
    axis, sense = np.zeros(N, np.int32), np.zeros(N, np.int32)
    scene, mat = full(1, 0, s["scene"], np.int32), full(1, 0, s["mat"], np.int32)
    for k, (p, ax, se, sc) in enumerate(s["walls"]):
        pos[k], axis[k], sense[k], scene[k], mat[k] = p, ax, se, sc, sc
    pos[nw:nb], fv[nw:nb], fk[nw:nb] = s["verts"][:, :3], s["verts"], s["fake"]
    shape = np.concatenate([np.full(nw, WALL), np.full(nf, FACET), np.full(ns, SPHERE)]).astype(np.int32)
    dev.set_field(gravity=s["gravity"], periodic=s["cell"] is not None, cell=s["cell"] or (1., 1., 1.))
    dev.set_materials(s["mats"])
    dev.upload_particles(shape=shape, pos=pos, radius=full(1, 0., s["radius"]), wallAxis=axis, wallSense=sense,
                         material=mat, mask=full(1, 3, 5, np.uint32), flags=full(1, 63, 0, np.uint32),
                         integrated=full(1, 0, 1, np.uint8), vel=full(3, 0., s["vel"]), mass=full(1, 0., s["mass"]),
                         inertia=full(3, 0., s["inertia"][:, None]), scene=scene,
                         **(dict(facetVerts=fv, fakeVel=fk) if nf else {}))
    if s["dts"] is not None:
        dev.set_scenes(s["dts"])


def _contact(s):
    return (dict(physKind=PHYS_HERTZ, lawKind=LAW_HERTZDMT, poisson=POISSON, en=EN) if s["hertz"] else
            dict(physKind=PHYS_FRICT, lawKind=LAW_IDEALELPL))


def _column(case, seed):
    """falling column of the learned step, as the engine takes it: one floor wall, spheres of 2
    to 3 mm, moving"""
    rng = np.random.default_rng([seed, 5])
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    p, r, _ = _bed(case["n"], 2e-3, 3e-3, rng, gen, phi=.58, aspect=2.2)
    arr = surrogate.engine_arrays(p, r)
    arr["vel"][1:] = rng.normal(0., .05, p.shape)
    return arr


def _params(seed):
    """weights of a trained network's size: Glorot uniform, small biases"""
    rng = np.random.default_rng([seed, 9])
    p = []
    for K, used, O in ((32, 7, 64), (160, 143, 64), (128, 128, 64), (160, 143, 64), (128, 128, 64), (64, 64, 3)):
        w = np.zeros((K, O))
        w[:used] = rng.uniform(-1, 1, (used, O)) * math.sqrt(6. / (used + O))
        p += [w.ravel(), rng.normal(0., .05, O)]
    p[-2] *= .05  # accelerations of the order of the training targets
    return np.concatenate(p).astype(np.float32)


def _targets(n, seed):
    return np.random.default_rng([seed, 11]).normal(0., .3, (n, 3)) * A0


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pack":
        rng = np.random.default_rng([seed, 3])
        n = case["n"]
        radius = rng.uniform(2e-3, 4e-3, n)
        L = (float(np.sum(4 / 3. * math.pi * radius ** 3)) / .55) ** (1 / 3.)
        pos = rng.uniform(0., L, (n, 3))
        dev = Device(0)
        dev.set_field(periodic=True, cell=(L,) * 3)
        dev.set_materials([dict(kind=0, density=1., young=1., ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
        dev.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=radius, mass=np.ones(n),
                             inertia=np.ones((n, 3)), vel=np.zeros((n, 3)))
        return dict(case=case, dev=dev, pos=pos)
    if kind in ("learned", "forward", "train"):
        arr = _column(case, seed)
        dev = Device(0)
        surrogate.upload(dev, arr)
        dev.collide(VERLET)
        net = Network(seed=1)
        net.set_params(_params(seed))
        st = dict(case=case, dev=dev, net=net)
        if kind == "learned":
            dev.snapshot(0)
        else:
            net.graph_from(dev, floorZ=0., force=True)
        if kind == "train":
            net.set_targets(_targets(len(arr["shape"]) - 1, seed))
            net.keep(0)
        return st
    s = _scene(case, seed)
    dev = Device(0)
    _load(dev, s)
    if kind == "fp32":
        dev.set_precision(32)
    if kind == "batch":
        dev.set_tuning(cfBlocks=2, graphSteps=8, skinSteps=16)
    cp = _contact(s)
    if kind != "fp32":  # (a rewind restarts the FP32 form's contact history)
        dev.run(ENGINES, WARM, 0, s["dt"], contact=cp, leapfrog=dict(damping=s["damping"]), dynDtPeriod=0)
    if kind != "observe":
        dev.snapshot(0)
    nb = len(s["walls"]) + len(s["verts"])
    return dict(case=case, dev=dev, dt=s["dt"], damping=s["damping"], contact=cp, nb=nb, cell=s["cell"],
                facets=np.arange(len(s["walls"]), nb))


def run(st):
    case, dev = st["case"], st["dev"]
    kind = case["kind"]
    if kind == "pack":
        dev.set("pos", st["pos"])
        ov, _ = dev.relax(SWEEPS, .005, tol=0.)
        return dict(pos=dev.get("pos"), overlap=ov)
    if kind == "forward":
        return st["net"].forward()
    if kind == "train":
        net = st["net"]
        loss = net.kept_loss(0)
        grads = net.grads()
        net.adam(1e-3)
        return dict(loss=loss, grads=grads)
    if kind == "learned":
        net = st["net"]
        dev.restore(0)
        dev.collide(VERLET)
        for _ in range(COARSE_STEPS):
            net.graph_from(dev, floorZ=0., maxDisp=.5e-3)
            net.forward(out=False)
            net.advance(dev, COARSE * surrogate.dem_dt())
        return dict(pos=dev.get("pos"), vel=dev.get("vel"))
    if kind == "observe":
        L = st["cell"]
        ob = dev.observables([.25 * x for x in L], [.75 * x for x in L])
        return dict(observables=np.array([ob["coordNumber"], ob["coordNumberSkipFree"], ob["solidFraction"]]),
                    stress=dev.stress(), kinetic=dev.kinetic_energy(), critDt=dev.crit_dt())
    dev.restore(0)
    if kind == "engines":
        for k in range(STEPS[kind]):
            dev.collide(-.05)
            dev.contact_loop(WARM + k, st["dt"], **st["contact"])
            dev.leapfrog(st["dt"], st["damping"])
        return dict(pos=dev.get("pos"), vel=dev.get("vel"), kinetic=dev.kinetic_energy())
    dev.run(DRUM_ENGINES if kind == "drum" else ENGINES, STEPS[kind], WARM if kind != "fp32" else 0, st["dt"],
            graph=case["graph"], contact=st["contact"], leapfrog=dict(damping=st["damping"]), dynDtPeriod=0)
    out = dict(pos=dev.get("pos"), vel=dev.get("vel"))
    if kind == "drum":
        out["nodeForce"], out["nodeTorque"] = dev.facet_nodes(st["facets"])
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Bytes: per step each particle's state read and written once and each contact's history
    read and written once (FP64); one result to the host. Flops: the law and the integrator, or
    the network's products."""
    kind, n = case["kind"], case["n"]
    per, con = 272., 1.  # bytes of a particle per step, contacts per particle
    if kind == "batch":
        n = n * 2700
    if kind in STEPS:
        k = STEPS[kind]
        con = .7 if kind in ("periodic", "fp32") else 1.5
        hist = 120. if kind == "fp32" else 232.
        return dict(bytes=k * n * (per + con * hist) + 48. * n, flops=k * n * (80. + 300. * con))
    if kind == "observe":
        return dict(bytes=n * (96. + .7 * 200.), flops=n * 200.)
    if kind == "pack":
        return dict(bytes=SWEEPS * n * 56. + 48. * n, flops=SWEEPS * n * 60.)
    deg = 7.
    fwd = 2. * n * (32 * 64 + 2 * (deg * 160 * 64 + 128 * 64) + 64 * 3)
    io = n * (64. + 12.) + n * deg * (64. + 8.)
    if kind == "learned":
        return dict(bytes=COARSE_STEPS * (io + n * 150.), flops=COARSE_STEPS * fwd)
    if kind == "forward":
        return dict(bytes=io, flops=fwd)
    return dict(bytes=2 * io, flops=3 * fwd)


def tolerance(case):
    kind = case["kind"]
    if kind in ("train", "forward"):
        return dict(rel=1e-2)     # BF16 activations and weights
    if kind == "learned":
        return dict(rel=5e-3)     # BF16 accelerations over five coarse steps
    if kind == "fp32":
        return dict(rel=1e-2)     # contact law in 32 bits: overlaps of 1e-3 radii keep four digits
    return dict(rel=1e-9)         # FP64 throughout; many steps amplify rounding


# ---------------------------------------------------------------- the same results in 64 bits
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


def _pairs(x, reach, cell=None):
    """index pairs closer than reach (nearest image in a periodic cell)"""
    n = len(x)
    lo = torch.zeros(3, device="cuda", dtype=torch.float64) if cell is not None else x.min(0).values
    ext = _t(cell) if cell is not None else (x.max(0).values - lo) + 1e-9
    nc = [max(1, min(300, int(float(e) / reach))) for e in ext]
    if n <= 3000 or (cell is not None and min(nc) < 3):
        i, j = torch.triu_indices(n, n, 1, device="cuda")
        return _close(x, i, j, reach, cell)
    h = ext / torch.tensor(nc, device="cuda", dtype=torch.float64)
    y = x - lo
    if cell is not None:
        y = y - torch.floor(y / ext) * ext
    nct = torch.tensor(nc, device="cuda")
    c = torch.minimum(torch.floor(y / h).long().clamp(min=0), nct - 1)
    key = (c[:, 2] * nc[1] + c[:, 1]) * nc[0] + c[:, 0]
    order = torch.argsort(key)
    start = torch.searchsorted(key[order], torch.arange(nc[0] * nc[1] * nc[2] + 1, device="cuda"))
    I, J = [], []
    for m in range(13, 27):  # this cell and half of its neighbours
        q = c + torch.tensor([m % 3 - 1, m // 3 % 3 - 1, m // 9 - 1], device="cuda")
        ok = torch.ones(n, dtype=torch.bool, device="cuda")
        if cell is not None:
            q = torch.remainder(q, nct)
        else:
            ok = ((q >= 0) & (q < nct)).all(1)
            q = q.clamp(min=0).minimum(nct - 1)
        k = (q[:, 2] * nc[1] + q[:, 1]) * nc[0] + q[:, 0]
        s0 = start[k]
        cnt = torch.where(ok, start[k + 1] - s0, 0)
        i = torch.repeat_interleave(torch.arange(n, device="cuda"), cnt)
        first = torch.cumsum(cnt, 0) - cnt
        j = order[torch.arange(len(i), device="cuda") - first[i] + s0[i]]
        if m == 13:
            i, j = i[i < j], j[i < j]
        i, j = _close(x, i, j, reach, cell)
        I.append(i)
        J.append(j)
    return torch.cat(I), torch.cat(J)


def _close(x, i, j, reach, cell):
    d = x[j] - x[i]
    if cell is not None:
        L = _t(cell)
        d = d - torch.floor(d / L + .5) * L
    k = d.square().sum(1) < reach * reach
    return torch.minimum(i[k], j[k]), torch.maximum(i[k], j[k])


def _dot(a, b):
    return (a * b).sum(-1)


def _unit(a):
    return a / a.norm(dim=-1, keepdim=True)


def _where(c, a, b):
    return torch.where(c[:, None], a, b)


def _closest(v, c):
    """closest point of triangles v [m, 3, 3] to points c [m, 3], and the plane distance"""
    v0, v1, v2 = v[:, 0], v[:, 1], v[:, 2]
    nn = torch.linalg.cross(v1 - v0, v2 - v0)
    nu = _unit(nn)
    pd = _dot(c - v0, nu)
    f = c - nu * pd[:, None]

    def seg(a, b):
        e = b - a
        return a + e * (_dot(f - a, e) / _dot(e, e)).clamp(0., 1.)[:, None]

    o = [_dot(torch.linalg.cross(b - a, nn), f - a) > 0 for a, b in ((v0, v1), (v1, v2), (v2, v0))]
    p = f
    for only, q in ((o[0] & ~o[1] & ~o[2], seg(v0, v1)), (o[1] & ~o[0] & ~o[2], seg(v1, v2)),
                    (o[2] & ~o[0] & ~o[1], seg(v2, v0)), (o[0] & o[1], v1), (o[0] & o[2], v0), (o[1] & o[2], v2)):
        p = _where(only, q, p)
    return p, pd


def _rotate(c0, c1, f):
    """f rotated by the orientation of a contact's node, and the node's rotated x axis. The
    orientation is the quaternion of the matrix with columns c0, c1, c0 x c1, which between
    renormalisations is not exactly a rotation (c1 is updated to second order)."""
    m = torch.stack([c0, c1, torch.linalg.cross(c0, c1)], 2)
    d = m.diagonal(dim1=1, dim2=2)
    tr = d.sum(1)
    q = torch.zeros(len(m), 4, device="cuda", dtype=torch.float64)
    i = d.argmax(1)
    for b in range(4):  # positive trace, else the largest diagonal element
        k = torch.nonzero(tr > 0 if b == 3 else (tr <= 0) & (i == b))[:, 0]
        M = m[k]
        if b == 3:
            t = (tr[k] + 1).sqrt()
            q[k, 3] = .5 * t
            for a in range(3):
                q[k, a] = (M[:, (a + 2) % 3, (a + 1) % 3] - M[:, (a + 1) % 3, (a + 2) % 3]) * .5 / t
        else:
            j, l = (b + 1) % 3, (b + 2) % 3
            t = (M[:, b, b] - M[:, j, j] - M[:, l, l] + 1).sqrt()
            q[k, b] = .5 * t
            q[k, 3] = (M[:, l, j] - M[:, j, l]) * .5 / t
            q[k, j] = (M[:, j, b] + M[:, b, j]) * .5 / t
            q[k, l] = (M[:, l, b] + M[:, b, l]) * .5 / t
    v, w = q[:, :3], q[:, 3:]

    def turn(u):
        uv = 2 * torch.linalg.cross(v, u)
        return u + w * uv + torch.linalg.cross(v, uv)

    x = torch.zeros_like(f)
    x[:, 0] = 1.
    return turn(f), turn(x)


class _Dem:
    """the engine's step (Hertz-DMT without adhesion, or linear friction) in torch, 64 bits"""

    def __init__(self, s):
        self.s, self.hertz = s, s["hertz"]
        self.nw, self.nf = len(s["walls"]), len(s["verts"])
        nb = self.nb = self.nw + self.nf
        z = lambda w: torch.zeros(nb, w, device="cuda", dtype=torch.float64)  # noqa: E731
        self.x, self.v = torch.cat([z(3), _t(s["pos"])]), torch.cat([z(3), _t(s["vel"])])
        self.w = torch.zeros_like(self.v)
        self.r = torch.cat([z(1)[:, 0], _t(s["radius"])])
        self.m = torch.cat([z(1)[:, 0], _t(s["mass"])])
        self.I = torch.cat([z(1)[:, 0], _t(s["inertia"])])
        sc = np.concatenate([[w[3] for w in s["walls"]], np.zeros(self.nf), s["scene"]]).astype(np.int64)
        self.sc = torch.as_tensor(sc, device="cuda")
        mt = np.concatenate([[w[3] for w in s["walls"]], np.zeros(self.nf), s["mat"]]).astype(np.int64)
        mt = torch.as_tensor(mt, device="cuda")
        self.young = _t([q["young"] for q in s["mats"]])[mt]
        self.tan = _t([q["tanPhi"] for q in s["mats"]])[mt]
        dts = s["dts"] if s["dts"] is not None else [s["dt"]]
        self.dt = _t(dts)[self.sc]
        for k, (p, ax, se, _) in enumerate(s["walls"]):
            self.x[k] = _t(p)
        self.axis = torch.tensor([w[1] for w in s["walls"]] or [0], device="cuda")
        self.sense = _t([w[2] for w in s["walls"]] or [0])
        self.verts, self.fake = _t(s["verts"]).reshape(-1, 3, 3), _t(s["fake"])
        self.L = _t(s["cell"]) if s["cell"] is not None else None
        self.g = _t(s["gravity"])
        self.skin = .1 * float(self.r[nb:].min())
        self.xl = None

    def neighbours(self):
        """pairs that can touch while no sphere moves more than the skin; old history carried"""
        nb, n = self.nb, len(self.x)
        old = None if self.xl is None else (self.key, self.real, self.H)
        self.xl = self.x.clone()
        i, j = _pairs(self.x[nb:], float(2 * self.r.max() + 2 * self.skin), self.s["cell"])
        i, j = i + nb, j + nb
        if self.s["dts"] is not None:
            k = self.sc[i] == self.sc[j]
            i, j = i[k], j[k]
        d = self.x[j] - self.x[i]
        sh = torch.zeros_like(d)
        if self.L is not None:
            sh = -torch.floor(d / self.L + .5) * self.L
        k = (d + sh).norm(dim=1) < self.r[i] + self.r[j] + 2 * self.skin
        A, B, S = [i[k]], [j[k]], [sh[k]]
        sph = torch.arange(nb, n, device="cuda")
        for q in range(self.nw):
            ax = self.s["walls"][q][1]
            k = ((self.x[nb:, ax] - self.x[q, ax]).abs() < self.r[nb:] + 2 * self.skin) & (self.sc[nb:] == self.sc[q])
            A.append(torch.full_like(sph[k], q))
            B.append(sph[k])
            S.append(torch.zeros(int(k.sum()), 3, device="cuda", dtype=torch.float64))
        for q in range(self.nf):
            v = self.verts[q]
            R = self.r[nb:, None] + 2 * self.skin
            k = ((self.x[nb:] > v.min(0).values - R) & (self.x[nb:] < v.max(0).values + R)).all(1)
            A.append(torch.full_like(sph[k], self.nw + q))
            B.append(sph[k])
            S.append(torch.zeros(int(k.sum()), 3, device="cuda", dtype=torch.float64))
        A, B, S = torch.cat(A), torch.cat(B), torch.cat(S)
        key = A * n + B
        o = torch.argsort(key)
        self.A, self.B, self.S, self.key = A[o], B[o], S[o], key[o]
        self.real = torch.zeros(len(o), dtype=torch.bool, device="cuda")
        self.H = torch.zeros(len(o), 11, device="cuda", dtype=torch.float64)  # normal, y axis, Ft, contact point
        if old is not None and len(old[0]) and len(o):
            at = torch.searchsorted(self.key, old[0]).clamp(max=len(o) - 1)
            k = (self.key[at] == old[0]) & old[1]
            self.real[at[k]] = True
            self.H[at[k]] = old[2][k]

    def geometry(self, A, B, S, real, N0):
        """normal, contact point, overlap, pA's position, velocities and radii, and whether a
        contact that is not real yet may start"""
        r1, r2 = self.r[A].clone(), self.r[B]
        x1, x2 = self.x[A], self.x[B] + S
        d = x2 - x1
        dist = d.norm(dim=1)
        uN = dist - (r1 + r2)
        nrm = d / dist.clamp(min=1e-300)[:, None]
        cp = x1 + nrm * (r1 + .5 * uN)[:, None]
        v1, w1 = self.v[A], self.w[A]
        start = uN <= 0
        wall, fac = A < self.nw, (A >= self.nw) & (A < self.nb)
        if self.nw:
            a = A.clamp(max=self.nw - 1)
            ax = self.axis[a][:, None]
            dw = (x2 - x1).gather(1, ax)[:, 0]
            e = torch.zeros_like(d).scatter_(1, ax, self.sense[a][:, None])
            nrm = _where(wall, e, nrm)
            uN = torch.where(wall, self.sense[a] * dw - r2, uN)
            cp = _where(wall, x2.scatter(1, ax, x1.gather(1, ax)), cp)
            start = torch.where(wall, dw.abs() <= r2, start)
            r1 = torch.where(wall, -r2, r1)
        if self.nf:
            f = torch.nonzero(fac)[:, 0]
            q = A[f] - self.nw
            p, pd = _closest(self.verts[q], x2[f])
            nv = x2[f] - p
            ds = nv.norm(dim=1)
            nrm, cp, uN, x1, v1, r1, start = (t.clone() for t in (nrm, cp, uN, x1, v1, r1, start))
            nrm[f] = nv / ds[:, None]
            cp[f], x1[f], uN[f], r1[f] = p, p, ds - r2[f], r2[f]
            start[f] = (pd.abs() <= r2[f]) & (ds <= r2[f])
            v1[f] = self.fake[q]
        keep = (uN <= 0) & (real | start)
        return nrm, cp, uN, x1, x2, v1, w1, r1, r2, keep

    def step(self, n):
        if self.xl is None or bool(((self.x - self.xl).norm(dim=1) > self.skin).any()):
            self.neighbours()
        g = self.geometry(self.A, self.B, self.S, self.real, self.H[:, :3])
        act = torch.nonzero(g[9])[:, 0]
        A, B = self.A[act], self.B[act]
        N1, cp, uN, x1, x2, v1, w1, r1, r2 = (t[act] for t in g[:9])
        real, H, dt = self.real[act], self.H[act], self.dt[B][:, None]
        v2, w2 = self.v[B], self.w[B]
        N0, Y0 = H[:, :3], H[:, 3:6]
        y, z = torch.zeros_like(N1), torch.zeros_like(N1)
        y[:, 1], z[:, 2] = 1., 1.
        Yn = torch.linalg.cross(N1, _where(N1[:, 1].abs() < N1[:, 2].abs(), y, z))
        Yn = _unit(Yn - N1 * _dot(Yn, N1)[:, None])
        mid = _unit(torch.where(real[:, None], .5 * (N0 + N1), N1))
        rt = torch.linalg.cross(N0, N1) + mid * dt * .5 * _dot(mid, w1 + w2)[:, None]
        M1 = Y0 - torch.linalg.cross(Y0, rt) / 2.
        M2 = torch.linalg.cross(mid, M1)
        Y = Y0 - torch.linalg.cross(M1, rt)
        if n % 100 == 0:
            Y = Y - N1 * _dot(Y, N1)[:, None]
            Y = Y / Y.norm(dim=1, keepdim=True).clamp(min=1e-300)
        mc = .5 * (H[:, 8:] + cp)
        c1, c2 = mc - (x1 - v1 * dt / 2.), mc - (x2 - v2 * dt / 2.)
        rel = v2 + torch.linalg.cross(w2, c2) - v1 - torch.linalg.cross(w1, c1)
        fresh = ~real
        Y = _where(fresh, Yn, Y)
        vel = [torch.where(real, _dot(e, rel), 0.) for e in (mid, M1, M2)]
        F1, F2 = (torch.where(real, H[:, k], 0.) for k in (6, 7))
        l0, l1, dt = r1.abs(), r2.abs(), dt[:, 0]
        tan = torch.minimum(self.tan[A], self.tan[B])
        E1, E2 = self.young[A], self.young[B]
        if self.hertz:
            nu = POISSON
            K = (4 / 3.) / ((1 - nu * nu) / E1 + (1 - nu * nu) / E2)
            R = 1. / (1. / l0 + 1. / l1)
            kn0 = K * R.sqrt()
            G = .5 * (E1 / (2 * (1 + nu)) + E2 / (2 * (1 + nu)))
            mA, mB = self.m[A], self.m[B]
            mb = torch.where(mA > 0, mA * mB / (mA + mB), mB)
            va = -math.sqrt(5) * math.log(EN) / math.sqrt(math.log(EN) ** 2 + math.pi ** 2)
            u = (-uN).clamp(min=0.)
            eta = va * (mb * kn0).sqrt() * u.sqrt().sqrt()
            Fe = -kn0 * u.sqrt() ** 3
            Fv = eta * vel[0]
            Fn = Fe + torch.where(Fe + Fv > 0, -Fe, Fv)
            kt = 2 * (4 * R).sqrt() * G / (2 - nu) * u.sqrt()
            lim = (Fn.clamp(max=0.) * tan).abs()
        else:
            kn = 1 / (1 / (E1 * self.area(r1, r2) / l0) + 1 / (E2 * self.area(r1, r2) / l1))
            kt, eta, Fn = .2 * kn, torch.zeros_like(kn), kn * uN
            lim = Fn.abs() * tan
        F1, F2 = F1 + dt * kt * vel[1], F2 + dt * kt * vel[2]
        Ft = (F1 * F1 + F2 * F2).sqrt()
        slip = Ft > lim
        q = torch.where(slip, lim / Ft.clamp(min=1e-300), 1.)
        F1 = torch.where(slip, F1 * q, F1 + eta * vel[1])
        F2 = torch.where(slip, F2 * q, F2 + eta * vel[2])
        F, ex = _rotate(N1, Y, torch.stack([Fn, F1, F2], 1))
        self.real = torch.zeros_like(self.real)
        self.real[act] = True
        self.H[act] = torch.cat([N1, Y, F1[:, None], F2[:, None], cp], 1)
        self.last = (A, B, F, cp, uN, ex, kt, (1.5 * kn0 * u.sqrt()) if self.hertz else Fn / uN, l0, l1)
        f = self.m[:, None] * self.g * (n > 0)  # gravity is set by the reset that ends a step
        t = torch.zeros_like(f)
        f.index_add_(0, A, F)
        f.index_add_(0, B, -F)
        t.index_add_(0, A, torch.linalg.cross(cp - self.x[A], F))
        t.index_add_(0, B, torch.linalg.cross(cp - x2, -F))
        self.integrate(f, t)

    @staticmethod
    def area(r1, r2):
        return math.pi * torch.where(r1 > 0, torch.minimum(r1, r2), r2) ** 2

    def integrate(self, f, t):
        nb, c = self.nb, self.s["damping"]
        dt = self.dt[nb:, None]
        self.xForce = self.x.clone()  # positions the contacts were evaluated at
        for a, b, q in ((f, self.v, self.m), (t, self.w, self.I)):
            acc = a[nb:] / q[nb:, None]
            if c:
                acc = acc * (1 - c * torch.sign(a[nb:] * (b[nb:] + .5 * dt * acc)))
            b[nb:] += dt * acc
        self.x[nb:] += self.v[nb:] * dt

    def nodes(self):
        """the last step's facet contact forces spread to the facets' nodes"""
        A, B, F, cp = self.last[:4]
        k = (A >= self.nw) & (A < self.nb)
        q, F, cp = A[k] - self.nw, F[k], cp[k]
        v = self.verts[q]
        b, c = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
        nu = _unit(torch.linalg.cross(b, c))
        d = cp - nu * _dot(cp - v[:, 0], nu)[:, None] - v[:, 0]
        bb, bc, cc, db, dc = _dot(b, b), _dot(b, c), _dot(c, c), _dot(d, b), _dot(d, c)
        det = bb * cc - bc * bc
        u, w = (cc * db - bc * dc) / det, (bb * dc - bc * db) / det
        fo = torch.zeros(self.nf, 3, 3, device="cuda", dtype=torch.float64)
        to = torch.zeros_like(fo)
        for i, wt in enumerate((1 - u - w, u, w)):
            Fi = F * wt[:, None]
            fo[:, i].index_add_(0, q, Fi)
            to[:, i].index_add_(0, q, torch.linalg.cross(cp - v[:, i], Fi))
        return fo, to


def _observe(D):
    """coordination, solid fraction, stress, kinetic energy, critical timestep of the state"""
    A, B, F, cp, uN, N1, kt, kn, l0, l1 = D.last
    n = len(D.x)
    one = torch.ones_like(uN)
    cnt = torch.zeros(n, device="cuda", dtype=torch.float64).index_add_(0, A, one).index_add_(0, B, one)
    C2, n0, n1 = cnt.sum(), (cnt == 0).sum(), (cnt == 1).sum()
    box = ((D.x >= .25 * D.L) & (D.x <= .75 * D.L)).all(1)
    vs = (4 / 3. * math.pi * D.r[box] ** 3).sum()
    ob = torch.stack([C2 / n, (C2 - n1) / (n - n0 - n1), vs / (.5 * D.L).prod()])
    S = D.S[torch.searchsorted(D.key, A * n + B)]
    d0 = (D.x[B] + S - D.x[A]).norm(dim=1)
    fN = _dot(F, N1)
    fT = F - N1 * fN[:, None]
    o = lambda a, b: a[:, :, None] * b[:, None, :]  # noqa: E731
    st = (d0[:, None, None] * (fN[:, None, None] * o(N1, N1) + .5 * (o(fT, N1) + o(N1, fT)))).sum(0) / D.L.prod()
    ek = .5 * (D.m * _dot(D.v, D.v)).sum() + .5 * (D.I * _dot(D.w, D.w)).sum()
    n2 = N1 * N1
    K = torch.zeros(n, 3, device="cuda", dtype=torch.float64)
    Kr = torch.zeros_like(K)
    for p, l in ((A, l0), (B, l1)):
        K.index_add_(0, p, n2 * (kn - kt)[:, None] + kt[:, None])
        Kr.index_add_(0, p, (l * l * kt)[:, None] * (n2.sum(1, keepdim=True) - n2)[:, [0, 1, 2]])
    q = torch.cat([(D.m[:, None] / K)[K > 0], (D.I[:, None] / Kr)[Kr > 0]])
    return dict(observables=ob, stress=st, kinetic=ek, critDt=(2 * q.min()).sqrt())


class _Net:
    """the message-passing network in torch, 64 bits"""

    def __init__(self, p, grad=False):
        self.p, o = [], 0
        for K, O in ((32, 64), (160, 64), (128, 64), (160, 64), (128, 64), (64, 3)):
            w = _t(p[o:o + K * O].reshape(K, O).astype(np.float64))
            b = _t(p[o + K * O:o + K * O + O].astype(np.float64))
            o += K * O + O
            self.p += [w.requires_grad_(grad), b.requires_grad_(grad)]

    def graph(self, x, v, r):
        i, j = _pairs(x, 1.1 * 2 * float(r.max()))
        k = (x[i] - x[j]).square().sum(1) < (1.1 * (r[i] + r[j])) ** 2
        i, j = torch.cat([i[k], j[k]]), torch.cat([j[k], i[k]])
        rs = r[i] + r[j]
        d = (x[j] - x[i]) / rs[:, None]
        dn = d.norm(dim=1)
        ov = (1 - dn) * 100.
        w = (v[j] - v[i]) / V0
        a, b = r[i] / R0, r[j] / R0
        nrm = d / dn[:, None]
        op = ov.clamp(min=0.)
        a3, b3 = a ** 3, b ** 3
        hz = op ** 1.5 * ((a * b).sqrt() * (a + b) / a3)
        mb, Rb = a3 * b3 / (a3 + b3), a * b / (a + b)
        dp = _dot(w, nrm) * op ** .25 * ((a + b) ** .25 * (mb * Rb.sqrt()).sqrt() / a3)
        E = torch.cat([d, ov.clamp(-2., 2.)[:, None], w, a[:, None], b[:, None], -nrm * hz[:, None],
                       nrm * dp[:, None], torch.zeros(len(i), 17, device="cuda", dtype=torch.float64)], 1)
        a = r / R0
        ov = (1 - x[:, 2] / r) * 100.
        op = ov.clamp(min=0.)
        X = torch.cat([v / V0, torch.stack([a, ov.clamp(-2., 2.), op ** 1.5 / a, v[:, 2] / V0 * op ** .25 / a], 1),
                       torch.zeros(len(r), 25, device="cuda", dtype=torch.float64)], 1)
        touch = (ov > 0).index_put((i[E[:, 3] > 0],), torch.tensor(True, device="cuda"))
        return X, E, i, j, touch

    def __call__(self, X, E, i, j, touch):
        p = self.p
        h = torch.relu(X @ p[0] + p[1])
        for k in (2, 6):
            m = torch.relu(h[i] @ p[k][:64] + h[j] @ p[k][64:128] + E @ p[k][128:] + p[k + 1])
            s = torch.zeros_like(h).index_add(0, i, m)
            h = h + torch.relu(h @ p[k + 2][:64] + s @ p[k + 2][64:] + p[k + 3])
        return h @ p[10] + p[11]


def _num(d):
    return {k: (v.detach() if torch.is_tensor(v) else v) for k, v in d.items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "pack":
        rng = np.random.default_rng([seed, 3])
        n = case["n"]
        radius = rng.uniform(2e-3, 4e-3, n)
        L = (float(np.sum(4 / 3. * math.pi * radius ** 3)) / .55) ** (1 / 3.)
        x, r, ov, xl = _t(rng.uniform(0., L, (n, 3))), _t(radius) * 1.005, 0., None
        skin = .2 * float(r.min())
        for _ in range(SWEEPS):
            if xl is None or bool(((x - xl).norm(dim=1) > skin).any()):
                i, j = _pairs(x, float(2 * r.max()) + 2 * skin, (L,) * 3)
                sh = -torch.floor((x[j] - x[i]) / L + .5) * L
                xl = x.clone()
            d = x[j] + sh - x[i]
            dist = d.norm(dim=1)
            o = (r[i] + r[j] - dist).clamp(min=0.)
            push = d * (.5 * o / dist)[:, None]
            ov = float(o.max())
            x = x.index_add(0, i, -push).index_add(0, j, push)
        return dict(pos=x, overlap=ov)
    if kind in ("learned", "forward", "train"):
        arr = _column(case, seed)
        x, v, r = _t(arr["pos"][1:]), _t(arr["vel"][1:]), _t(arr["radius"][1:])
        net = _Net(_params(seed), grad=kind == "train")
        if kind == "learned":
            dt = COARSE * surrogate.dem_dt()
            for _ in range(COARSE_STEPS):
                g = net.graph(x, v, r)
                a = _where(g[4], net(*g) * A0, _t([[0., 0., -9.81]]).expand(len(x), 3))
                v = v + a * dt
                x = x + v * dt
            z = torch.zeros(1, 3, device="cuda", dtype=torch.float64)
            return dict(pos=torch.cat([z, x]), vel=torch.cat([z, v]))
        g = net.graph(x, v, r)
        if kind == "forward":
            return net(*g) * A0
        d = (net(*g) - _t(_targets(len(x), seed) / A0)) * g[4][:, None]
        loss = d.square().sum() / len(x)
        grads = torch.autograd.grad(loss, net.p)
        return dict(loss=float(loss.detach()), grads=torch.cat([q.reshape(-1) for q in grads]))
    D = _Dem(_scene(case, seed))
    if kind == "fp32":
        for k in range(STEPS[kind]):
            D.step(k)
        return dict(pos=D.x, vel=D.v)
    for k in range(WARM):
        D.step(k)
    if kind == "observe":
        return _num(_observe(D))
    for k in range(STEPS[kind]):
        D.step(WARM + k)
    out = dict(pos=D.x, vel=D.v)
    if kind == "engines":
        out["kinetic"] = float(.5 * (D.m * _dot(D.v, D.v)).sum() + .5 * (D.I * _dot(D.w, D.w)).sum())
    if kind == "drum":
        # (a facet's position is its first vertex)
        out["pos"] = D.x.clone()
        out["pos"][D.nw:D.nb] = D.verts[:, 0]
        out["nodeForce"], out["nodeTorque"] = D.nodes()
    return _num(out)
