"""Kernels at the sizes where their tiling and reductions can go wrong: one workgroup, ragged last
workgroups, and the smallest and largest of what each launch covers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 65, 1500, 9000])
def test_relax_reports_the_largest_overlap(n):
    # one sweep reports the largest overlap of the inflated radii before it moves anything
    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    radius = rng.uniform(2e-3, 4e-3, n)
    L = (float(np.sum(4 / 3. * np.pi * radius ** 3)) / .5) ** (1 / 3.) if n > 2 else 0.02
    pos = rng.uniform(0., L, (n, 3))
    if n == 2:
        pos[1] = pos[0] + (3e-3, 0., 0.)
    d = Device(0)
    d.set_field(periodic=True, cell=(max(L, .04),) * 3)
    d.set_materials([dict(kind=0, density=1., young=1., ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=radius, mass=np.ones(n),
                       inertia=np.ones((n, 3)), vel=np.zeros((n, 3)))
    ov, it = d.relax(1, .01, tol=0.)
    cell = max(L, .04)
    best = 0.
    for k in range(0, n, 500):
        dx = pos[k:k + 500, None] - pos[None]
        dx -= cell * np.round(dx / cell)
        o = 1.01 * (radius[k:k + 500, None] + radius[None]) - np.sqrt(np.sum(dx * dx, -1))
        o[np.arange(len(o)), k + np.arange(len(o))] = 0.
        best = max(best, float(o.max()))
    assert it == 1
    # the same operations in another order: a few ulps of the cell edge
    assert abs(ov - best) <= 16 * np.finfo(float).eps * cell


@pytest.mark.parametrize("n,fill,periodic", [(513, .3, True), (2049, .3, False), (4100, .5, True), (3000, 1e-3, True),
                                              (3000, 2e-6, True), (3000, 1e-5, False)])
def test_pair_set_over_cells_per_sphere(n, fill, periodic):
    # dense cells (ordered by counting), a few cells per sphere, and far more cells than spheres
    # (ordered by sorting, or hashed): the potential pairs are those of an all-pairs test, and a
    # second refresh of the same positions keeps them
    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    r = rng.uniform(2e-3, 3e-3, n)
    L = (float(np.sum(4 / 3. * np.pi * r ** 3)) / fill) ** (1 / 3.)
    pos = rng.uniform(0., L, (n, 3))
    # half of the spheres close to another, so that sparse scenes have pairs too
    pos[1::2] = pos[0::2][:len(pos[1::2])] + rng.normal(0., 2e-3, (len(pos[1::2]), 3))
    d = Device(0)
    d.set_field(periodic=periodic, cell=(L,) * 3)
    d.set_materials([dict(kind=0, density=1., young=1., ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=r, mass=np.ones(n),
                       inertia=np.ones((n, 3)), vel=np.zeros((n, 3)))
    vd = .05 * float(r.min())
    want = set()
    for k in range(0, n, 500):
        dx = pos[k:k + 500, None] - pos[None]
        if periodic:
            dx -= L * np.round(dx / L)
        hit = np.all(np.abs(dx) <= (r[k:k + 500, None] + r[None] + 2 * vd)[..., None], axis=-1)
        i, j = np.nonzero(hit)
        want |= {(a + k, b) for a, b in zip(i.tolist(), j.tolist()) if a + k < b}
    for _ in range(2):
        d.collide(-.05, forceInit=True)
        ids = d.contacts(real_only=False, data=False)[0]
        assert {(min(a, b), max(a, b)) for a, b in ids.tolist()} == want
    np.testing.assert_array_equal(d.get("pos"), pos)


@pytest.mark.parametrize("n", [3, 511, 512, 39999, 40001, 100001])
def test_pairs_over_lanes_per_sphere(n):
    # the pair pass's lanes per sphere change with the size; the real contacts of a jittered lattice
    # are those found cell by cell on the host
    from scipy.spatial import cKDTree

    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3.)))
    pos = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 2e-3
    pos = pos + rng.uniform(-1e-4, 1e-4, pos.shape)
    r = rng.uniform(.9e-3, 1.05e-3, n)
    mass = 1e-5 * np.ones(n)
    d = Device(0)
    d.set_field(periodic=False)
    d.set_materials([dict(kind=0, density=1., young=1e6, ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=r, mass=mass,
                       inertia=np.repeat((.4 * mass * r * r)[:, None], 3, 1), vel=np.zeros((n, 3)))
    d.collide(-.05)
    d.contact_loop(0, 1e-7)
    got = d.contacts(real_only=True, data=False)[0]
    p = cKDTree(pos).query_pairs(2.2e-3, output_type="ndarray")
    p = p[np.linalg.norm(pos[p[:, 0]] - pos[p[:, 1]], axis=1) < r[p[:, 0]] + r[p[:, 1]]]
    want = np.sort(p, axis=1)
    assert len(want) > n // 4 or n == 3
    np.testing.assert_array_equal(np.sort(got, axis=1), want[np.lexsort((want[:, 1], want[:, 0]))])


@pytest.mark.parametrize("n", [60, 700, 41000, 100001])
def test_forces_where_pairs_outnumber_the_staging(n):
    # a sphere with more pairs than are staged: its slots are generated again in place, in whatever
    # order, and every sphere still sums its own contacts
    from scipy.spatial import cKDTree

    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3.)))
    pos = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 2.3e-3
    pos = pos + rng.uniform(-1e-4, 1e-4, pos.shape)
    pos[:45] = pos[n // 2] + rng.uniform(-.6e-3, .6e-3, (45, 3))  # 44 neighbours each
    r = rng.uniform(.95e-3, 1.05e-3, n)
    d = Device(0)
    d.set_field(periodic=False)
    E = 1e6
    d.set_materials([dict(kind=0, density=1., young=E, ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=r, mass=np.ones(n), inertia=np.ones((n, 3)),
                       vel=np.zeros((n, 3)))
    d.collide(-.05)
    d.contact_loop(0, 1e-9)
    got = d.get("force")
    i, j = cKDTree(pos).query_pairs(2.2e-3, output_type="ndarray").T
    x = pos[j] - pos[i]
    dist = np.linalg.norm(x, axis=1)
    k = dist < r[i] + r[j]
    i, j, x, dist = i[k], j[k], x[k], dist[k]
    A = np.pi * np.minimum(r[i], r[j]) ** 2
    F = (1 / (1 / (E * A / r[i]) + 1 / (E * A / r[j])) * (dist - r[i] - r[j]) / dist)[:, None] * x
    want, size = np.zeros((n, 3)), np.zeros((n, 3))
    for s, e in ((1., i), (-1., j)):
        np.add.at(want, e, s * F)
        np.add.at(size, e, np.abs(F))
    # a few dozen roundings per term, the overlap's cancellation in uN included
    assert np.all(np.abs(got - want) <= 1e-12 * (size + size.max()))


@pytest.mark.parametrize("n", [2, 255, 257, 5000, 262145 + 300])
@pytest.mark.parametrize("stepped", [False, True])
def test_observables_over_workgroups(n, stepped):
    # one workgroup, ragged ones, and more workgroups than one pass of the last reduction takes; the
    # contacts straight from the refresh, and after steps
    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3.)))
    pos = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] * 2e-3
    r = rng.uniform(.95e-3, 1.05e-3, n)
    r[0] = r[n - 1] = 1.05e-3
    mass = rng.uniform(1e-5, 2e-5, n)
    vel = rng.normal(0., 1e-4, (n, 3))
    E, kdk = 1e6, .2
    d = Device(0)
    d.set_field(periodic=False)
    d.set_materials([dict(kind=0, density=1., young=E, ktDivKn=kdk, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=pos, radius=r, mass=mass,
                       inertia=np.repeat((.4 * mass * r * r)[:, None], 3, 1), vel=vel)
    d.collide(-.05)
    d.contact_loop(0, 1e-9)
    if stepped:
        d.leapfrog(1e-9)
        d.contact_loop(1, 1e-9)
    pos, vel = d.get("pos"), d.get("vel")
    ids = d.contacts(real_only=True, data=False)[0]
    assert len(ids)
    cnt = np.bincount(ids.reshape(-1), minlength=n)
    o = d.observables((-1., -1., -1.), (1., 1., 1.))
    n0, n1 = np.sum(cnt == 0), np.sum(cnt == 1)
    assert o["coordNumber"] == cnt.sum() / n
    if n > n0 + n1:
        assert o["coordNumberSkipFree"] == (cnt.sum() - n1) / (n - n0 - n1)
    eps = np.finfo(float).eps
    # sums of n terms of one sign over 256-wide trees and a 1,024-wide last stage
    tol = 32 * eps
    assert abs(o["solidFraction"] / (np.sum(4 / 3. * np.pi * r ** 3) / 8.) - 1) <= tol
    ek = np.sum(.5 * mass * np.sum(vel ** 2, 1)) + np.sum(.5 * .4 * mass * r * r * np.sum(d.get("angVel") ** 2, 1))
    assert abs(d.kinetic_energy() / ek - 1) <= tol
    # the stiffness of every particle, a few dozen roundings per contact term
    i, j = ids.T
    kn = 1 / (1 / (E * np.pi * np.minimum(r[i], r[j]) ** 2 / r[i]) + 1 / (E * np.pi * np.minimum(r[i], r[j]) ** 2 / r[j]))
    nn = pos[j] - pos[i]
    n2 = (nn / np.linalg.norm(nn, axis=1)[:, None]) ** 2
    kt, kr = np.zeros((n, 3)), np.zeros((n, 3))
    for e in (i, j):
        np.add.at(kt, e, n2 * (kn * (1 - kdk))[:, None] + (kdk * kn)[:, None])
        np.add.at(kr, e, (r[e] ** 2 * kdk * kn)[:, None] * (1 - n2))
    with np.errstate(divide="ignore"):
        crit = np.sqrt(2 * min(np.min(mass[:, None] / kt), np.min((.4 * mass * r * r)[:, None] / kr)))
    assert abs(d.crit_dt() / crit - 1) <= 64 * eps


@pytest.mark.parametrize("n", [1, 2, 511, 4095, 4096, 4097, 9000])
def test_long_lists_of_a_floor(n):
    # a floor's list sorted by one workgroup up to 4,096 entries, by the radix sort above; the force on
    # the floor is summed in that order whichever way it was sorted, and is that of the engine's
    # unsorted contacts up to rounding
    from woo_amd._native import SPHERE, WALL, Device

    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** .5))
    r = 1e-3
    xy = (np.stack(np.meshgrid(np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 2)[:n] + .5) * 2.3e-3
    z = rng.uniform(.97, .99, n) * r
    pos = np.column_stack([xy, z])[rng.permutation(n)]
    wall = np.zeros((1, 3))
    d = Device(0)
    d.set_field(periodic=False)
    E = 1e6
    d.set_materials([dict(kind=0, density=1., young=E, ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.array([WALL] + [SPHERE] * n, np.int32), pos=np.vstack([wall, pos]),
                       radius=np.r_[0., np.full(n, r)], mass=np.ones(n + 1), inertia=np.ones((n + 1, 3)),
                       vel=np.zeros((n + 1, 3)), wallAxis=np.r_[2, np.zeros(n)].astype(np.int32))
    out = []
    for _ in range(2):
        d.force_reset()
        d.collide(-.05, forceInit=True)
        d.contact_loop(0, 1e-9)
        out.append(d.get("force"))
    np.testing.assert_array_equal(out[0], out[1])
    F = E * np.pi * r * (pos[:, 2] - r) / 2.  # two equal lengths in series
    assert abs(out[0][0, 2] - F.sum()) <= 1e-12 * np.abs(F).sum() * (r / np.abs(pos[:, 2] - r).min())


@pytest.mark.parametrize("n", [1, 32768, 32769, 43690, 43691])
def test_fields_to_and_from_the_host(n):
    # rows through pinned memory and directly, on both sides of the size where the way changes; the
    # storage order differs from the user's after a refresh
    from woo_amd._native import SPHERE, Device

    rng = np.random.default_rng(n)
    d = Device(0)
    d.set_field(periodic=True, cell=(1., 1., 1.))
    d.set_materials([dict(kind=0, density=1., young=1., ktDivKn=.2, tanPhi=.5, surfEnergy=0., alpha=0.)])
    d.upload_particles(shape=np.full(n, SPHERE, np.int32), pos=rng.uniform(0., 1., (n, 3)), radius=np.full(n, 1e-3),
                       mass=np.ones(n), inertia=np.ones((n, 3)), vel=np.zeros((n, 3)))
    d.collide(-.05)
    sent = {}
    for f, w in (("vel", 3), ("ori", 4), ("mass", 1), ("inertia", 3), ("angVel", 3)):
        sent[f] = rng.uniform(.5, 1., (n, w) if w > 1 else n)
        d.set(f, sent[f])
    d.collide(-.05, forceInit=True)
    for f, a in sent.items():
        np.testing.assert_array_equal(d.get(f), a, err_msg=f)


@pytest.mark.parametrize("n,flat,steps", [(20, False, 1), (300, False, 7), (300, False, 130), (4900, True, 40)])
@pytest.mark.parametrize("track", [False, True])
def test_steps_ahead_equal_engine_calls(n, flat, steps, track):
    # wdg_run's batches of gated steps against the engines called one by one: short wall lists (summed
    # in the leapfrog) and a floor with more than 2,048 contacts (cut into parts), several refreshes
    from tests.scenes import GpuRunner, contact_kw, deposition

    sc = deposition(n=n, seed=n, dense=True, vel_sigma=.3)
    if flat:  # one layer on the floor, slightly in contact with it
        m = int(round(n ** .5))
        r = sc["radius"][0]
        g = np.stack(np.meshgrid(np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 2)
        sc["pos"] = np.column_stack([(g + .5) * 2.01 * r, np.full(len(g), .999 * r)])
        for w in sc["walls"][3:]:
            w["pos"][w["axis"]] = 2.01 * r * m
    a, b = GpuRunner(sc), GpuRunner(sc)
    eng = ["Collider", "ContactLoop", "Leapfrog"]
    if track:
        a.d.set_energy_tracking(True)
        b.d.set_energy_tracking(True)
    a.run(eng, steps)
    b.d.run(eng, steps, 0, sc["dt"], contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0)
    for f in ("pos", "vel", "angVel", "ori", "force", "torque"):
        np.testing.assert_array_equal(a.d.get(f), b.d.get(f), err_msg=f)
    np.testing.assert_array_equal(a.d.contacts(data=False)[0], b.d.contacts(data=False)[0])
    sa, sb = a.d.stats(), b.d.stats()
    assert sa["nSteps"] == sb["nSteps"] and sa["nRefresh"] == sb["nRefresh"]
    if flat:
        assert sa["nCandidates"] > 2 * 2048
    if track:  # every term, by the same sums of the same steps; skipped steps add nothing
        ea, eb = a.d.energy(), b.d.energy()
        assert ea == eb and ea["kinetic"] > 0 and (steps == 1 or ea["plast"] > 0)


@pytest.mark.parametrize("track", [False, True])
def test_steps_ahead_with_facet_nodes(track):
    # the list with IntraForce: the forces on the facets' nodes are those of the last step that ran
    from tests.scenes import GpuRunner, contact_kw, drum

    sc = drum(n=1500, vel_sigma=.3)
    a, b = GpuRunner(sc), GpuRunner(sc)
    eng = ["Collider", "ContactLoop", "IntraForce", "Leapfrog"]
    ids = np.arange(len(sc["walls"]), len(sc["walls"]) + len(sc["facets"]))
    for g in (a, b):
        g.d.set_energy_tracking(track)
    st = 0
    for steps in (1, 7, 60):
        a.run(eng, steps)
        st, _ = b.d.run(eng, steps, st, sc["dt"], contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]),
                        dynDtPeriod=0)
        na, nb = np.array(a.d.facet_nodes(ids)), np.array(b.d.facet_nodes(ids))
        assert np.any(na)
        np.testing.assert_array_equal(na, nb)
        for f in ("pos", "vel", "angVel", "force", "torque"):
            np.testing.assert_array_equal(a.d.get(f), b.d.get(f), err_msg=f)
    assert a.d.stats()["nRefresh"] == b.d.stats()["nRefresh"] > 2
    if track:
        assert a.d.energy() == b.d.energy()


@pytest.mark.parametrize("n,walls", [(300, False), (5000, False), (5000, True)])
def test_contacts_pulled_out_of_reach(n, walls):
    # real contacts that are no near pairs at a refresh are appended behind the new pairs, and the real set
    # and the adjacency made again with them: they persist (noBreak) and pull as in the oracle
    from tests.scenes import build_gpu, build_oracle, contact_kw, deposition

    sc = deposition(n=n, seed=n, dense=True, vel_sigma=.02)
    sc["walls"] = [w for w in sc["walls"] if walls and (w["axis"], w["sense"]) != (0, -1)]
    sc["gravity"] = (0., 0., 0.)
    eng = ["Collider", "ContactLoop", "Leapfrog"]
    o, d = build_oracle(sc, noBreak=1), build_gpu(sc)
    kw = dict(contact=dict(contact_kw(sc), noBreak=1), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0)
    st, _ = d.run(eng, 6, 0, sc["dt"], **kw)
    o.run(eng, 6)
    ids = d.contacts(real_only=True, data=False)[0]
    pos = d.get("pos")
    right = np.arange(len(pos)) < n  # spheres come before walls
    right &= pos[:, 0] > sc["box"] / 2
    pos[right, 0] += 3 * sc["radius"][0]
    d.set("pos", pos)
    o.set("pos", pos)
    far = np.sum(right[ids[:, 0]] != right[ids[:, 1]])
    assert far > n ** (2 / 3.) / 2
    d.collide(-.05)
    np.testing.assert_array_equal(d.contacts(real_only=True, data=False)[0], ids)
    for steps in (1, 20):
        st, _ = d.run(eng, steps, st, sc["dt"], **kw)
        o.run(eng, steps)
        np.testing.assert_array_equal(d.contacts(real_only=True, data=False)[0], o.contacts(real_only=True, data=False)[0])
        for f in ("pos", "vel", "angVel", "ori"):
            np.testing.assert_array_equal(d.get(f), o.get(f), err_msg=f)


def _network_graph(rng, N, kind):
    # both directions of every pair, by receiver; "hub": node 0 exchanges with everyone; "double":
    # pairs twice, with opposite edges that are not each other's opposite
    pairs = {(i, (i + d) % N) for i in range(N) for d in (1, 2, 5) if (i + d) % N != i} if N > 1 else set()
    pairs = {(min(p), max(p)) for p in pairs if rng.random() < .7}
    if kind == "hub":
        pairs |= {(0, j) for j in range(1, N)}
    p = np.array(sorted(pairs), dtype=np.int64).reshape(-1, 2)
    if kind == "double":
        p = np.repeat(p, 2, axis=0)
    n = len(p)
    recv, send = np.concatenate([p[:, 0], p[:, 1]]), np.concatenate([p[:, 1], p[:, 0]])
    back = np.concatenate([np.arange(n) + n, np.arange(n)])
    if kind == "double":  # the second half's opposites are swapped within each pair of edges
        back[n:] = back[n:] ^ 1
    o = np.argsort(recv, kind="stable")
    at = np.empty(2 * n, dtype=np.int64)
    at[o] = np.arange(2 * n)
    return (np.concatenate([[0], np.cumsum(np.bincount(recv, minlength=N))]), send[o], at[back[o]],
            rng.normal(size=(N, 7)), rng.normal(size=(2 * n, 15)), rng.normal(size=(N, 3)))


@pytest.mark.parametrize("N,kind", [(1, ""), (2, ""), (16, ""), (17, "hub"), (70, "hub"), (63, "double"), (2100, "")])
def test_network_at_tile_edges(N, kind):
    # partly filled wavefronts, nodes without edges and with more than a tile of them, a caller's graph
    # whose rev is not an involution
    from oracle.mpnn import Net, layout
    from tests.test_mpnn_oracle import random_params
    from woo_amd.surrogate import A0, Graph, Network

    f32 = lambda a: np.asarray(a, dtype=np.float32).astype(np.float64)
    rng = np.random.default_rng(100 + N)
    rowOff, send, rev, x, ef, t = _network_graph(rng, N, kind)
    p, x, ef, t = (f32(q) for q in (random_params(rng), x, ef, t))
    x[:, 4] = np.where(np.arange(N) % 3 == 0, -1., x[:, 4])
    net = Network(seed=1)
    net.set_params(p)
    g = Graph(rowOff, send, rev, x, ef)
    out = net.predict(g) / A0
    ref = Net(p, emulate=True)
    a_cpu, _ = ref.forward(x, rowOff, send, ef)
    # activations round to BF16 between the layers: values on a rounding boundary differ by 2^-8
    assert np.max(np.abs(out - a_cpu)) <= 1e-2 * np.max(np.abs(a_cpu))
    loss = net.loss_grad(g, t * A0)
    grad = net.grads().astype(np.float64)
    loss_cpu, grad_cpu = ref.loss_grad(x, rowOff, send, rev, ef, t)
    assert abs(loss - loss_cpu) <= 1e-2 * loss_cpu
    for name, (o, s) in layout()[0].items():
        a, b = grad[o:o + s], grad_cpu[o:o + s]
        assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b), name


def test_network_keeps_an_overflow_to_its_neighbours():
    # a node whose messages overflow changes no output beyond the two rounds of messages
    from tests.test_mpnn_oracle import random_params
    from woo_amd.surrogate import Graph, Network

    rng = np.random.default_rng(5)
    N = 40
    e = np.array([(i, j) for i in range(N) for j in (i - 1, i + 1) if 0 <= j < N])
    rowOff = np.concatenate([[0], np.cumsum(np.bincount(e[:, 0], minlength=N))])
    rev = np.array([np.flatnonzero((e[:, 0] == j) & (e[:, 1] == i))[0] for i, j in e])
    x, ef = rng.normal(size=(N, 7)), rng.normal(size=(len(e), 15))
    net = Network(seed=1)
    net.set_params(np.asarray(random_params(rng), dtype=np.float32))
    a = net.predict(Graph(rowOff, e[:, 1], rev, x, ef))
    x[5] = 3e38 * np.sign(x[5])
    b = net.predict(Graph(rowOff, e[:, 1], rev, x, ef))
    far = np.abs(np.arange(N) - 5) > 2
    np.testing.assert_array_equal(a[far], b[far])
    assert not np.all(np.isfinite(b[~far])) or np.any(np.abs(b[~far]) > 1e30)


# needle triangles whose vertices are collinear up to rounding: near them the signs of the three edge
# tests are rounding noise, and about a fifth of the positions lie outside all three edges
NEEDLES = {64: ((-0.11411671584340066, -0.08510797192370884, -0.015578443378596867),
                (-0.04603145941331931, -0.03433015160313763, -0.00628390397326742)),
           32: ((-0.09294396638870239, 0.07020442187786102, -0.024254076182842255),
                (-0.06973002105951309, 0.05266996845602989, -0.018196310847997665))}


def needle_scene(bits, n=8000, far=3.5e-3):
    # a bed of several groups of slots, and spheres that come within reach of a needle after some steps
    from tests.scenes import deposition

    sc = deposition(n=n, seed=3, r=2e-3, dense=True, vel_sigma=.05)
    r = sc["radius"][0]
    v = np.array([(0., 0., 0.), *NEEDLES[bits]])
    # the normal as this precision computes it: rounding noise, so not at right angles to the edges
    nn = np.cross(*v[1:].astype(np.float64 if bits == 64 else np.float32)).astype(np.float64)
    nn /= np.linalg.norm(nn)
    t = np.arange(.1, .95, 2.2 * r / np.linalg.norm(v[1]))
    k = len(t)
    sc["pos"] = np.vstack([sc["pos"], t[:, None] * v[1] + ((1 + far) * r - t * (v[1] @ nn))[:, None] * nn])
    sc["vel"] = np.vstack([sc["vel"], np.repeat(-1e-3 * r / sc["dt"] * nn[None], k, 0)])
    for q in ("radius", "mass", "inertia"):
        sc[q] = np.concatenate([sc[q], np.repeat(sc[q][:1], k, 0)])
    sc.update(facets=[dict(verts=v)], walls=[], gravity=(0., 0., 0.))
    return sc


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("graph", [False, True])
def test_an_error_ends_a_batch_after_its_step(bits, graph):
    # the filter itself raises an error (a sphere outside all edges of a needle facet): its step runs to
    # the end on every workgroup, the next one on none, as when the engines are called one by one
    from tests.scenes import GpuRunner, contact_kw

    sc = needle_scene(bits)
    a, b = GpuRunner(sc), GpuRunner(sc)
    for d in (a.d, b.d):
        d.set_precision(bits)
    with pytest.raises(Exception, match="impossible sphere-facet"):
        a.run(["Collider", "ContactLoop", "Leapfrog"], 32)
    assert 2 < a.step < 16
    with pytest.raises(Exception, match="impossible sphere-facet"):
        b.d.run(["Collider", "ContactLoop", "Leapfrog"], 32, 0, sc["dt"], contact=contact_kw(sc),
                leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0, graph=graph)
    assert a.d.stats()["nCandidates"] > 10 * 2048
    for f in ("pos", "vel", "angVel", "ori", "force", "torque"):
        np.testing.assert_array_equal(a.d.get(f), b.d.get(f), err_msg=f)
    np.testing.assert_array_equal(a.d.contacts(data=False)[0], b.d.contacts(data=False)[0])


@pytest.mark.parametrize("how", ["collide", "sync", "run"])
def test_an_error_is_reported_once(how):
    # whichever call reports a step's error, the collider's next call goes on
    from tests.scenes import GpuRunner, contact_kw

    sc = needle_scene(64)
    g = GpuRunner(sc)
    eng = ["Collider", "ContactLoop", "Leapfrog"]
    if how == "run":
        report = lambda: g.d.run(eng, 32, 0, sc["dt"], contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]),
                                 dynDtPeriod=0)
    else:
        g.run(eng, 5)
        report = (lambda: g.d.collide(g.vd)) if how == "collide" else g.d.sync
    with pytest.raises(Exception, match="impossible sphere-facet"):
        report()
    g.d.collide(g.vd)
    g.d.sync()


@pytest.mark.parametrize("n,periodic", [(20, False), (300, False), (1500, True)])
def test_steps_in_calls_of_any_length(n, periodic):
    # calls of a few steps (launched one after the other) and of more (launched ahead) mixed: the same
    # steps, refreshes and states as one call for all
    from tests.scenes import build_gpu, contact_kw, deposition, periodic_hertz

    sc = periodic_hertz(n=n, spacing=.95, vel_sigma=2.) if periodic else deposition(n=n, seed=n, dense=True, vel_sigma=.3)
    kw = dict(contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0)
    eng = ["Collider", "ContactLoop", "Leapfrog"]
    a, b = build_gpu(sc), build_gpu(sc)
    calls = [1, 1, 2, 3, 4, 5, 6, 1, 9, 4, 17, 1, 2]
    a.run(eng, sum(calls), 0, sc["dt"], **kw)
    st = 0
    for k in calls:
        st, _ = b.run(eng, k, st, sc["dt"], **kw)
    assert st == sum(calls)
    for f in ("pos", "vel", "angVel", "ori", "force", "torque"):
        np.testing.assert_array_equal(a.get(f), b.get(f), err_msg=f)
    sa, sb = a.stats(), b.stats()
    assert sa["nSteps"] == sb["nSteps"] and sa["nRefresh"] == sb["nRefresh"] > 1
