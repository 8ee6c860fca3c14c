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
