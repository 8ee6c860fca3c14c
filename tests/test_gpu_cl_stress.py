"""ContactLoop.evalStress / ContactLoop.stress (ContactLoop.cpp:117,123,216-229,243-244) on the
HIP engine against the oracle: in a periodic cell each contact loop sums F branch^T over its
real contacts and divides by the cell volume. The sums run in another order than the oracle's,
so the bar is 1e-10 of the largest component; the oracle itself is pinned by DemFuncs' stress
(the symmetric part) and the contact torques (the antisymmetric part)."""
import numpy as np
import pytest

from tests.scenes import build_gpu, build_oracle, contact_kw, deposition, periodic_hertz

pytestmark = pytest.mark.gpu

ENG = ["Collider", "ContactLoop", "Leapfrog"]


@pytest.mark.parametrize("graph", [False, True])
def test_contact_loop_stress_matches_oracle(graph):
    sc = periodic_hertz(n=1200, spacing=0.92, seed=35, vel_sigma=1.)
    o = build_oracle(sc, evalStress=1)
    d = build_gpu(sc)
    d.set_eval_stress(True)
    kw = dict(contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0, graph=graph)
    step = 0
    for k in range(3):
        o.run(ENG, 30)
        step, _ = d.run(ENG, 30, step, sc["dt"], **kw)
        so, sg = o.cl_stress(), d.contact_loop_stress()
        scale = float(np.max(np.abs(so)))
        print(f"step {step}: max |stress| {scale:.4e}, difference {np.max(np.abs(sg - so)):.3e}", flush=True)
        assert scale > 0
        np.testing.assert_allclose(sg, so, rtol=0, atol=1e-10 * scale)
    # not symmetric: the tangential forces' moments are in it
    assert np.max(np.abs(sg - sg.T)) > 1e-8 * scale
    d.set_eval_stress(False)
    d.run(ENG, 1, step, sc["dt"], **kw)
    assert not d.contact_loop_stress().any()
    d.close()


def test_contact_loop_stress_is_zero_in_aperiodic_scenes():
    sc = deposition(n=400, seed=9, dense=True, vel_sigma=.05)
    d = build_gpu(sc)
    d.set_eval_stress(True)
    d.run(ENG, 5, 0, sc["dt"], contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0)
    assert d.stats()["nReal"] > 0
    assert not d.contact_loop_stress().any()
    d.close()


@pytest.mark.parametrize("graph", [False, True])
def test_contact_loop_stress_while_the_slot_list_grows(graph):
    # spread spheres (one group of slots), then moved into a dense block (more groups than the partial
    # sums held): the gated steps allocate nothing, and the stress is that of the engines called one by one
    from tests.scenes import GpuRunner

    sc = periodic_hertz(n=6000, rmin=3.9e-3, spacing=1.2, seed=36, vel_sigma=.1)
    sc["pos"][1] = sc["pos"][0] + (7.7e-3, 0., 0.)  # one contact
    m = int(np.ceil(6000 ** (1 / 3.)))
    dense = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:6000] + .5) * 7.75e-3
    a, d = GpuRunner(sc), build_gpu(sc)
    kw = dict(contact=contact_kw(sc), leapfrog=dict(damping=sc["damping"]), dynDtPeriod=0, graph=graph)
    step = 0
    for dev in (a.d, d):
        dev.set_eval_stress(True)
    for k in range(2):
        a.run(ENG, 24)
        step, _ = d.run(ENG, 24, step, sc["dt"], **kw)
        s = d.contact_loop_stress()
        assert s.any()
        np.testing.assert_array_equal(s, a.d.contact_loop_stress())
        np.testing.assert_array_equal(d.get("pos"), a.d.get("pos"))
        if k == 0:
            assert 0 < d.stats()["nCandidates"] <= 2048
            for dev in (a.d, d):
                dev.set("pos", dense)
    assert d.stats()["nCandidates"] > 7 * 2048
    d.close()
