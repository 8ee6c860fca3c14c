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
