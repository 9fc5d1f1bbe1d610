"""A second, larger upload into a context whose settings were made for the
first one (MI355X): every per-particle array follows the particles."""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


def floor_layer(side):
    """A square layer of spheres resting 1 um deep in the bottom plane."""
    rng = np.random.default_rng(side)
    g = np.stack(np.meshgrid(np.arange(side), np.arange(side), indexing="ij"), -1).reshape(-1, 2)
    n = len(g)
    r = rng.uniform(0.9e-3, 1e-3, n)
    x = np.column_stack([2e-3 + 2.1e-3 * g, r - 1e-6])
    return dict(x=x, v=rng.uniform(-0.01, 0.01, (n, 3)), omega=rng.uniform(-5, 5, (n, 3)), radius=r,
                rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0, type=np.ones(n, np.int32),
                tag=np.arange(1, n + 1, dtype=np.int32))


@pytest.mark.parametrize("sides", [(2, 3), (3, 60), (60, 3)])
def test_observed_plane(sides):
    eng = load_engine()
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.14, 0.14, 0.02], periodic=[0, 0, 0], dt=1e-6, skin=2e-4, cdf=1.0,
                neigh_every=10, neigh_delay=0, neigh_check=False, rolling="off",
                materials=eng.workloads._materials(), planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81),
                observe_plane=0)
    a = eng.Simulation(spec, floor_layer(sides[0]))
    a.setup()
    a.step(5)
    a.upload(floor_layer(sides[1]))
    b = eng.Simulation(spec, floor_layer(sides[1]))
    for s in (a, b):
        s.setup()
        s.step(25)
    oa, ob = a.observables(), b.observables()
    assert ob[0, 2] > 0.0
    assert np.array_equal(oa, ob)
    for k, v in b.state().items():
        assert np.array_equal(a.state()[k], v), k
