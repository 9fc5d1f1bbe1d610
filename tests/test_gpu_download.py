"""dem_download in upload order, on both sides of its one-copy limit and with
some of the arrays left out (MI355X)."""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 8192, 8193])
def test_download_order(n):
    eng = load_engine()
    W = eng.workloads
    rng = np.random.default_rng(n)
    g = np.stack(np.meshgrid(*[np.arange(21)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = 2e-3 + 3e-3 * g[rng.permutation(len(g))[:n]]     # apart, in random order
    r = np.full(n, 1e-3)
    atoms = dict(x=x, v=rng.normal(size=(n, 3)), omega=rng.normal(size=(n, 3)), radius=r, rmass=1e-6 * (1 + rng.random(n)),
                 type=np.ones(n, np.int32), tag=rng.permutation(n).astype(np.int32) + 1)
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.07] * 3, periodic=[0, 0, 0], dt=1e-6, skin=2e-4, cdf=1.0, neigh_every=10,
                neigh_delay=0, neigh_check=False, rolling="off", materials=W._materials(), planes=[],
                gravity=(0.0, 0.0, -9.81))
    s = eng.Simulation(spec, atoms)
    s.setup()
    st = s.state()
    for k in ("x", "v", "omega"):
        assert np.array_equal(st[k], atoms[k])
    assert np.array_equal(st["f"], atoms["rmass"][:, None] * np.array([0.0, 0.0, -9.81]))
    assert not st["torque"].any()
    from liggghts_inl_amd.engine import _dp

    v, f = np.zeros((n, 3)), np.zeros((n, 3))
    s._chk(s.L.dem_download(s.h, None, _dp(v), None, _dp(f), None))
    assert np.array_equal(v, atoms["v"]) and np.array_equal(f, st["f"])
