"""Several adjoint windows on one context (MI355X).

The second window has the first one's checkpoint interval and more list
entries per particle, so its records are larger; its gradient is, bit for bit,
that of a context of its own.
"""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


def lattice(side, gap):
    rng = np.random.default_rng(7)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(g)
    r = np.full(n, 1e-3)
    x = 0.9985e-3 + gap * g + rng.uniform(-5e-7, 5e-7, g.shape)
    return dict(x=x, v=rng.uniform(-0.02, 0.02, (n, 3)), omega=rng.uniform(-5, 5, (n, 3)), radius=r,
                rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0, type=np.ones(n, np.int32),
                tag=np.arange(1, n + 1, dtype=np.int32))


def window(s, steps=40, every=20):
    s.setup()
    s.adjoint_forward(steps, every)
    return s.adjoint_backward(np.ones(1), np.ones(1))


@pytest.mark.parametrize("sides", [(4, 4), (4, 6), (6, 4)])
def test_second_window_with_a_larger_list(sides):
    eng = load_engine()
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.03] * 3, periodic=[0, 0, 0], dt=1e-6, skin=9e-4, cdf=1.0, neigh_every=10,
                neigh_delay=0, neigh_check=False, rolling="off", materials=eng.workloads._materials(),
                planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81), observe_plane=0)
    loose, dense = lattice(sides[0], 3.5e-3), lattice(sides[1], 1.996e-3)
    fresh = eng.Simulation(spec, dense)
    want = window(fresh)
    s = eng.Simulation(spec, loose)
    window(s)
    few = s.list_stats()[0]
    s.upload(dense)
    got = window(s)
    assert few < 1.0 < 10.0 < s.list_stats()[0]
    assert np.isfinite(want).all() and np.abs(want).max() > 0.0
    assert np.array_equal(got, want)


def replaced(s, how, dense):
    """What leaves a finished window without its particles or its list."""
    if how == "setup":
        s.setup()
    elif how == "rebuild":
        s.rebuild()
    elif how == "step":
        s.step(25)   # rebuilds every 10
    elif how == "upload":
        s.upload(lattice(6, 1.996e-3))
    elif how == "history":
        ti, tj, sh, hi, fl = s.pairs()
        s.set_history(ti[fl != 0], tj[fl != 0], hi[fl != 0])
    elif how == "failed":   # a later window that ends early, with fewer checkpoints
        s.upload(dict(dense, v=dense["v"] + 100.0))
        s.setup()
        with pytest.raises(load_engine().DemError, match="half the skin"):
            s.adjoint_forward(40, 40)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("how", ["setup", "rebuild", "step", "upload", "history", "failed"])
def test_window_ends_with_its_particles_or_list(how, graph):
    eng = load_engine()
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.03] * 3, periodic=[0, 0, 0], dt=1e-6, skin=9e-4, cdf=1.0, neigh_every=10,
                neigh_delay=0, neigh_check=False, rolling="off", materials=eng.workloads._materials(),
                planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81), observe_plane=0, graph=graph)
    dense = lattice(4, 1.996e-3)
    s = eng.Simulation(spec, dense)
    s.setup()
    s.step(45)       # with a graph: its periods are recorded
    s.setup()
    s.adjoint_forward(40, 5)
    one = np.ones(1)
    first = s.adjoint_backward(one, one)
    assert np.array_equal(s.adjoint_backward(one, one), first)   # the window stays until then
    replaced(s, how, dense)
    with pytest.raises(eng.DemError, match="dem_adjoint_forward first"):
        s.adjoint_backward(one, one)
