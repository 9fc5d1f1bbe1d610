"""Stepping under the distance check without a graph (MI355X): runs of steps
whose checks stay on the device give, bit for bit, the state of the same steps
taken one call at a time, where the host asks after every check.

The columns' spheres are fast enough that checks halt a run several times, so
runs end early, grow and shrink; a contact pass that integrates checks the next
step itself (columns, pour), a mesh or bonds keep the check apart.
"""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


def column(n, vmax, seed, **kw):
    W = load_engine().workloads
    spec, atoms = W.packed_column(n=n, slab_n=n, Lxy=0.02)
    rng = np.random.default_rng(seed)
    spec = dict(spec, neigh_every=1, neigh_check=True, skin=2e-4, **kw)
    return spec, dict(atoms, v=rng.uniform(-vmax, vmax, (n, 3)), omega=rng.uniform(-20, 20, (n, 3)))


CASES = {
    "column": lambda: (column(1500, 1.5, 1), "fp64", 700),
    "column-mixed": lambda: (column(1501, 3.0, 2), "mixed", 500),
    "lanes": lambda: (column(1500, 1.5, 1), "fp64", 400),
    "pour": lambda: (load_engine().workloads.pour_box(n=1000, spacing=2.02e-3, jitter=2e-5), "fp64", 400),
    "hopper": lambda: (load_engine().workloads.hopper(n=2000, ntheta=60, wall_overlap=2e-5), "fp64", 200),
    "fibres": lambda: (load_engine().workloads.fibres(nchains=20, nsph=10), "fp64", 300),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("graph", [False, True])
def test_runs_equal_single_steps(name, graph):
    eng = load_engine()
    (spec, atoms), precision, steps = CASES[name]()
    spec = dict(spec, neigh_every=1, neigh_check=True, skin=1e-6 if name == "fibres" else spec["skin"])
    a = eng.Simulation(dict(spec, graph=graph), atoms, precision=precision)
    b = eng.Simulation(spec, atoms, precision=precision)
    for s in (a, b):
        if name == "lanes":
            s.set_contact_shape(4, 0)
        s.setup()
    for chunk in (steps // 3, 2, steps - steps // 3 - 2):
        a.step(chunk)
        for _ in range(chunk):
            b.step(1)
        sa, sb = a.state(), b.state()
        for k in ("x", "v", "omega", "f", "torque"):
            assert np.array_equal(sa[k], sb[k]), (name, k)
    assert a.timestep() == b.timestep()
    pa, pb = a.pairs(), b.pairs()
    for p, q in zip(pa, pb):
        assert np.array_equal(p, q)
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [False, True])
def test_runs_between_insertions(graph):
    """A pour under the distance check into which atoms are inserted every 37
    steps: rebuilds that an insertion forces lie between those that a check
    asks for, and each run ends before the next insertion."""
    eng = load_engine()
    spec, atoms = eng.workloads.pour_box(n=800, spacing=2.02e-3, jitter=2e-5)
    hi = spec["box_hi"]
    spec = dict(spec, neigh_every=1, neigh_check=True, skin=6e-5)
    ins = dict(seed=15485863, dist_seed=15485867, templates=[dict(type=1, radius=0.9e-3, density=2500.0)],
               weights=[1.0], region=((0.0, 0.0, 0.6 * hi[2]), tuple(hi)), volumefraction_region=0.2,
               maxattempt=20, insert_every=37, all_in=True,
               vel=("uniform", (0.0, 0.0, -0.6), (0.2, 0.2, 0.2)), group_mask=0)
    a = eng.Simulation(dict(spec, graph=graph), atoms)
    b = eng.Simulation(spec, atoms)
    for s in (a, b):
        s.add_insert_pack(ins)
        s.setup()
    for chunk in (150, 2, 148):
        a.step(chunk)
        for _ in range(chunk):
            b.step(1)
        assert a.n == b.n > 800
        sa, sb = a.state(), b.state()
        for k in ("x", "v", "omega", "f", "torque"):
            assert np.array_equal(sa[k], sb[k]), k
    for p, q in zip(a.pairs(), b.pairs()):
        assert np.array_equal(p, q)
    a.close()
    b.close()
