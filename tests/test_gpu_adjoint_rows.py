"""The reverse step on rows longer than one pass of a particle's lanes (8
entries), against central differences (MI355X).

A touching lattice whose skin lists the face and edge neighbours (6 + 12), in
two instances of different sizes, over a short window; edge neighbours do not
touch, so their entries only pass the history on.
"""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


def lattice(side, b):
    rng = np.random.default_rng(side)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    return 0.999e-3 + 1.996e-3 * g + rng.uniform(-5e-7, 5e-7, g.shape), np.full(len(g), b, np.int32)


def test_long_rows_against_finite_differences():
    eng = load_engine()
    W = eng.workloads
    xs, inst = (np.concatenate(z) for z in zip(lattice(4, 0), lattice(5, 1)))
    n = len(xs)
    rng = np.random.default_rng(3)
    r = np.full(n, 1e-3)
    atoms = dict(x=xs, v=rng.uniform(-0.02, 0.02, (n, 3)), omega=rng.uniform(-5, 5, (n, 3)), radius=r,
                 rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0, type=np.ones(n, np.int32),
                 tag=np.arange(1, n + 1, dtype=np.int32))
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.02] * 3, periodic=[0, 0, 0], dt=1e-6, skin=9e-4, cdf=1.0, neigh_every=10,
                neigh_delay=0, neigh_check=False, rolling="off", materials=W._materials(),
                planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81), observe_plane=0)
    par = dict(Y=np.array([4e6, 6e6]), mu=np.array([0.3, 0.5]), e=np.array([0.5, 0.8]))
    adj = __import__("importlib").import_module("liggghts_inl_amd.adjoint")
    import torch

    spec0 = {k: v for k, v in spec.items()}
    leaf = [torch.tensor(par[k], requires_grad=True) for k in ("Y", "mu", "e")]
    h, w = adj.BatchObservables.apply(*leaf, spec0, atoms, inst, 60, 25)
    grad = torch.autograd.grad((1e2 * h + w).sum(), leaf)

    def value(p):
        s = eng.Simulation(dict(spec, instances=dict(inst=inst, **p)), atoms)
        s.setup()
        s.step(60)
        assert s.list_stats()[0] > 10.0   # rows past one pass
        o = s.observables()
        s.close()
        return 1e2 * o[:, 1] / o[:, 0] + o[:, 2]

    for k, g in zip(("Y", "mu", "e"), grad):
        step = 1e-5 * par[k]
        fd = (value(dict(par, **{k: par[k] + step})) - value(dict(par, **{k: par[k] - step}))) / (2 * step)
        # as the pours' gradients are bounded; the difference quotient itself
        # rounds at 1e-16 / 1e-5 of the value
        assert np.all(np.abs(g.numpy() - fd) <= 1e-4 * np.abs(fd) + 1e-8 / par[k]), (k, g, fd)
