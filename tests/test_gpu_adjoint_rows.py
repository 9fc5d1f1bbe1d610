"""The reverse step on rows whose touching entries need several passes of a
particle's lanes (8 entries a pass), against central differences (MI355X).

Two instances of one context over a short window: a sphere of 2.5 mm touched
by 40 of 0.8 mm, cut by the periodic x boundary (five passes of touching
entries, some of them images, and a row past the rebuild's staging rows), and
108 equal spheres in a face-centred packing (twelve touching partners inside,
two passes).  Touching partners come first in a row, the others after them.
"""
import importlib

import numpy as np
import pytest
import torch

from conftest import load_engine

pytestmark = pytest.mark.gpu

SIDE = 0.02
STEPS, EVERY = 45, 20


def shell():
    R, r, m = 2.5e-3, 0.8e-3, 40
    k = np.arange(m) + 0.5
    ct = 1.0 - 2.0 * k / m
    st, ph = np.sqrt(1.0 - ct * ct), np.pi * (1.0 + 5.0 ** 0.5) * k
    rng = np.random.default_rng(1)
    d = (R + r - rng.uniform(2e-6, 3e-6, m))[:, None] * np.stack([st * np.cos(ph), st * np.sin(ph), ct], 1)
    x = np.concatenate([np.zeros((1, 3)), d]) + [0.7e-3, 8e-3, 0.0]
    rad = np.concatenate([[R], np.full(m, r)])
    x[:, 2] -= (x[:, 2] - rad).min() + 2e-6     # the lowest one 2 um deep in the floor
    x[:, 0] = np.mod(x[:, 0], SIDE)
    return x, rad


def packing():
    g = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    x = 1.9965e-3 * 2 ** 0.5 * (g + 0.5 * np.array([[0, 0, 0], [1, 1, 0], [1, 0, 1], [0, 1, 1]])).reshape(-1, 3)
    x = x + np.random.default_rng(2).uniform(-3e-7, 3e-7, x.shape) + [4e-3, 4e-3, 0.9985e-3]
    return x, np.full(len(x), 1e-3)


def moving(x, r, seed):
    rng = np.random.default_rng(seed)
    n = len(r)
    return dict(x=x, v=rng.uniform(-0.02, 0.02, (n, 3)), omega=rng.uniform(-80, 80, (n, 3)), radius=r,
                rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0)


def test_long_rows_against_finite_differences():
    eng = load_engine()
    # spins that slide some contacts; seeds with no contact event between the
    # runs of the differences (their quotients agree to 1e-5 from 1e-5 to 1e-6)
    beds = [moving(*shell(), 9), moving(*packing(), 8)]
    atoms = {k: np.concatenate([b[k] for b in beds]) for k in beds[0]}
    inst = np.repeat(np.arange(2, dtype=np.int32), [len(b["radius"]) for b in beds])
    n = len(inst)
    atoms.update(type=np.ones(n, np.int32), tag=np.arange(1, n + 1, dtype=np.int32))
    spec = dict(box_lo=[0.0] * 3, box_hi=[SIDE] * 3, periodic=[1, 0, 0], dt=1e-6, skin=9e-4, cdf=1.0, neigh_every=10,
                neigh_delay=0, neigh_check=False, rolling="off", materials=eng.workloads._materials(),
                planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81), observe_plane=0)
    par = dict(Y=np.array([4e6, 6e6]), mu=np.array([0.3, 0.5]), e=np.array([0.5, 0.8]))
    adj = importlib.import_module("liggghts_inl_amd.adjoint")

    leaf = [torch.tensor(par[k], requires_grad=True) for k in ("Y", "mu", "e")]
    h, w = adj.BatchObservables.apply(*leaf, spec, atoms, inst, STEPS, EVERY)
    value0 = (1e2 * h + w).detach().numpy()
    grad = torch.autograd.grad((1e2 * h + w).sum(), leaf)

    def run(p):
        s = eng.Simulation(dict(spec, instances=dict(inst=inst, **p)), atoms)
        s.setup()
        s.step(STEPS)
        return s

    def value(p):
        s = run(p)
        o = s.observables()
        s.close()
        return 1e2 * o[:, 1] / o[:, 0] + o[:, 2]

    s = run(par)
    ti, tj, sh, _, fl = s.pairs()
    rows = np.bincount(ti[fl != 0], minlength=n + 1)[1:]
    assert rows[inst == 0].max() == 40 and rows[inst == 1].max() == 12
    assert np.bincount(ti, minlength=n + 1)[1:][inst == 1].max() > 12   # others behind the touching ones
    images = (fl != 0) & (sh != 13)             # 13: no periodic shift
    assert (images & (ti == 1)).any()           # of the large sphere's row
    s.close()

    for k, g in zip(("Y", "mu", "e"), grad):
        step = 1e-5 * par[k]
        fd = (value(dict(par, **{k: par[k] + step})) - value(dict(par, **{k: par[k] - step}))) / (2 * step)
        # as the pours' gradients are bounded; the quotient itself rounds at
        # 1e-16 / 1e-5 of the value
        floor = 1e-11 * np.abs(value0) / par[k]
        assert np.all(np.abs(fd) > 1e4 * floor), (k, fd, floor)
        assert np.all(np.abs(g.numpy() - fd) <= 1e-4 * np.abs(fd) + floor), (k, g, fd)
