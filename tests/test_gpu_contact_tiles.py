"""The tiled contact pass at its edges (MI355X), against the oracle.

A lattice of spheres that do not touch at the build, with a skin that lists
tens of partners per sphere, contracts until every neighbour touches, without a
rebuild: all contacts then come from the rows' second part, so a tile's queue
overflows into full batches, its entry map (16 per particle) runs out, and the
first range is empty.  A second run rebuilds on the way, so both ranges are in
use.  Sizes leave tiles of one, of all but one and of every particle, for
every tile width and history layout.

Layers passing over each other under a contact distance factor: entries of
both parts touch and part within reach of the factor, which resets their
history; with periodic images, two types and frozen spheres.
"""
import numpy as np
import pytest

from conftest import load_engine
from oracle import Oracle
from test_gpu_parity import HYST, check_forces, check_pairs

pytestmark = pytest.mark.gpu


def contracting(n, skin, rolling, normal, every):
    rng = np.random.default_rng(n)
    r0, gap = 1e-3, 2.004e-3
    side = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = 0.02 + gap * g + rng.uniform(-1e-6, 1e-6, (n, 3))
    r = np.full(n, r0)
    W = load_engine().workloads
    mats = W._materials(mur=0.1, etar=0.3)
    if normal != "hertz":
        mats["hysteretic"] = HYST
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.06] * 3, periodic=[0, 0, 0], dt=1e-6, skin=skin, cdf=1.0,
                neigh_every=every, neigh_delay=0, neigh_check=False, rolling=rolling, normal=normal,
                wall_normal="hertz", materials=mats, planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81))
    atoms = dict(x=x, v=-60.0 * (x - x.mean(0)), omega=rng.uniform(-20, 20, (n, 3)), radius=r,
                 rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0, type=np.ones(n, np.int32),
                 tag=np.arange(1, n + 1, dtype=np.int32))
    return spec, atoms


@pytest.mark.parametrize("rolling,normal", [("off", "hertz"), ("epsd", "hertz"), ("epsd", "hysteretic/nonlinear1"),
                                            ("off", "hysteretic/nonlinear1")])
@pytest.mark.parametrize("every", [1000, 10])
def test_tiles_at_their_edges(rolling, normal, every):
    eng = load_engine()
    for n, skin in ((1, 2e-3), (9, 2e-3), (63, 2.2e-3), (65, 2.2e-3), (343, 2.2e-3)):
        spec, atoms = contracting(n, skin, rolling, normal, every)
        o = Oracle(spec, atoms)
        o.setup()
        o.run(60)
        for tile in (-8, -16, -32, -64):
            for precision in ("fp64", "mixed") if normal == "hertz" else ("fp64",):
                s = eng.Simulation(spec, atoms, precision=precision)
                s.set_contact_shape(tile, 64 if tile != -16 else 256)
                s.setup()
                s.step(60)
                # 60 steps of rounding, as the parity tests bound a short
                # horizon; the mixed law's 1e-7 grows like it
                if n > 1:
                    check_forces(s, o, 1e-9 if precision == "fp64" else 1e-4)
                    if precision == "fp64":
                        check_pairs(s, o, hist_tol=1e-9)
                s.close()
        if n == 343:
            touching = (np.asarray(o.pairs()[4]) != 0).sum()
            assert touching >= 2 * 3 * 7 * 7 * 6, touching   # every lattice neighbour, both ways


def passing(n, rolling, normal, every):
    """Layers moving in +x and -x by turns, 0.1 um closer than they can pass."""
    rng = np.random.default_rng(4)
    side = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    odd = g[:, 2] % 2 == 1
    x = g * [2.05e-3, 2.05e-3, 1.9999e-3] + [-5e-3, 5e-3, 0.9995e-3]
    x[odd, 0] += rng.uniform(-1e-5, 6e-5, odd.sum())
    x[:, 0] = np.mod(x[:, 0], 0.03)
    r = np.full(n, 1e-3)
    mats = load_engine().workloads._materials(mur=0.1, etar=0.3, ntypes=2)
    mats["mu"][1, 2] = mats["mu"][2, 1] = 0.2
    mats["e"][2, 2] = 0.6
    mats["hysteretic"] = {k: np.full((3, 3), v[1, 1]) for k, v in HYST.items()}
    spec = dict(box_lo=[0.0] * 3, box_hi=[0.03] * 3, periodic=[1, 0, 0], dt=1e-6, skin=2e-4, cdf=1.05,
                neigh_every=every, neigh_delay=0, neigh_check=False, rolling=rolling, normal=normal,
                wall_normal="hertz", materials=mats, planes=[(2, 0.0, 1)], gravity=(0.0, 0.0, -9.81), freeze=True)
    atoms = dict(x=x, v=np.where(odd, -2.5, 2.5)[:, None] * [1.0, 0.0, 0.0] + rng.uniform(-0.01, 0.01, (n, 3)),
                 omega=rng.uniform(-20, 20, (n, 3)), radius=r, rmass=4.0 / 3.0 * np.pi * r ** 3 * 2500.0,
                 type=rng.integers(1, 3, n).astype(np.int32), tag=np.arange(1, n + 1, dtype=np.int32),
                 freeze=(rng.random(n) < 0.1).astype(np.int32))
    return spec, atoms


@pytest.mark.parametrize("rolling,normal", [("off", "hertz"), ("epsd", "hertz"), ("epsd", "hysteretic/nonlinear1"),
                                            ("off", "hysteretic/nonlinear2")])
@pytest.mark.parametrize("every", [1000, 10])
def test_history_reset_within_the_distance_factor(rolling, normal, every):
    eng = load_engine()
    spec, atoms = passing(215, rolling, normal, every)
    for tile in (-8, -16, -32, -64):
        for precision in ("fp64", "mixed") if normal == "hertz" else ("fp64",):
            o = Oracle(spec, atoms)
            o.add_freeze()
            o.setup()
            s = eng.Simulation(spec, atoms, precision=precision)
            s.set_contact_shape(tile, 0)
            s.setup()
            at_build = (o.pairs()[4] != 0).sum()
            kept = []
            for _ in range(3):   # most touch, then many have parted, then nearly all
                s.step(8)
                o.run(8)
                kept.append((np.abs(o.pairs()[3]).max(1) > 0).sum())
                # 24 steps of rounding, as above
                check_forces(s, o, 1e-9 if precision == "fp64" else 1e-4)
                check_pairs(s, o, hist_tol=1e-9 if precision == "fp64" else 1e-4)
                # a reset history is zero, not small
                gi, gj, gs, gh, gf = s.pairs()
                zero = {(i, j) for i, j, h in zip(*o.pairs()[:2], o.pairs()[3]) if not h.any()}
                assert all((i, j) not in zero for i, j, h in zip(gi, gj, gh) if h.any())
                assert (gf != 0).sum() == (o.pairs()[4] != 0).sum()
            assert kept[0] > at_build > kept[1] > kept[2]
            s.close()


@pytest.mark.parametrize("rolling", ["off", "epsd"])
@pytest.mark.parametrize("wall", ["hysteretic/nonlinear1", "hysteretic/nonlinear2"])
def test_hertz_pairs_with_hysteretic_walls(wall, rolling):
    """Every tile that is compiled for this chain, and the width that the
    particle count gives, with a floor whose history has twelve slots more."""
    eng = load_engine()
    for n in (7, 215):
        spec, atoms = passing(n, rolling, "hertz", 10)
        spec = dict(spec, wall_normal=wall)
        for tile in (0, -8, -16, -32):
            for precision in ("fp64", "mixed"):
                o = Oracle(spec, atoms)
                o.add_freeze()
                o.setup()
                s = eng.Simulation(spec, atoms, precision=precision)
                s.set_contact_shape(tile, 0)
                s.setup()
                s.step(12)
                o.run(12)
                check_forces(s, o, 1e-9 if precision == "fp64" else 1e-4)
                if n > 7:
                    check_pairs(s, o, hist_tol=1e-9 if precision == "fp64" else 1e-4)
                w, ow = s.wall_history(), o.wall_history().reshape(s.wall_history().shape)
                assert np.abs(w).max() > 0
                # the slots range over several orders: a scalar against its own
                # largest, a component (shear, rolling torque) against its vector's
                top = np.abs(ow).reshape(-1, ow.shape[-1]).max(0)
                for k in range(12, len(top), 3):
                    top[k:k + 3] = top[k:k + 3].max()
                assert (np.abs(w - ow).reshape(-1, ow.shape[-1]).max(0)
                        <= (1e-9 if precision == "fp64" else 1e-4) * top).all()
                s.close()


@pytest.mark.parametrize("normal,wall,shapes", [
    ("hertz", "hysteretic/nonlinear1", (-8, -16, -32)), ("hysteretic/nonlinear1", "hertz", (-8, -16, -32, -64)),
    ("hysteretic/nonlinear2", "hysteretic/nonlinear1", (-32,))])
def test_autotune_keeps_to_compiled_shapes(normal, wall, shapes):
    """The shape that the autotuner returns is one that runs for the chain."""
    eng = load_engine()
    spec, atoms = passing(215, "epsd", normal, 10)
    for _ in range(4):
        s = eng.Simulation(dict(spec, wall_normal=wall), atoms)
        s.setup()
        lanes, block, ms = s.autotune(reps=1)
        assert lanes in shapes and block in (64, 128, 256) and ms > 0.0
        s.close()
