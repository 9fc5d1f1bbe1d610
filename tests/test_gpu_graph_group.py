"""A recorded graph and fix nve/sphere on a group (MI355X): a change of the
integrated group after recording is followed, on a rebuild cadence and under
the distance check, bit for bit as without the graph."""
import numpy as np
import pytest

from conftest import load_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("check", [False, True])
def test_graph_follows_integrated_group(check):
    eng = load_engine()
    spec, atoms = eng.workloads.packed_column(n=3000, slab_n=3000)
    spec = dict(spec, neigh_check=check, neigh_every=1 if check else 10)
    some = (np.arange(3000) % 3 != 0).astype(np.int32)

    def run(graph):
        s = eng.Simulation(dict(spec, graph=graph), atoms)
        s.set_group(2, some)
        s.setup()
        out = []
        for bit, steps in ((-1, 47), (2, 61), (-1, 62)):
            s.set_integrate_group(bit)
            s.step(steps)
            out.append(s.state())
        s.close()
        return out

    plain, graph = run(False), run(True)
    for a, b in zip(plain, graph):
        for k in ("x", "v", "omega", "f", "torque"):
            assert np.array_equal(a[k], b[k]), k
    # while only the group was integrated, the others stood still
    still = some == 0
    assert np.array_equal(plain[0]["v"][still], plain[1]["v"][still])
    assert not np.array_equal(plain[1]["v"][still], plain[2]["v"][still])
