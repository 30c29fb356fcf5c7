"""Steps inside one call (whose second half drift and the next step's first
one are done in one pass over the atoms) against the same steps called one at
a time (each half drift by itself, parity-tested against the oracle): the
same slots, ids, positions and momenta, bit for bit."""
import numpy as np
import pytest

import comd_amd as CA
from helpers import DT_INTERNAL, compact, seeded_atoms

pytestmark = pytest.mark.gpu

CUT = 2.0
RMASS = CA.AMU_TO_ME


def gas(nb, per_cell, hop, seed):
    """Nearly free atoms in nb cells per dimension of edge a little above
    CUT, moving up to hop cells per half step."""
    rng = np.random.default_rng(seed)
    bounds = np.array([CUT * n + 0.05 for n in nb])
    n = int(per_cell * np.prod(nb))
    x = rng.uniform(0.0, 1.0, (n, 3)) * bounds
    step = rng.uniform(-1.0, 1.0, (n, 3)) * hop * (bounds / np.array(nb))
    return bounds, x, step * RMASS / (0.5 * DT_INTERNAL)


def same(a, b, what):
    a, b = dict(a), dict(b)
    assert np.array_equal(a["natoms"], b["natoms"]), what
    ca, cb = compact(a), compact(b)
    for k in ("id", "itype", "r", "p", "f"):
        assert np.array_equal(ca[k], cb[k]), f"{what}: {k}"


def both_ways(make, steps, what, graph=0):
    a, b = make(), make()
    a.tune(graph=graph)
    for s in (a, b):
        s.force()
    for block in steps:
        a.steps(block, 1.0e-15)
        for _ in range(block):
            b.steps(1, 1.0e-15)
        for s in (a, b):
            s.force()
        if isinstance(a, CA.Batch):
            for r in range(a.nrep):
                same(a.download(r), b.download(r), f"{what} replica {r}")
        else:
            same(a.download(), b.download(), what)
        a.sync()
        b.sync()
    return a, b


# hop below 1: an atom moves one cell at most; above: arrivals that move
# again, in either pass, take the serial replay
@pytest.mark.parametrize("nb", [(1, 1, 1), (2, 3, 1), (3, 3, 3), (5, 4, 7), (11, 3, 6)])
@pytest.mark.parametrize("hop", [0.05, 0.45, 0.95, 1.3, 2.6])
@pytest.mark.parametrize("periodic", [True, False])
def test_gas(gpu, nb, hop, periodic):
    pot = CA.LJPotential(sigma=0.4, epsilon=1e-12, cutoff=CUT, mass=1.0)
    bounds, x, p = gas(nb, 6, hop, 7)

    def make():
        s = CA.Simulation(pot, bounds, periodic=periodic)
        s.tune(skin=0.0)
        s.bin_atoms(x, p, itype=3)
        return s

    both_ways(make, (2, 5, 9), f"gas {nb} {hop} {periodic}")


@pytest.mark.parametrize("per_cell", [26, 36])
def test_dense_cells(gpu, per_cell):
    """Mean occupancy below and above half the slots (the rule's line)."""
    pot = CA.LJPotential(sigma=0.05, epsilon=1e-14, cutoff=CUT, mass=1.0)
    bounds, x, p = gas((5, 5, 5), per_cell, 0.1, 3)

    def make():
        s = CA.Simulation(pot, bounds)
        s.bin_atoms(x, p)
        return s

    both_ways(make, (6,), f"dense {per_cell}")


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_crystal_with_rebuilds(gpu, cu500, graph, precision):
    xyz, p, bounds = seeded_atoms(7, 3.615, 63.55, temp=2500.0, disp=0.1, seed=4)

    def make():
        s = CA.Simulation(cu500, bounds, precision=precision)
        s.bin_atoms(xyz, p, itype=1)
        return s

    a, b = both_ways(make, (3, 30, 2, 25), f"crystal {precision}", graph)
    assert a.list_info() == b.list_info() and a.list_info()["builds"] > 3


@pytest.mark.parametrize("hop", [0.3, 1.4])
def test_lists_follow_the_replay(gpu, hop):
    """Neighbour lists on, atoms close enough to interact, and passes that
    need the serial replay: its id -> slot map and list positions."""
    pot = CA.LJPotential(sigma=0.9, epsilon=1e-8, cutoff=CUT, mass=1.0)
    nb = np.array([9, 8, 7])
    bounds = CUT * nb + 0.05
    grid = np.stack(np.meshgrid(*[np.arange(int(b / 1.5)) for b in bounds], indexing="ij"), -1).reshape(-1, 3)
    rng = np.random.default_rng(5)
    x = (grid + 0.5) * 1.5 + rng.uniform(-0.2, 0.2, grid.shape)
    p = rng.uniform(-0.02, 0.02, x.shape) * CUT * RMASS / (0.5 * DT_INTERNAL)
    fast = rng.choice(len(x), 4, replace=False)
    p[fast] = 0.0
    p[fast, rng.integers(0, 3, 4)] = hop * CUT * RMASS / (0.5 * DT_INTERNAL)

    def make():
        s = CA.Simulation(pot, bounds)
        s.bin_atoms(x, p)
        return s

    a, b = both_ways(make, (2, 7), f"replay with lists {hop}")
    assert a.list_info() == b.list_info() and a.list_info()["valid"] == 1


def test_batch_with_one_fast_replica(gpu):
    pot = CA.LJPotential(sigma=0.4, epsilon=1e-12, cutoff=CUT, mass=1.0)
    made = [gas((4, 5, 3), 5, 0.4, 1), gas((6, 3, 3), 5, 1.7, 2), gas((3, 3, 3), 5, 0.9, 3)]

    def make():
        b = CA.Batch([dict(pot=pot, bounds=m[0]) for m in made], precision="fp64")
        b.tune(skin=0.0)
        for r, m in enumerate(made):
            b.bin_atoms(r, m[1], m[2])
        return b

    both_ways(make, (2, 6, 3), "batch", graph=1)
