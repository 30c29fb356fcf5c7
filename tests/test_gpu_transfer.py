"""State transfers: every byte of the slot arrays comes back as it went in,
for one chunk, several, the chunk edges and the two-thread sizes."""
import numpy as np
import pytest

import comd_amd as CA

pytestmark = pytest.mark.gpu


def random_slots(ncells, seed):
    """Slot arrays with values in every slot, empty ones included."""
    rng = np.random.default_rng(seed)
    S = ncells * CA.MAXATOMS
    natoms = rng.integers(0, 3, ncells).astype(np.int32)
    return dict(natoms=natoms, id=rng.permutation(S).astype(np.int32), itype=rng.integers(0, 9, S).astype(np.int32),
                r=rng.uniform(0.0, 2.0, (S, 3)), p=rng.standard_normal((S, 3)))


# cells per dimension: a full download takes 6660 bytes per cell and an
# upload 3588, chunks are 1 MB below 64 MB (157 and 292 cells) and 4 MB above
@pytest.mark.parametrize("nb", [(3, 3, 3), (157, 1, 1), (158, 1, 1), (292, 1, 1), (293, 1, 1), (9, 13, 17),
                                (22, 22, 21), (27, 27, 27)])
def test_slots_round_trip(nb):
    pot = CA.LJPotential(sigma=1.0, epsilon=0.01, cutoff=2.0, mass=1.0)
    sim = CA.Simulation(pot, [2.0 * n + 0.01 for n in nb])
    assert sim.nbx == nb
    given = random_slots(sim.ncells, 5)
    sim.upload(*[given[k] for k in ("natoms", "id", "itype", "r", "p")])
    got = sim.download()
    for k, v in given.items():
        assert np.array_equal(got[k], v), k
    for k in ("f", "rho", "fi"):
        assert not got[k].any(), k


def test_batch_parts_and_missing_fields():
    pot = CA.LJPotential(sigma=1.0, epsilon=0.01, cutoff=2.0, mass=1.0)
    sizes = [(3, 4, 5), (40, 5, 3), (7, 3, 3)]
    b = CA.Batch([dict(pot=pot, bounds=[2.0 * n + 0.01 for n in nb]) for nb in sizes], precision="fp64")
    hip = CA.libraries()[0]
    given = [random_slots(int(np.prod(nb)), 11 + r) for r, nb in enumerate(sizes)]
    for r, g in enumerate(given):
        b.upload(r, *[g[k] for k in ("natoms", "id", "itype", "r", "p")])
    for r, g in enumerate(given):
        got = b.download(r)
        for k, v in g.items():
            assert np.array_equal(got[k], v), (r, k)
    # no types and no momenta: zeros; a single field alone comes back
    g = given[1]
    assert hip.comd_batch_upload(b.ctx, 1, CA._ptr(g["natoms"], CA.C.c_int), CA._ptr(g["id"], CA.C.c_int), None,
                                 CA._ptr(g["r"]), None) == 0
    got = b.download(1)
    assert np.array_equal(got["r"], g["r"]) and not got["p"].any() and not got["itype"].any()
    rho = np.full(len(g["id"]), 7.0)
    assert hip.comd_batch_download(b.ctx, 1, None, None, None, None, None, None, CA._ptr(rho), None) == 0
    assert not rho.any()
    assert hip.comd_batch_download(b.ctx, 1, None, None, None, None, None, None, None, None) == 0
    for r in (0, 2):
        assert np.array_equal(b.download(r)["r"], given[r]["r"])


def test_large_transfer_with_another_device_current():
    """The second copying thread's stream belongs to the context's device, not
    to the one that is current when the first large transfer is made."""
    torch = pytest.importorskip("torch")
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two devices")
    pot = CA.LJPotential(sigma=1.0, epsilon=0.01, cutoff=2.0, mass=1.0)
    torch.cuda.set_device(0)
    try:
        sim = CA.Simulation(pot, [2.0 * n + 0.01 for n in (27, 27, 27)])  # 71 MB up, 131 MB down
        given = random_slots(sim.ncells, 5)
        torch.cuda.set_device(1)
        sim.upload(*[given[k] for k in ("natoms", "id", "itype", "r", "p")])
        got = sim.download()
        for k, v in given.items():
            assert np.array_equal(got[k], v), k
    finally:
        torch.cuda.set_device(0)
