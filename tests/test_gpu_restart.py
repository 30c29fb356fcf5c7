"""Restart from a snapshot (comd_snapshot_save / comd_snapshot_load): N
steps run straight through and the same N steps split by a save, a new
context and a load end in the same state, bit for bit -- slot order,
positions, momenta, forces and energies -- with the neighbour lists
rebuilt on both sides of the save."""
import numpy as np
import pytest

import comd_amd as CA
from helpers import seeded_atoms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,lanes", [("fp64", None), ("mixed", None), ("fp64", 4)])
def test_restart_continues_bit_for_bit(gpu, cu500, tmp_path, precision, lanes):
    """lanes: the saving context's lanes per atom in the list passes (the
    order of their sums), which the snapshot carries to a context left at
    its default."""
    xyz, p, bounds = seeded_atoms(8, 3.615, 63.55, temp=3000.0, disp=0.05, seed=61)

    def fresh():
        s = CA.Simulation(cu500, bounds, defgrad=0.0, precision=precision)
        s.bin_atoms(xyz, p)
        s.rebox()
        return s

    a = fresh()
    if lanes:
        a.tune(list_lanes=lanes)
    a.nsteps(20)
    builds_before = a.list_info()["builds"]
    path = tmp_path / "state.snap"
    a.snapshot_save(path)
    a.nsteps(30)
    ga = a.download()
    ea = a.energy()
    builds_after = a.list_info()["builds"]
    print(f"[restart {precision}] list builds {builds_before} at the save, {builds_after} at the end", flush=True)
    assert builds_after > builds_before  # the lists were rebuilt after the save

    b = CA.Simulation(cu500, bounds, defgrad=0.0, precision=precision)
    b.snapshot_load(path)
    b.nsteps(30)
    gb = b.download()
    for k in ("natoms", "id", "itype", "r", "p", "f", "rho", "fi"):
        assert np.array_equal(ga[k], gb[k]), k
    assert b.energy() == ea


@pytest.mark.parametrize("lanes", [8, 16])
def test_restart_with_more_lanes(gpu, cu500, tmp_path, lanes):
    """The lanes per atom come from the file for any number there is."""
    test_restart_continues_bit_for_bit(gpu, cu500, tmp_path, "fp64", lanes)


def test_restart_from_lists_of_the_earlier_default_shape(gpu, cu500, tmp_path):
    """Snapshots of 32 000 atoms were written with 2 x 2 x 1 cells to a group
    by default, now 2 x 2 x 2: a context with the default takes the file's
    shape and continues bit for bit; one whose shape was tuned refuses it."""
    n = 20
    xyz, p, bounds = seeded_atoms(n, 3.615, cu500.mass, temp=600.0, disp=0.1, seed=5)
    path = str(tmp_path / "s.bin")
    a = CA.Simulation(cu500, bounds, defgrad=0.0)
    a.tune(list_groups=4)
    a.bin_atoms(xyz, p)
    a.force()
    a.nsteps(5)
    a.snapshot_save(path)
    b = CA.Simulation(cu500, bounds, defgrad=0.0)
    b.snapshot_load(path)
    c = CA.Simulation(cu500, bounds, defgrad=0.0)
    c.tune(list_groups=2)
    with pytest.raises(CA.ComdError):
        c.snapshot_load(path)
    for s in (a, b):
        s.nsteps(30)
    assert b.list_info()["valid"] == 1
    ga, gb = a.download(), b.download()
    for k in ("natoms", "id", "itype", "r", "p", "f", "rho", "fi"):
        assert np.array_equal(ga[k], gb[k]), k


@pytest.mark.parametrize("how", ["bin", "upload", "tune", "autotune"])
def test_the_earlier_shape_ends_with_its_atoms(gpu, cu500, tmp_path, how):
    """A context that took a file's lists in the earlier default shape has
    today's shape again once its atoms are replaced or the shape is tuned."""
    xyz, p, bounds = seeded_atoms(20, 3.615, cu500.mass, temp=600.0, disp=0.1, seed=5)
    path = str(tmp_path / "s.bin")
    a = CA.Simulation(cu500, bounds, defgrad=0.0)
    a.bin_atoms(xyz, p)
    today = a.list_occupancy()
    a.tune(list_groups=4)
    earlier = a.list_occupancy()
    assert earlier != today
    a.force()
    a.snapshot_save(path)
    b = CA.Simulation(cu500, bounds, defgrad=0.0)
    b.snapshot_load(path)
    assert b.list_occupancy() == earlier
    if how == "bin":
        b.bin_atoms(xyz, p)
    elif how == "upload":
        s = b.download()
        b.upload(*[s[k] for k in ("natoms", "id", "itype", "r", "p")])
    elif how == "tune":
        b.tune(list_groups=-1)
    else:
        b.autotune_lists()
        b.tune(list_groups=-1, list_rows_lds=-1, list_threads_div=1)
    assert b.list_occupancy() == today
