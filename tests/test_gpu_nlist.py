"""GPU tests of the Verlet neighbour lists (COMD_TUNE_SKIN_MILLI): the list
kernels must give what the link-cell kernels give (themselves parity-tested
against the oracle and the reference's fixtures) on the same atoms: the same
neighbour counts exactly, forces, energies, rho and F' to 1e-12, and the same
trajectories, including across list rebuilds triggered on the device.

The mixed-precision list passes read positions in 32-bit periodic fixed
point (L / 2^32 per unit, 6.7e-9 A for these 29 A boxes) and F' as a float;
they are held to the mixed-precision bar, 1e-6 against the FP64 link-cell
kernels.
"""
import numpy as np
import pytest

import comd_amd as CA
from helpers import compact, force_rel_error, scalar_rel_error, seeded_atoms

pytestmark = pytest.mark.gpu


def pair_of_sims(pot, n, lat, temp, disp, seed, evaluation="table", precision="fp64"):
    xyz, p, bounds = seeded_atoms(n, lat, pot.mass, temp=temp, disp=disp, seed=seed)
    out = []
    for skin in (0.4, 0.0):
        s = CA.Simulation(pot, bounds, defgrad=0.0, evaluation=evaluation, precision=precision)
        s.tune(skin=skin)
        s.bin_atoms(xyz, p)
        s.rebox()
        out.append(s)
    return out


def assert_same(a, b, what, tol=1e-12, lj=False, stol=None):
    """Forces to tol; energies, rho and F' to stol (default tol)."""
    stol = tol if stol is None else stol
    ga, gb = a.download(), b.download()
    assert np.array_equal(ga["natoms"], gb["natoms"]), what
    ca, cb = compact(ga), compact(gb)
    assert np.array_equal(ca["id"], cb["id"]), what
    ef = force_rel_error(ca["f"], cb["f"]).max()
    ee = scalar_rel_error(ca["f"][:, 3], cb["f"][:, 3]).max()
    print(f"[{what}] lists vs cells: force {ef:.2e} energy {ee:.2e}", flush=True)
    assert ef <= tol and ee <= stol, what
    if not lj:
        assert scalar_rel_error(ca["rho"], cb["rho"]).max() <= stol
        assert scalar_rel_error(ca["fi"], cb["fi"]).max() <= stol
    na, _ = a.download_aux()
    nb, _ = b.download_aux()
    assert np.array_equal(na, nb), f"{what}: neighbour counts"
    pa, pb = a.energy(), b.energy()
    assert abs(pa[0] - pb[0]) <= stol * abs(pb[0])
    assert abs(pa[2] - pb[2]) <= max(stol, 1e-10) * max(abs(pb[2]), 1e-30)


@pytest.mark.parametrize("evaluation,precision", [("table", "fp64"), ("cheby", "fp64"), ("table", "mixed"), ("cheby", "mixed")])
def test_eam_lists_equal_cells(gpu, cu500, evaluation, precision):
    a, b = pair_of_sims(cu500, 8, 3.615, 600.0, 0.1, 3, evaluation, precision)
    if precision == "mixed":
        b.set_precision("fp64")
    a.force()
    b.force()
    info = a.list_info()
    print(f"[lists] {info}", flush=True)
    assert info["active"] == 1 and info["valid"] == 1 and info["builds"] == 1
    assert b.list_info()["active"] == 0
    # mixed Chebyshev: the value series (phi, rho) are FP32 Clenshaw sums
    # from FP32 coefficients, so energies and densities carry their rounding,
    # amplified by the series' cancellation (per atom about 5e-6 of the FP64
    # energy, the total about 2e-6); forces stay within the 1e-6 bar
    tol = 1e-12 if precision == "fp64" else 1e-6
    stol = 2e-5 if (evaluation, precision) == ("cheby", "mixed") else tol
    assert_same(a, b, f"eam {evaluation} {precision}", tol=tol, stol=stol)


@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("evaluation,precision", [("table", "fp64"), ("cheby", "fp64"), ("table", "mixed")])
def test_lanes_per_atom_equal_cells(gpu, cu500, lanes, evaluation, precision):
    """Small systems default to two lanes per home atom in the list passes
    (COMD_TUNE_LIST_LANES); one and four must give the link-cell results
    too (each lane takes every lanes-th chunk of the atom's list and the
    lanes add their sums)."""
    a, b = pair_of_sims(cu500, 8, 3.615, 600.0, 0.1, 5, evaluation, precision)
    a.tune(list_lanes=lanes)
    if precision == "mixed":
        b.set_precision("fp64")
    a.force()
    b.force()
    assert a.list_info()["active"] == 1 and a.list_info()["valid"] == 1
    assert a.list_lanes() == lanes and b.list_lanes() == 0
    assert_same(a, b, f"eam {evaluation} {precision}, {lanes} lanes", tol=1e-12 if precision == "fp64" else 1e-6)
    a.nsteps(10)
    b.nsteps(10)
    ca, cb = compact(a.download()), compact(b.download())
    assert np.array_equal(ca["id"], cb["id"])
    assert force_rel_error(ca["f"], cb["f"]).max() <= (1e-10 if precision == "fp64" else 5e-5)


def test_lj_lanes_equal_cells(gpu):
    lj = CA.copper_lj()
    for lanes in (1, 2, 4):
        a, b = pair_of_sims(lj, 7, lj.lat, 600.0, 0.05, 6)
        a.force()
        assert a.list_lanes() == 2  # the default below 128 atoms per CU
        a.tune(list_lanes=lanes)
        a.force()
        b.force()
        assert a.list_info()["active"] == 1 and a.list_lanes() == lanes
        assert_same(a, b, f"lj, {lanes} lanes", lj=True)


def test_mixed_lists_after_fp64_steps(gpu, cu500):
    """Steps in FP64 keep only the double list positions current; switching
    to mixed precision must refresh the fixed-point ones."""
    a, b = pair_of_sims(cu500, 7, 3.615, 1500.0, 0.05, 11)
    a.force()
    b.force()
    a.nsteps(15)
    b.nsteps(15)
    a.set_precision("mixed")
    a.force()
    b.force()
    assert a.list_info()["valid"] == 1
    assert_same(a, b, "mixed after fp64 steps", tol=1e-6)
    a.nsteps(5)
    a.set_precision("fp64")
    b.nsteps(5)
    a.force()
    b.force()
    ca, cb = compact(a.download()), compact(b.download())
    assert np.array_equal(ca["id"], cb["id"])
    assert force_rel_error(ca["f"], cb["f"]).max() <= 1e-5


def test_lj_lists_equal_cells(gpu):
    lj = CA.copper_lj()
    a, b = pair_of_sims(lj, 7, lj.lat, 600.0, 0.05, 4)
    a.force()
    b.force()
    assert a.list_info()["active"] == 1
    assert_same(a, b, "lj", lj=True)


def test_trajectory_with_rebuilds(gpu, cu500):
    """3000 K for 40 steps: atoms move well past half the skin, so the lists
    are rebuilt on the device several times; the trajectory must follow the
    link-cell one."""
    a, b = pair_of_sims(cu500, 6, 3.615, 3000.0, 0.05, 9)
    a.force()
    b.force()
    for chunk in range(4):
        pa = a.nsteps(10)
        pb = b.nsteps(10)
        assert abs(pa - pb) <= 1e-9 * abs(pb)
    info = a.list_info()
    print(f"[rebuilds] {info}", flush=True)
    assert info["valid"] == 1 and info["builds"] >= 3
    assert_same(a, b, "after 40 steps at 3000 K", tol=1e-8)


def test_upload_path_sets_up_lists(gpu, cu500):
    a, b = pair_of_sims(cu500, 6, 3.615, 300.0, 0.1, 5)
    st = b.download()
    c = CA.Simulation(cu500, a.bounds, defgrad=0.0)
    c.upload(st["natoms"], st["id"], st["itype"], st["r"], st["p"])
    c.force()
    b.force()
    assert c.list_info()["active"] == 1
    assert_same(c, b, "uploaded state")


@pytest.mark.parametrize("groups,rows,div", [(0, 1, 1), (1, 1, 2), (2, 0, 1), (3, 1, 2), (4, 1, 1), (0, 0, 2)])
@pytest.mark.parametrize("n", [5, 7])
def test_group_options_equal_cells(gpu, cu500, groups, rows, div, n):
    """Every group size (4x4x3 .. 2x2x1 auxiliary cells), table rows in LDS
    or not, one or two home atoms per thread, and boxes of 3 auxiliary cells
    per dimension (n = 5: a group's halo holds the same cell twice, at two
    images): the same pairs and forces as the link-cell kernels."""
    for prec in ("fp64", "mixed"):
        a, b = pair_of_sims(cu500, n, 3.615, 900.0, 0.1, 30 + n, "table", prec)
        a.tune(list_groups=groups, list_rows_lds=rows, list_threads_div=div)
        if prec == "mixed":
            b.set_precision("fp64")
        a.force()
        b.force()
        info = a.list_info()
        assert info["active"] == 1 and info["valid"] == 1, info
        what = f"groups {groups} rows {rows} div {div} n {n} {prec}"
        assert_same(a, b, what, tol=1e-12 if prec == "fp64" else 1e-6)
        a.nsteps(20)
        b.nsteps(20)
        assert_same(a, b, what + ", 20 steps", tol=1e-10 if prec == "fp64" else 1e-5)


def test_overflow_falls_back_to_cells(gpu, cu500):
    """A Cu 8^3 lattice whose slab x < 18 A is squeezed 2.25-fold: the lists
    are set up for the mean density, but the fullest 7.2 A auxiliary cell
    gets 72 atoms, more than the 64 one holds (the fullest 5.8 A link cell
    56).  The build marks the lists invalid and the link-cell passes,
    launched beside the list passes, give the forces -- first with the small
    grid they get while the lists were last seen valid, then with the full
    grid once the host has seen them invalid."""
    xyz, p, bounds = seeded_atoms(8, 3.615, cu500.mass, temp=0.0, disp=0.02, seed=41)
    slab = xyz[:, 0] < 18.0
    xyz[slab, 0] /= 2.25
    out = []
    for skin in (0.4, 0.0):
        s = CA.Simulation(cu500, bounds, defgrad=0.0)
        s.tune(skin=skin)
        s.bin_atoms(xyz, p)
        s.rebox()
        out.append(s)
    a, b = out
    a.force()
    b.force()
    info = a.list_info()
    print(f"[overflow] {info}", flush=True)
    assert info["active"] == 1 and info["valid"] == 0
    assert_same(a, b, "overflow, first force")
    a.nsteps(2)
    b.nsteps(2)
    assert_same(a, b, "overflow, after steps", tol=1e-10)


def test_force_after_replayed_step_graph(gpu, cu500):
    """A force call after steps replayed from an already captured step graph
    (the second steps() call reuses the graph of the first) sees the atoms'
    current positions: each step ends with a drift that leaves the list
    positions stale, whether the step ran eagerly, was captured, or was
    replayed."""
    a, b = pair_of_sims(cu500, 8, 3.615, 600.0, 0.05, 77)
    for chunk in (4, 9, 9):
        for s in (a, b):
            s.steps(chunk)
            s.force()
        assert a.list_info()["active"] == 1
        assert_same(a, b, f"after a {chunk}-step graph chunk", tol=1e-10)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_autotune_tunes_list_passes(gpu, cu500, precision):
    """comd_autotune on a context with lists times the list passes' shapes:
    the choice is applied (lists valid, occupancy reported for it), the
    forces of the state stay those of the link-cell kernels, and steps
    after it follow them."""
    a, b = pair_of_sims(cu500, 12, 3.615, 300.0, 0.05, 91, "table", precision)
    if precision == "mixed":
        b.set_precision("fp64")
    a.force()
    b.force()
    before = a.download()["f"].copy()
    res = a.autotune_lists()
    occ = a.list_occupancy()
    print(f"[autotune lists {precision}] {res} occupancy {occ}", flush=True)
    assert res["ms"] > 0.0 and res["groups"] in range(-1, 5) and res["threads_div"] in (1, 2)
    info = a.list_info()
    assert info["active"] == 1 and info["valid"] == 1
    f = a.download()["f"]
    m = np.abs(before[:, :3]).max()
    assert np.abs(f[:, :3] - before[:, :3]).max() <= (1e-12 if precision == "fp64" else 1e-6) * m
    w, bpc, bal, ms = a.autotune()  # with lists: the same tuner
    assert ms > 0.0
    tol = 1e-12 if precision == "fp64" else 1e-6
    assert_same(a, b, f"autotuned {precision}", tol=tol)
    a.nsteps(10)
    b.nsteps(10)
    assert_same(a, b, f"autotuned {precision}, 10 steps", tol=1e-10 if precision == "fp64" else 1e-5)


@pytest.mark.parametrize("groups,div,precision", [(4, 4, "fp64"), (3, 3, "mixed"), (4, 4, "mixed"), (0, 4, "fp64")])
@pytest.mark.parametrize("n", [5, 9])
def test_halo_tables_of_small_blocks(gpu, cu500, groups, div, precision, n):
    """Blocks with few threads stage many halo entries each, so their halo
    slots take several words per thread; across a rebuild."""
    a, b = pair_of_sims(cu500, n, 3.615, 900.0, 0.1, 17, precision=precision)
    b.set_precision("fp64")
    a.tune(list_groups=groups, list_threads_div=div)
    tol = 1e-12 if precision == "fp64" else 1e-6
    for s in (a, b):
        s.force()
    assert a.list_info()["valid"] == 1
    assert_same(a, b, f"groups {groups} div {div} {precision}", tol=tol)
    for s in (a, b):
        s.nsteps(25)
    assert a.list_info()["builds"] > 1
    if precision == "fp64":  # mixed trajectories differ by their rounding
        assert_same(a, b, "after a rebuild", tol=1e-9)


@pytest.mark.parametrize("per_cell", [1, 6, 10, 11, 18, 21, 30])
def test_runs_of_every_length(gpu, per_cell):
    """Runs of three cells of a few to some ninety atoms (the build tests 32
    at a time, 8 by 8), uneven from cell to cell: the lists hold every pair
    that the link cells find, each once."""
    pot = CA.LJPotential(sigma=0.1, epsilon=1e-12, cutoff=2.0, mass=1.0)
    rng = np.random.default_rng(per_cell)
    bounds = np.array([14.6, 12.2, 10.1])
    xyz = rng.uniform(0.0, 1.0, (int(per_cell * 210), 3)) * bounds
    xyz[:: 3, 0] *= 0.7  # denser on one side
    out = []
    for skin in (0.4, 0.0):
        s = CA.Simulation(pot, bounds)
        s.tune(skin=skin)
        s.bin_atoms(xyz)
        s.force()
        out.append(s)
    a, b = out
    assert a.list_info()["active"] == 1 and b.list_info()["active"] == 0
    # from 21 on an auxiliary cell passes 64 atoms: the link cells take over
    assert a.list_info()["valid"] == (1 if per_cell < 21 else 0)
    m = np.arange(64)[None, :] < a.download()["natoms"][:, None]
    na, nb = (s.download_aux()[0].reshape(-1, 64)[m] for s in out)
    assert np.array_equal(na, nb)
    assert a.pair_count() == b.pair_count()


# (a mixed batch takes smaller auxiliary cells, which hold this box)
@pytest.mark.parametrize("kind,precision", [("table", "fp64"), ("table", "mixed"), ("cheby", "fp64"), ("cheby", "mixed"),
                                            ("lj", "fp64"), ("lj", "mixed"), ("batch", "fp64")])
def test_invalid_lists_inside_and_beside_the_passes(gpu, cu500, kind, precision):
    """Boxes whose auxiliary cells overflow: the link cells' work inside the
    list passes (until the host has seen it) and by their own kernels (after)
    is that of a context without lists."""
    rng = np.random.default_rng(8)
    lj = CA.LJPotential(sigma=1.9, epsilon=1e-4, cutoff=4.95, mass=63.55)
    bounds = np.array([29.0, 27.5, 28.1])
    grid = np.stack(np.meshgrid(*[np.arange(int(b / 1.9)) for b in bounds], indexing="ij"), -1).reshape(-1, 3)
    xyz = (grid + 0.5) * 1.9 + rng.uniform(-0.1, 0.1, grid.shape)  # 0.146 atoms per A^3: some 30 a cell
    close = xyz[:, 0] < 7.0
    xyz = np.concatenate([xyz, xyz[close] + 0.95])  # and twice that in a slab: above 64
    xyz %= bounds

    def make(skin):
        if kind == "batch":
            few = xyz[::9]
            b = CA.Batch([dict(pot=p, bounds=bounds) for p in (cu500, lj, cu500)], precision=precision)
            b.tune(skin=skin)
            for r, x in enumerate((few, few, xyz)):
                b.bin_atoms(r, x)
            return b
        s = CA.Simulation(lj if kind == "lj" else cu500, bounds, precision=precision,
                          evaluation="cheby" if kind == "cheby" else "table")
        s.tune(skin=skin)
        s.bin_atoms(xyz)
        return s

    def state(s):
        parts = [s.download(r) for r in range(s.nrep)] if kind == "batch" else [s.download()]
        parts = [compact(p) for p in parts]
        return [np.concatenate([p[k] for p in parts]) for k in ("f", "rho", "fi")]

    a, b = make(0.4), make(0.0)
    b.force()
    want = state(b)
    for _ in range(2):
        a.force()
        got = state(a)
        assert a.list_info()["active"] == 1 and a.list_info()["valid"] == 0
        for g, w in zip(got, want):
            assert scalar_rel_error(g, w).max() <= 1e-12
        a.sync()  # the host looks


@pytest.mark.parametrize("lanes", [8, 16])
@pytest.mark.parametrize("evaluation,precision", [("table", "fp64"), ("cheby", "fp64"), ("table", "mixed"), ("cheby", "mixed")])
def test_eight_and_sixteen_lanes_equal_one(gpu, cu500, lanes, evaluation, precision):
    """More lanes than an atom's list has chunks, and fewer: the passes give
    the forces of one lane per atom, whose sums run in another order: 1e-12;
    the mixed table passes add 8 pairs' values in single precision before
    they enter the double sums, and which 8 depends on the block size:
    7 x 2^-24 = 4e-7, held to 1e-6."""
    a, b = pair_of_sims(cu500, 8, 3.615, 600.0, 0.1, 5, evaluation, precision)
    b.tune(skin=0.4, list_lanes=1)
    a.tune(list_lanes=lanes)
    for s in (a, b):
        s.force()
        assert s.list_info()["active"] == 1 and s.list_info()["valid"] == 1
    assert a.list_lanes() == lanes and b.list_lanes() == 1
    assert_same(a, b, f"eam {evaluation} {precision}, {lanes} lanes",
                tol=1e-6 if (evaluation, precision) == ("table", "mixed") else 1e-12)


@pytest.mark.parametrize("evaluation,lanes", [("table", 4), ("cheby", 4)])
def test_default_lanes_of_small_systems(gpu, cu500, evaluation, lanes):
    a, _ = pair_of_sims(cu500, 6, 3.615, 600.0, 0.1, 5, evaluation, "fp64")
    a.force()
    assert a.list_lanes() == lanes


@pytest.mark.parametrize("ncheb", [3, 8, 9, 24, 31])
def test_series_sums_of_the_list_passes(gpu, ncheb):
    """The list passes share one basis between the FP64 series of phi, phi'
    and rho where these have one domain; the link cells sum each series by
    itself.  Equal domains and another one for rho; series of several
    lengths.  Both sum n terms of size |c_k| with errors of k^2 2^-53 each
    (the recurrences near the ends of the domain): 1e-12 for n <= 32."""
    for shift in (0.0, 0.37):
        pot = CA.EAMPotential("cu500", ncheb=ncheb)
        pot.cheb_dom[1, 1] += shift
        a, b = pair_of_sims(pot, 6, 3.615, 600.0, 0.1, 7, evaluation="cheby")
        for s in (a, b):
            s.force()
        assert a.list_info()["valid"] == 1
        assert_same(a, b, f"{ncheb} terms, shift {shift}", tol=1e-12)


def test_occupancy_of_small_halos(gpu, cu500):
    """The mixed Chebyshev density pass of a small crystal stages less than
    one wave of the link cells' work takes (the halo alone: 12 bytes a staged
    atom), which its launch can be asked to do: the launch has that much LDS
    at least, in whole 16-byte words, and so reports it."""
    wave = 14192  # density pass: 3 x 288 doubles, 27 shifts, two 24 x 64 queues, counts and stencil; to 16 bytes
    a, _ = pair_of_sims(cu500, 6, 3.615, 300.0, 0.05, 3, "cheby", "mixed")
    a.tune(list_groups=4)  # 2 x 2 x 1 cells, 4 x 4 x 3 staged: 48 cells of some 13 atoms, 9 KB
    a.force()
    occ = a.list_occupancy()
    assert a.list_info()["valid"] == 1
    assert occ["lds_bytes"][0] >= wave and occ["lds_bytes"][0] % 16 == 0
    assert all(b > 0 for b in occ["blocks_per_cu"])


@pytest.mark.parametrize("n,precision", [(6, "fp64"), (10, "fp64"), (10, "mixed"), (20, "fp64")])
@pytest.mark.parametrize("evaluation", ["table", "cheby"])
def test_link_cells_inside_the_passes_of_few_groups(gpu, cu500, n, evaluation, precision):
    """A crystal slab in a box four times as long, whose lists overflow: few
    groups, small blocks, cells without a group's block to each CU.  The link
    cells' work inside the list launches covers every cell (forces of a context
    without lists, as above) and takes no longer than half as much again as the
    link-cell kernels that replace it once the host has seen the lists invalid
    (with the waves of the lists' own shape alone it took two to five times as
    long)."""
    xyz, p, (lx, ly, lz) = seeded_atoms(n, 3.615, 63.55, temp=300.0, disp=0.1, seed=2)

    def make(skin):
        s = CA.Simulation(cu500, (4.0 * lx, ly, lz), defgrad=0.0, precision=precision, evaluation=evaluation)
        s.tune(skin=skin)
        s.bin_atoms(xyz, p)
        s.force()
        return s

    a, b = make(0.4), make(0.0)
    assert a.list_info()["active"] == 1 and a.list_info()["valid"] == 0
    assert_same(a, b, f"slab {n} {evaluation} {precision}")
    a.timing(True)

    def best(passes):
        times = []
        for _ in range(10):
            before = a.timing_read()[0]
            a.force()
            after = a.timing_read()[0]
            times.append(sum(after[k] - before[k] for k in passes))
        return min(times)

    inside = best((CA.K_DENSITY, CA.K_EMBED_FORCE))
    a.sync()  # the host looks
    beside = best((CA.K_CELL_FALLBACK,))
    print(f"[slab {n} {evaluation} {precision}] inside {1e3 * inside:.1f} us, beside {1e3 * beside:.1f} us", flush=True)
    assert beside > 0.0 and inside <= 1.5 * beside


@pytest.mark.parametrize("lists", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [3, 8, 9, 17, 24, 25, 31])
def test_short_series_equal_their_zero_padded_32(gpu, cu500, n, precision, lists):
    """A series of n terms and the one of 32 with zeros behind are the same
    sums: Clenshaw's recurrence starts with exact zeros at those terms, and
    the shared basis adds exact zeros.  So the passes give the same bits, for
    every stride of the series (8, 16, 24, 32) and in both precisions."""
    short = np.ascontiguousarray(cu500.cheb[:3, :n])
    padded = np.zeros((3, 32))
    padded[:, :n] = short
    got = []
    for pot, coef in ((CA.EAMPotential(cu500.name, ncheb=n), short), (cu500, padded)):
        s = pair_of_sims(pot, 6, 3.615, 600.0, 0.1, 7, "cheby", precision)[0 if lists else 1]
        s.set_cheb(coef)
        s.force()
        assert s.list_info()["active"] == lists and (not lists or s.list_info()["valid"] == 1)
        got.append(compact(s.download()))
    for k in ("f", "rho", "fi"):
        assert np.isfinite(got[0][k]).all() and np.array_equal(got[0][k], got[1][k]), k


def clenshaw32_bound(c, a, b, x):
    """What an FP32 Clenshaw sum of the series c on [a, b] at x (arrays), from
    FP32 coefficients, may differ from the exact one: the rounding of each
    term's recurrence (three operations, and the coefficient's own) reaches the
    sum times |U_k(y)| <= k + 1; an argument off by the rounding of its own
    forming (x, a, b to FP32, two additions and a product) and by the 2e-8 A of
    the fixed-point positions, times |S'(y)| <= sum k^2 |c_k|."""
    u = 2.0 ** -24
    n = len(c)
    y = (2.0 * x - a - b) / (b - a)
    d = dd = np.zeros_like(y)
    err = np.zeros_like(y)
    for k in range(n - 1, -1, -1):
        size = np.abs(2.0 * y * d) + np.abs(dd) + np.abs(c[k])
        err = err + (k + 1) * 4.0 * u * size
        d, dd = 2.0 * y * d - dd + c[k], d
    arg = (6.0 * u * (2.0 * np.abs(x) + abs(a) + abs(b)) + 4e-8) / (b - a)
    return err + arg * np.sum(np.arange(n) ** 2 * np.abs(c))


@pytest.mark.parametrize("n", [3, 9, 24, 31])
@pytest.mark.parametrize("shift", [0.0, 0.37])
def test_mixed_series_sums_of_the_list_passes(gpu, n, shift):
    """As test_series_sums_of_the_list_passes in mixed precision: the lists and
    the link cells sum phi and rho in FP32, each within clenshaw32_bound of
    the exact series per pair, and the list passes their eight pairs' values
    too (7 x 2^-24 of them).  So rho differs by twice that times the
    neighbours at most, the energy by half of phi's and F'(rho) times rho's."""
    pot = CA.EAMPotential("cu500", ncheb=n)
    pot.cheb_dom[1, 1] += shift
    a, b = pair_of_sims(pot, 6, 3.615, 600.0, 0.1, 7, "cheby", "mixed")
    for s in (a, b):
        s.force()
    assert a.list_info()["valid"] == 1
    ga, gb = (compact(s.download()) for s in (a, b))
    m = np.arange(64)[None, :] < b.download()["natoms"][:, None]
    nnb = b.download_aux()[0].reshape(-1, 64)[m]
    r = np.linspace(2.0, pot.cutoff, 4000)

    def per_pair(k):
        lo, hi = pot.cheb_dom[k]
        c = pot.cheb[k, :n]
        y = (2.0 * r - lo - hi) / (hi - lo)
        value = np.abs(np.polynomial.chebyshev.chebval(y, c) - 0.5 * c[0]).max()
        return (clenshaw32_bound(c, lo, hi, r) + 8.0 * 2.0 ** -24 * value).max()

    drho = 2.0 * nnb * per_pair(1)
    de = nnb * per_pair(0) + np.abs(gb["fi"]) * drho * 1.01
    err_rho, err_e = np.abs(ga["rho"] - gb["rho"]), np.abs(ga["f"][:, 3] - gb["f"][:, 3])
    print(f"[mixed series {n} {shift}] rho {(err_rho / drho).max():.3f}, energy {(err_e / de).max():.3f} of the bound;"
          f" relative bound rho {(drho / np.abs(gb['rho'])).max():.1e}", flush=True)
    assert (err_rho <= drho).all() and (err_e <= de).all()
