"""CPU model of the fused pair of half drifts (comd_amd/csrc/bin_rebox.hip)
against the oracle's reBoxAll run twice with a drift between: every atom's
two moves are found in one pass over the atoms; a move of the second pass is
recorded under the atom's slot of before the first, whose gather renames it;
and the serial replay of a first pass that needs it, from the positions of
before the second drift that departing atoms keep in their slots."""
import numpy as np
import pytest

import oracle_py as O
from helpers import POTS
from test_rebox_model import M, destination


def layout(natoms, dest):
    """One pass: dest maps slots to cells.  Returns the new counts and, for
    the touched cells, the old slot of each new one."""
    arrivals, touched, rank, perm = {}, set(), {}, {}
    for s in sorted(dest):
        arrivals.setdefault(dest[s], []).append(s)
        touched |= {dest[s], s // M}
    for c in touched:
        nlow = sum(1 for s in arrivals.get(c, []) if s // M < c)
        lst = [c * M + i for i in range(natoms[c])] + [-1 - k for k in range(nlow)]  # -1 - k: the k-th low arrival
        k = rk = 0
        while k < len(lst):
            if lst[k] in dest:
                rank[lst[k]] = rk
                rk += 1
                lst[k] = lst[-1]
                lst.pop()
            else:
                k += 1
        perm[c] = lst
    new = natoms.copy()
    out = {}
    for c in touched:
        arr = sorted(arrivals.get(c, []), key=lambda s: (s // M, rank[s]))
        low = [s for s in arr if s // M < c]
        out[c] = [low[-1 - s] if s < 0 else s for s in perm[c]] + [s for s in arr if s // M > c]
        new[c] = len(out[c])
    return new, out


def hops_again(rn, d, c, nbx, bs, periodic):
    return d > c and destination(rn, d, nbx, bs, periodic)[0] >= 0


def plain_serial(natoms, ids, r, nbx, bs, periodic):
    """reBoxAll as serial_pass<0> runs it."""
    for c in range(len(natoms)):
        i = 0
        while i < natoms[c]:
            o = c * M + i
            j, rn = destination(r[o], c, nbx, bs, periodic)
            if j < 0:
                i += 1
                continue
            t = j * M + natoms[j]
            ids[t], r[t] = ids[o], rn
            natoms[j] += 1
            natoms[c] -= 1
            if natoms[c] > i:
                last = c * M + natoms[c]
                ids[o], r[o] = ids[last], r[last]


def fused(st, u, nbx, bs, periodic):
    """u: the drift of an atom id between the passes (added twice in all)."""
    natoms, ids, r = st["natoms"].copy(), st["id"].copy(), st["r"].copy()
    ncells = len(natoms)
    dest_a, dest_b, two, flags = {}, {}, {}, 0  # two: position in its cell after the passes' drifts
    for c in range(ncells):
        for i in range(natoms[c]):
            s = c * M + i
            x = r[s] + u[ids[s]]
            d, rn = destination(x, c, nbx, bs, periodic)
            if d < 0:
                r[s] = x + u[ids[s]]
                db, rb = destination(r[s], c, nbx, bs, periodic)
                if db >= 0:
                    dest_b[s] = db
                    flags |= 2 * hops_again(rb, db, c, nbx, bs, periodic)
            else:
                r[s] = x
                dest_a[s] = d
                two[s] = np.array(rn) + u[ids[s]]
                flags |= hops_again(rn, d, c, nbx, bs, periodic)
    if flags & 1:
        leave = {s: True for s in dest_a}
        for c in range(ncells):
            i = 0
            while i < natoms[c]:
                o = c * M + i
                if not leave.get(o):
                    i += 1
                    continue
                j, rn = destination(r[o], c, nbx, bs, periodic)
                if j < 0:
                    r[o] = r[o] + u[ids[o]]
                    i += 1
                    continue
                t = j * M + natoms[j]
                ids[t], r[t] = ids[o], rn
                natoms[j] += 1
                if j > c:
                    leave[t] = True
                else:
                    r[t] = r[t] + u[ids[t]]
                natoms[c] -= 1
                last = c * M + natoms[c]
                if natoms[c] > i:
                    ids[o], r[o] = ids[last], r[last]
                    if not leave.get(last):
                        leave[o] = False
                    leave[last] = False
                else:
                    leave[o] = False
            for i in range(M):
                leave[c * M + i] = False
    else:
        new, cells = layout(natoms, dest_a)
        ids0, r0, old_b = ids.copy(), r.copy(), dict(dest_b)
        for c, srcs in cells.items():
            for i in range(M):
                dest_b.pop(c * M + i, None)
        for c, srcs in cells.items():
            for k, s in enumerate(srcs):
                o = c * M + k
                ids[o] = ids0[s]
                if s // M == c:
                    r[o] = r0[s]
                    if s in old_b:
                        dest_b[o] = old_b[s]
                else:
                    r[o] = two[s]
                    db, rb = destination(r[o], c, nbx, bs, periodic)
                    if db >= 0:
                        dest_b[o] = db
                        flags |= 2 * hops_again(rb, db, c, nbx, bs, periodic)
        natoms = new
    if flags:
        plain_serial(natoms, ids, r, nbx, bs, periodic)
    else:
        new, cells = layout(natoms, dest_b)
        ids0, r0 = ids.copy(), r.copy()
        for c, srcs in cells.items():
            for k, s in enumerate(srcs):
                o = c * M + k
                ids[o] = ids0[s]
                r[o] = r0[s] if s // M == c else destination(r0[s], s // M, nbx, bs, periodic)[1]
        natoms = new
    return natoms, ids, r, flags


@pytest.mark.parametrize("hop,expect", [(0.02, 0), (0.2, 0), (0.45, 0), (0.8, None), (1.2, None), (2.4, None)])
@pytest.mark.parametrize("seed", range(5))
def test_fused_model_equals_two_passes(seed, hop, expect):
    rng = np.random.default_rng(40 + seed)
    pot = O.OraclePot.eam(POTS, "cu500")
    n = int(rng.integers(3, 7))
    L = n * 3.615
    sim = O.OracleSim.from_atoms(pot, (L, L, L), rng.uniform(0, L, size=(4 * n ** 3, 3)))
    info = sim.info()
    nbx, bs = info["nbx"], np.array(info["boxsize"])
    st = sim.state()
    u = np.zeros((st["id"].max() + 1, 3))
    moving = rng.uniform(size=len(u)) < 0.5
    u[moving] = rng.uniform(-hop, hop, size=(moving.sum(), 3)) * bs

    def drift(s):
        m = (np.arange(M)[None, :] < s["natoms"][:, None]).reshape(-1)
        s["r"][m] = s["r"][m] + u[s["id"][m]]
        sim.set_state(s)
        sim.rebox()

    natoms, ids, r, flags = fused(st, u, nbx, bs, True)
    drift(st)
    drift(sim.state())
    got = sim.state()
    assert expect is None or flags == expect
    assert np.array_equal(got["natoms"], natoms)
    m = (np.arange(M)[None, :] < natoms[:, None]).reshape(-1)
    assert np.array_equal(got["id"][m], ids[m])
    assert np.array_equal(got["r"][m], r[m])


def test_replay_of_the_second_pass_alone():
    """Atoms of the second cells in x that go down 1.6 cells per drift: lower
    cells first (not examined again), then across the boundary into higher
    ones, still outside."""
    rng = np.random.default_rng(9)
    pot = O.OraclePot.eam(POTS, "cu500")
    L = 6 * 3.615
    sim = O.OracleSim.from_atoms(pot, (L, L, L), rng.uniform(0, L, size=(864, 3)))
    info = sim.info()
    nbx, bs = info["nbx"], np.array(info["boxsize"])
    st = sim.state()
    u = np.zeros((864, 3))
    for c in range(len(st["natoms"])):
        if c % nbx[0] == 1 and st["natoms"][c] > 1:
            u[st["id"][c * M + 1], 0] = -1.6 * bs[0]
    natoms, ids, r, flags = fused(st, u, nbx, bs, True)
    assert flags == 2
    for _ in range(2):
        m = (np.arange(M)[None, :] < st["natoms"][:, None]).reshape(-1)
        st["r"][m] = st["r"][m] + u[st["id"][m]]
        sim.set_state(st)
        sim.rebox()
        st = sim.state()
    m = (np.arange(M)[None, :] < natoms[:, None]).reshape(-1)
    assert np.array_equal(st["natoms"], natoms) and np.array_equal(st["id"][m], ids[m])
    assert np.array_equal(st["r"][m], r[m])


def scan_by_slots(n0, nlow, leaves):
    """The reference's scan of one cell: rank of each departure, and what is
    in each slot at the end (64 and up: the low arrivals)."""
    perm = list(range(n0)) + [M + k for k in range(nlow)]
    rank, p, n = {}, 0, n0 + nlow
    while p < n:
        e = perm[p]
        if e < M and e in leaves:
            rank[e] = len(rank)
            n -= 1
            perm[p] = perm[n]
        else:
            p += 1
    return rank, perm[:n]


def scan_by_departures(n0, nlow, leaves):
    """The same, walking the departures alone (k_rebox_scan)."""
    left, rank, n = sorted(leaves), {}, n0 + nlow
    perm = [k if k < n0 else M + k - n0 for k in range(n)]
    while left:
        p = e = left.pop(0)
        while True:
            rank[e] = len(rank)
            n -= 1
            if n == p:
                break
            if n in left:
                e = n
                left.remove(n)
                continue
            perm[p] = n if n < n0 else M + n - n0
            break
    return rank, perm[:n]


def test_scan_by_departures_equals_scan_by_slots():
    rng = np.random.default_rng(3)
    for _ in range(4000):
        n0, nlow = int(rng.integers(0, M + 1)), int(rng.choice([0, 0, 1, 2, 5, 20, 64]))
        k = int(rng.integers(0, n0 + 1)) if rng.uniform() < 0.5 else min(n0, int(rng.integers(0, 4)))
        leaves = set(rng.permutation(n0)[:k].tolist())
        assert scan_by_slots(n0, nlow, leaves) == scan_by_departures(n0, nlow, leaves)
