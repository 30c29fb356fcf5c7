// rebox_serial.h -- the serial replay of reBoxAll (src-flat/domains.c:347-389)
// for replicas whose parallel pass would not give the reference's order.  One
// thread per replica; run by a kernel of its own or, inside a multi-step call,
// by the first kernel of the list check that follows the rebin.
#pragma once

#include "comd_internal.h"

// Destination cell of an atom of cell c = (ix, iy, iz) at (x, y, z) by the
// rules of reBoxAll (domains.c:356-377), -1 when it stays, and its position
// in that cell.
__device__ __forceinline__ int hop(const Grid &g, int c, int ix, int iy, int iz, double x, double y, double z,
                                   double &ax, double &ay, double &az)
{
#pragma clang fp contract(off)
    int nx = ix, ny = iy, nz = iz;
    ax = x;
    ay = y;
    az = z;
    if (x < 0.0) { nx = ix - 1; ax = x + g.bs0; } else if (x >= g.bs0) { nx = ix + 1; ax = x - g.bs0; }
    if (y < 0.0) { ny = iy - 1; ay = y + g.bs1; } else if (y >= g.bs1) { ny = iy + 1; ay = y - g.bs1; }
    if (z < 0.0) { nz = iz - 1; az = z + g.bs2; } else if (z >= g.bs2) { nz = iz + 1; az = z - g.bs2; }
    const int j = cell_wrap(g, nx, ny, nz);
    return j == c ? -1 : j;
}

// Serial pass of the replicas in which k_move found an arrival that would
// move again (one block each, its first thread walking the replica's cells):
// reBoxAll exactly as the reference runs it, in place. 
__device__ static void serial_copy(const DevState &d, int from, int to)
{
    if (d.nl_slot) d.nl_slot[grid_of(d, to / CM_SLOTS).nl_id_base + d.id[from]] = to;
    d.id[to] = d.id[from];
    d.nlr[to] = d.nlr[from];
    d.itype[to] = d.itype[from];
    d.rx[to] = d.rx[from];
    d.ry[to] = d.ry[from];
    d.rz[to] = d.rz[from];
    d.px[to] = d.px[from];
    d.py[to] = d.py[from];
    d.pz[to] = d.pz[from];
}

// One pass over the cells of grid g.  FIRST: pass A of a fused pair: the atoms
// of ra.leave hold their position of before the second drift and are
// examined, with their arrivals in cells yet to come; each is drifted (by dtd)
// where it ends.  The others have moved on already and stay.
template <int FIRST>
__device__ static unsigned serial_pass(const DevState &d, const Grid &g, double dtd)
{
#pragma clang fp contract(off)
    unsigned fl = 0;
    unsigned long long *leave = d.ra.leave;
    auto settle = [&](int s, int ix, int iy, int iz) {
#pragma clang fp contract(off)
        double x = d.rx[s], y = d.ry[s], z = d.rz[s];
        x = x + dtd * d.px[s] / g.rmass;
        y = y + dtd * d.py[s] / g.rmass;
        z = z + dtd * d.pz[s] / g.rmass;
        d.rx[s] = x;
        d.ry[s] = y;
        d.rz[s] = z;
        if (d.nl_pos) {
            double cx, cy, cz;
            corner_of(g, ix, iy, iz, cx, cy, cz);
            d.nl_pos[__float_as_int(d.nlr[s].w)] = CmPos{cx + x, cy + y, cz + z};
        }
    };
    for (int c = g.cell_base; c < g.cell_base + g.ncells; c++) {
        int ix, iy, iz;
        cell_xyz(g, c, ix, iy, iz);
        int i = 0;
        while (i < d.natoms[c]) {
            const int o = c * CM_SLOTS + i;
            if (FIRST && !((leave[c] >> i) & 1ull)) {
                i++;
                continue;
            }
            double ax, ay, az;
            const int j = hop(g, c, ix, iy, iz, d.rx[o], d.ry[o], d.rz[o], ax, ay, az);
            if (j < 0) {
                if (FIRST) settle(o, ix, iy, iz);
                i++;
                continue;
            }
            d.rx[o] = ax;
            d.ry[o] = ay;
            d.rz[o] = az;
            const int nj = d.natoms[j];
            if (nj >= CM_SLOTS) {  // no room: the reference aborts here
                fl |= CM_FLAG_OVERFLOW;
                i++;
                continue;
            }
            const int t = j * CM_SLOTS + nj;
            serial_copy(d, o, t);
            d.natoms[j] = nj + 1;
            if (nj + 1 >= CM_SLOTS) fl |= CM_FLAG_OVERFLOW;
            if (FIRST) {
                if (j > c) {
                    leave[j] |= 1ull << nj;  // examined when its cell is
                } else {
                    int jx, jy, jz;
                    cell_xyz(g, j, jx, jy, jz);
                    settle(t, jx, jy, jz);
                }
            }
            // the cell's last atom fills the hole; none to move when the
            // departed atom was the last (a self-copy would point its id ->
            // slot entry back at the slot it left)
            const int ni = --d.natoms[c];
            if (ni > i) {
                serial_copy(d, c * CM_SLOTS + ni, o);
                if (FIRST && !((leave[c] >> ni) & 1ull)) leave[c] &= ~(1ull << i);
            }
            if (FIRST && ni < CM_SLOTS) leave[c] &= ~(ni > i ? 1ull << ni : 1ull << i);
        }
        if (FIRST) leave[c] = 0;
    }
    return fl;
}

// Replays replica r's passes if they asked for it.  fused: after a fused pair
// of half drifts (dtd: a half drift's time).
__device__ static void replay_replica(const DevState &d, int r, int fused, double dtd)
{
    const int mh = d.mh[r];
    if (!mh) return;
    const Grid g = d.ngrids == 1 ? d.g0 : d.grids[r];
    unsigned fl = 0;
    if (fused && (mh & 1)) fl |= serial_pass<1>(d, g, dtd);
    fl |= serial_pass<0>(d, g, 0.0);
    d.mh[r] = 0;
    if (fl) atomicOr(d.flags, fl);
}
