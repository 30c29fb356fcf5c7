// bin_rebox.hip -- atom binning (GPU counting sort) and a parallel, in-place
// emulation of reBoxAll, with the kick/drift that precedes every rebin of the
// position-Verlet step fused in.
//
// reBoxAll (src-flat/domains.c:347-389) scans cells in ascending order; an
// atom that left its cell is appended to the destination (moveAtom,
// domains.c:224-236) and the source's last atom fills the hole, which is
// examined next.  Its result is reproduced without a serial scan:
//   * whether an atom leaves, and where to, depends only on its own r;
//   * the order of departures from cell c depends only on c's own list and
//     on the NUMBER n_low of atoms that arrived from lower-indexed cells
//     before c was scanned (they are appended and never leave again);
//   * arrivals into c come in (source cell, departure rank) order; those
//     from lower cells fill the n_low placeholder positions, those from
//     higher cells are appended after c's scan.
// Only cells that lose or gain atoms change, so the pass works on the list of
// movers and of touched cells (a few per thousand atoms per half step) and
// updates the slot arrays in place.  The argument holds while no arrival
// into a higher-indexed cell would move again in the same pass; k_move flags
// that case for the atom's replica, whose cells the parallel kernels then
// leave alone, and a serial kernel (one block per flagged replica) redoes
// that replica's pass exactly as the reference does.
//
// Fused half drifts.  Inside a multi-step call a step's second half drift and
// rebin (pass A) are followed at once by the next step's first half drift and
// rebin (pass B), with nothing between that reads the state.  The move kernels
// are bound by HBM (4.7 TB/s over the sparse slot rows), so one pass over the
// atoms does the kick and both half drifts: 232 bytes per atom become 160 and
// two launches one.  An atom that stays in pass A gets its position after
// both drifts, and its move in pass B, if any, is recorded with its slot of
// before A; A's gather, which rewrites the slots of the cells A touches,
// renames those records' slots and finds the moves in B of the atoms that
// arrive.  Pass B then scans and gathers its own lists.  When a replica needs
// A's serial replay, its departing atoms still hold the position of between
// the drifts (slot) and are known (leave); the serial kernel moves them, drifts
// them and replays B.  Slot order, positions and flags are those of the two
// passes, bit for bit.  2 048 000 atoms: two move passes of 68 us -> one of
// 100, with one launch of the serial kernel in place of two; a step of 256 000
// atoms FP64 216 -> 190 us, of 864 atoms 62 -> 49 us.
#include "comd_internal.h"
#include "rebox_serial.h"

#define CM_ACAP 64  // arrivals recorded per cell and pass

__device__ static inline void mark_touched(const RebinSet &p, int c)
{
    if (atomicExch(&p.touched[c], 1) == 0) {
        const int i = atomicAdd(p.ntc, 1);
        p.tc[i] = c;
    }
}

// An arrival in dst (above c) that is still outside it is moved again in the
// same pass (it is examined again when dst is scanned).
__device__ __forceinline__ bool hops_again(const Grid &g, int c, int dst, double ax, double ay, double az)
{
    if (dst < c) return false;
    int jx, jy, jz;
    cell_xyz(g, dst, jx, jy, jz);
    double bx, by, bz;
    return hop(g, dst, jx, jy, jz, ax, ay, az, bx, by, bz) >= 0;
}

// The replica's pass (bit 1) or a fused pair's second one (bit 2) is to be
// replayed serially.
__device__ __forceinline__ void request_replay(const DevState &d, const Grid &g, int bit)
{
    atomicOr(&d.mh[g.pot], bit);
    atomicOr(&d.counts[3], 1);
}

struct Mover {
    double x, y, z, px, py, pz;  // position in the destination cell, momentum
    float4 nlr;
    int id, itype;
};

// Records the departure of slot s (cell c) to dst in pass P; the caller sets
// the slot's bit in P.leave.
__device__ __forceinline__ void put_mover(const DevState &d, const RebinSet &P, int c, int s, int dst, const Mover &v)
{
    const int m = atomicAdd(&d.counts[0], 1);  // capacity: one record per slot
    d.mv_slot[m] = s;
    d.mv_id[m] = v.id;
    d.mv_nlr[m] = v.nlr;
    d.mv_itype[m] = v.itype;
    d.mv_rx[m] = v.x;
    d.mv_ry[m] = v.y;
    d.mv_rz[m] = v.z;
    d.mv_px[m] = v.px;
    d.mv_py[m] = v.py;
    d.mv_pz[m] = v.pz;
    d.mvidx[s] = m;
    const int k = atomicAdd(&P.arr_cnt[dst], 1);
    if (k < CM_ACAP) P.arr[dst * CM_ACAP + k] = m;
    mark_touched(P, c);
    mark_touched(P, dst);
}

// ---------------------------------------------------------------------------
// kick (p -= dtk f, src-flat/timestep.c:62-74), drift (r += (dtd p)/rmass,
// timestep.c:76-104) and the per-atom destination of reBoxAll
// (domains.c:356-377) of the atom in slot s of cell c = (ix, iy, iz);
// departing atoms are recorded as movers.  TWO: the kick, both half drifts and
// the destinations of both passes (see above); kick, drift and rebin are then
// taken as 1.
template <int TWO>
__device__ __forceinline__ void move_atom(const DevState &d, const Grid &g, int c, int ix, int iy, int iz, int s,
                                          double dtk, double dtd, int kick, int drift, int rebin)
{
    const double rmass = g.rmass;
    if (TWO) kick = drift = rebin = 1;
    // every load first (the arrays may alias as far as the compiler can
    // tell, so a load after a store would wait for it)
    double x = d.rx[s], y = d.ry[s], z = d.rz[s];
    double px = d.px[s], py = d.py[s], pz = d.pz[s];
    double fx = 0.0, fy = 0.0, fz = 0.0;
    if (kick) {
        fx = d.fx[s];
        fy = d.fy[s];
        fz = d.fz[s];
    }
    const bool upkeep = drift && d.nl_pos;
    float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (upkeep) q = d.nlr[s];  // position at the last build, build position
    if (kick) {
        px = px - dtk * fx;
        py = py - dtk * fy;
        pz = pz - dtk * fz;
        d.px[s] = px;
        d.py[s] = py;
        d.pz[s] = pz;
    }
    double ux = 0.0, uy = 0.0, uz = 0.0;
    if (drift) {
        ux = dtd * px / rmass;
        uy = dtd * py / rmass;
        uz = dtd * pz / rmass;
        x = x + ux;
        y = y + uy;
        z = z + uz;
    }
    double ax = x, ay = y, az = z;
    int dst = -1;  // of pass A
    if (rebin) dst = hop(g, c, ix, iy, iz, x, y, z, ax, ay, az);
    // the position kept in the slot: a departing atom's is its mover record's,
    // the slot's own serves the serial replay alone
    int hx = ix, hy = iy, hz = iz;  // the cell that (wx, wy, wz) is relative to
    double wx = x, wy = y, wz = z;
    if (TWO) {
        if (dst >= 0) cell_xyz(g, dst, hx, hy, hz), wx = ax + ux, wy = ay + uy, wz = az + uz;
        else wx = x + ux, wy = y + uy, wz = z + uz;
    }
    if (drift) {
        const bool first = TWO && dst >= 0;
        d.rx[s] = first ? x : wx;
        d.ry[s] = first ? y : wy;
        d.rz[s] = first ? z : wz;
        if (upkeep) {
            // absolute position for the neighbour lists, and the rebuild
            // request once the atom has moved half the skin (nearest image)
            double cx, cy, cz;
            corner_of(g, hx, hy, hz, cx, cy, cz);
            const double bx = cx + wx, by = cy + wy, bz = cz + wz;
            d.nl_pos[__float_as_int(q.w)] = CmPos{bx, by, bz};
            double ex = bx - q.x, ey = by - q.y, ez = bz - q.z;
            ex -= g.L0 * rint(ex * g.iL0);
            ey -= g.L1 * rint(ey * g.iL1);
            ez -= g.L2 * rint(ez * g.iL2);
            // one request per wave is enough
            const bool far = ex * ex + ey * ey + ez * ez > d.nl_half2;
            const unsigned long long who = __ballot(far);
            if (who != 0 && (int)__ffsll((long long)who) - 1 == (int)(threadIdx.x & 63))
                atomicOr(d.nl_flags, (unsigned)CM_NL_REBUILD);
        }
    }
    if (!rebin) return;
    if (TWO && dst < 0) {
        // stays in pass A; a move of pass B, under its slot of before A
        double bx, by, bz;
        const int dstb = hop(g, c, ix, iy, iz, wx, wy, wz, bx, by, bz);
        if (dstb < 0) return;
        if (hops_again(g, c, dstb, bx, by, bz)) request_replay(d, g, 2);
        put_mover(d, d.rb, c, s, dstb, Mover{bx, by, bz, px, py, pz, d.nlr[s], d.id[s], d.itype[s]});
        atomicOr(&d.rb.leave[c], 1ull << (s - c * CM_SLOTS));
        return;
    }
    if (dst < 0) return;
    if (hops_again(g, c, dst, ax, ay, az)) request_replay(d, g, 1);
    const Mover v = TWO ? Mover{wx, wy, wz, px, py, pz, d.nlr[s], d.id[s], d.itype[s]}
                        : Mover{ax, ay, az, px, py, pz, d.nlr[s], d.id[s], d.itype[s]};
    put_mover(d, d.ra, c, s, dst, v);
    atomicOr(&d.ra.leave[c], 1ull << (s - c * CM_SLOTS));
}

// Any number of replicas: four consecutive global cells per wave, 16 lanes
// each (a cell's atoms beyond 16 taken in further rounds).  Held to 96
// registers for five waves per SIMD instead of four (the 64-replica batch
// step 0.462 -> 0.459 ms).
template <int TWO>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5)))
void k_move(DevState d, double dtk, double dtd, int kick, int drift, int rebin)
{
    const int c = blockIdx.x * 4 + (threadIdx.x >> 4);
    if (c >= d.ncells) return;
    const int n = d.natoms[c];
    if ((threadIdx.x & 15) >= n) return;
    const Grid g = grid_of(d, c);
    int ix, iy, iz;
    cell_xyz(g, c, ix, iy, iz);
    for (int t = threadIdx.x & 15; t < n; t += 16)
        move_atom<TWO>(d, g, c, ix, iy, iz, c * CM_SLOTS + t, dtk, dtd, kick, drift, rebin);
}

// One replica: four cells per wave, 16 lanes each, cell coordinates from the
// 3-D grid (x: groups of four cells).
template <int TWO>
__global__ __launch_bounds__(64) void k_move4(DevState d, double dtk, double dtd, int kick, int drift, int rebin)
{
    const Grid &g = d.g0;
    const int ix = blockIdx.x * 4 + (threadIdx.x >> 4);
    const int iy = blockIdx.y, iz = blockIdx.z;
    if (ix >= g.nbx0) return;
    const int c = ix + g.nbx0 * (iy + g.nbx1 * iz);
    const int n = d.natoms[c];
    for (int t = threadIdx.x & 15; t < n; t += 16)
        move_atom<TWO>(d, g, c, ix, iy, iz, c * CM_SLOTS + t, dtk, dtd, kick, drift, rebin);
}

// The two kernels below are chains of cache misses (the lists were written by
// other XCDs), so what a cell needs is read in as few turns as its addresses
// allow, wanted or not: the cell beside the number of touched cells, then its
// words, arrivals and movers, then the movers' records.  With the scan in
// registers (it ran in LDS, one lane over every slot), the four launches of a
// step: 864 atoms 50.5 -> 48.5 us a step, 32 000 70 -> 66, 48 484 131.7 -> 128,
// 256 000 FP64 152 -> 148.7, 2 048 000 632 -> 629.

// Touched cell i of pass P, read beside their number; -1 past the end.
__device__ __forceinline__ int first_touched(const RebinSet &P, int i)
{
    int c = P.tc[i], n = *P.ntc;
    asm volatile("" : "+v"(c), "+v"(n));  // both loads before the branch
    return __builtin_amdgcn_readfirstlane(i < n ? c : -1);
}

// Per touched cell (one wave each): count arrivals from lower/higher cells,
// then the cell's own swap-with-last scan with n_low never-departing
// placeholders appended, recording each departure's rank and the resulting
// arrangement.  Only departures are walked: the atoms and placeholders beyond
// the shrinking end are where they began, so the element that fills a hole, or
// leaves in its turn, is known from its place (lane L keeps slot L's rank and
// what ends in it).
// second: pass B of a fused pair (P: its lists).  A replica with a flag of the
// pass or an earlier one is left out.
__global__ __launch_bounds__(64) void k_rebox_scan(DevState d, RebinSet P, int second)
{
    const int L = threadIdx.x;
    const int replay = second ? 3 : 1;
    int c = first_touched(P, blockIdx.x);
    if (c < 0) return;
    const int ntc = *P.ntc;
    for (int i = blockIdx.x;;) {
        int rep = d.mh[rep_of(d, c)], n0 = d.natoms[c], na = P.arr_cnt[c];
        unsigned long long leaves = P.leave[c];  // set by k_move per departure
        int m = P.arr[c * CM_ACAP + L], mv = d.mvidx[c * CM_SLOTS + L];
        asm volatile("" : "+v"(rep), "+v"(n0), "+v"(na), "+v"(leaves), "+v"(m), "+v"(mv));
        n0 = __builtin_amdgcn_readfirstlane(n0);
        na = __builtin_amdgcn_readfirstlane(na);
        if (!(__builtin_amdgcn_readfirstlane(rep) & replay)) {  // else replayed serially
            unsigned fl = 0;
            if (na > CM_ACAP) {
                fl |= CM_FLAG_OVERFLOW;
                na = CM_ACAP;
            }
            bool low = false;
            if (L < na) low = d.mv_slot[m] / CM_SLOTS < c;
            unsigned long long left = (unsigned)__builtin_amdgcn_readfirstlane((int)leaves) |
                                      (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(leaves >> 32)) << 32;
            if (n0 < CM_SLOTS) left &= (1ull << n0) - 1;
            const bool leaving = (left >> L) & 1ull;
            const int nlow = __popcll(__ballot(low));
            const int nhigh = na - nlow;
            if (nlow > 0 && n0 + nlow >= CM_SLOTS) fl |= CM_FLAG_OVERFLOW;
            int len = n0 + nlow;
            if (len > 127) len = 127;
            int rank = 0, rk = 0;
            int in = L < n0 ? L : CM_SLOTS + (L - n0);  // what slot L holds at the end
            while (left) {
                const int p = __ffsll((long long)left) - 1;  // the next hole
                left &= left - 1;
                for (int e = p;;) {
                    if (L == e) rank = rk;
                    rk++;
                    len--;
                    if (len == p) break;  // the last one itself
                    if (len < CM_SLOTS && ((left >> len) & 1ull)) {
                        e = len;  // the last one fills the hole and leaves too
                        left &= ~(1ull << e);
                        continue;
                    }
                    if (L == p) in = len < n0 ? len : CM_SLOTS + (len - n0);
                    break;
                }
            }
            if (leaving) d.mv_rank[mv] = rank;
            if (nhigh > 0 && len + nhigh >= CM_SLOTS) fl |= CM_FLAG_OVERFLOW;
            const int keep = len < CM_SLOTS ? len : CM_SLOTS;
            if (L < keep) d.perm[c * CM_SLOTS + L] = (uint8_t)in;
            if (L == 0) {
                d.meta[4 * c + 0] = len;
                d.meta[4 * c + 1] = nlow;
                d.meta[4 * c + 2] = nhigh;
                d.meta[4 * c + 3] = n0;
                if (fl) atomicOr(d.flags, fl);
            }
        }
        i += gridDim.x;
        if (i >= ntc) return;
        c = P.tc[i];
    }
}

// Per touched cell (one wave each, lane = output slot): order the arrivals by
// (source cell, rank), then write survivors and low arrivals in the scanned
// arrangement followed by the high arrivals.  Lane L reads arrival L's record,
// the output lanes take it from there.  All lanes read before any lane
// writes, so the cell is updated in place.  Clears the cell's pass state.
// FIRST: pass A of a fused pair; the moves of pass B by the cell's atoms are
// put under their new slots, and those of its arrivals recorded.
template <int FIRST>
__global__ __launch_bounds__(64) void k_rebox_gather(DevState d, RebinSet P, int second)
{
    __shared__ int sm[2][CM_SLOTS];  // arrivals by low / high order
    const int L = threadIdx.x;
    const int replay = second ? 3 : 1;
    int c = first_touched(P, blockIdx.x);
    if (c < 0) return;
    const int ntc = *P.ntc;
    for (int i = blockIdx.x;;) {
        int rep = d.mh[rep_of(d, c)], len = d.meta[4 * c + 0], nhigh = d.meta[4 * c + 2], na = P.arr_cnt[c];
        int m = P.arr[c * CM_ACAP + L], e = d.perm[c * CM_SLOTS + L];
        unsigned long long leave_b = FIRST ? d.rb.leave[c] : 0ull;
        asm volatile("" : "+v"(rep), "+v"(len), "+v"(nhigh), "+v"(na), "+v"(m), "+v"(e), "+v"(leave_b));
        len = __builtin_amdgcn_readfirstlane(len);
        nhigh = __builtin_amdgcn_readfirstlane(nhigh);
        na = __builtin_amdgcn_readfirstlane(na);
        // cells of a replica whose pass is replayed serially are left as the
        // move kernel left them (the same in every lane)
        const bool serial = (__builtin_amdgcn_readfirstlane(rep) & replay) != 0;
        if (!serial) {
            na = na < CM_ACAP ? na : CM_ACAP;
            const int tot = len + nhigh;
            const int nout = tot < CM_SLOTS ? tot : CM_SLOTS;
            const int keep = len < CM_SLOTS ? len : CM_SLOTS;
            int src = 0, rk = 0;
            Mover in = {};  // arrival L
            if (L < na) {
                src = d.mv_slot[m] / CM_SLOTS;
                rk = d.mv_rank[m];
                in = Mover{d.mv_rx[m], d.mv_ry[m], d.mv_rz[m], d.mv_px[m], d.mv_py[m], d.mv_pz[m],
                           d.mv_nlr[m], d.mv_id[m], d.mv_itype[m]};
            }
            Mover out = {};
            const int own = L < keep && e < CM_SLOTS ? c * CM_SLOTS + e : -1;
            int mb = -1;
            if (own >= 0) {
                if (FIRST && ((leave_b >> e) & 1ull)) mb = d.mvidx[own];
                out = Mover{d.rx[own], d.ry[own], d.rz[own], d.px[own], d.py[own], d.pz[own],
                            d.nlr[own], d.id[own], d.itype[own]};
            }
            bool arrived = false;
            if (na > 0) {
                // rank among arrivals of the same class, by (source cell, rank)
                const bool low = src < c;
                int pos = 0;
                for (int u = 0; u < na; u++) {
                    const int su = __shfl(src, u, 64);
                    const int ru = __shfl(rk, u, 64);
                    const bool lu = su < c;
                    pos += (lu == low) && (su < src || (su == src && ru < rk));
                }
                if (L < na && pos < CM_SLOTS) sm[low ? 0 : 1][pos] = L;
                __syncthreads();
                int from = L;
                if (L < nout && own < 0) {
                    arrived = true;
                    from = L < keep ? sm[0][(e - CM_SLOTS) & (CM_SLOTS - 1)] : sm[1][(L - len) & (CM_SLOTS - 1)];
                }
                auto take = [&](double &o, double v) {
                    v = __shfl(v, from, 64);
                    if (arrived) o = v;
                };
                take(out.x, in.x);
                take(out.y, in.y);
                take(out.z, in.z);
                take(out.px, in.px);
                take(out.py, in.py);
                take(out.pz, in.pz);
                const float qx = __shfl(in.nlr.x, from, 64), qy = __shfl(in.nlr.y, from, 64),
                            qz = __shfl(in.nlr.z, from, 64), qw = __shfl(in.nlr.w, from, 64);
                const int id = __shfl(in.id, from, 64), itype = __shfl(in.itype, from, 64);
                if (arrived) {
                    out.nlr = make_float4(qx, qy, qz, qw);
                    out.id = id;
                    out.itype = itype;
                }
            }
            __syncthreads();  // every lane has read its source before any slot is overwritten
            const int o = c * CM_SLOTS + L;
            if (L < nout) {
                if (d.nl_slot) d.nl_slot[grid_of(d, c).nl_id_base + out.id] = o;
                d.id[o] = out.id;
                d.nlr[o] = out.nlr;
                d.itype[o] = out.itype;
                d.rx[o] = out.x;
                d.ry[o] = out.y;
                d.rz[o] = out.z;
                d.px[o] = out.px;
                d.py[o] = out.py;
                d.pz[o] = out.pz;
            }
            if (L == 0) d.natoms[c] = nout;
            if (FIRST) {
                // pass B: the cell's own movers renamed, its arrivals' found
                if (mb >= 0) {
                    d.mvidx[o] = mb;
                    d.mv_slot[mb] = o;
                }
                const Grid g = grid_of(d, c);
                double bx = 0, by = 0, bz = 0;
                int dstb = -1;
                if (arrived) {
                    int ix, iy, iz;
                    cell_xyz(g, c, ix, iy, iz);
                    dstb = hop(g, c, ix, iy, iz, out.x, out.y, out.z, bx, by, bz);
                }
                const unsigned long long leave = __ballot(mb >= 0 || dstb >= 0);
                if (L == 0) d.rb.leave[c] = leave;
                if (dstb >= 0) {
                    if (hops_again(g, c, dstb, bx, by, bz)) request_replay(d, g, 2);
                    put_mover(d, d.rb, c, o, dstb, Mover{bx, by, bz, out.px, out.py, out.pz, out.nlr, out.id, out.itype});
                }
            }
        }
        if (L == 0) {
            P.arr_cnt[c] = 0;
            P.touched[c] = 0;
            // pass A's replay of a fused pair reads which atoms leave
            if (!(FIRST && serial)) P.leave[c] = 0;
        }
        __syncthreads();
        i += gridDim.x;
        if (i >= ntc) return;
        c = P.tc[i];
    }
}

// fused: after a fused pair of half drifts (dtd: a half drift's time)
__global__ void k_rebox_serial(DevState d, int fused, double dtd)
{
    if (threadIdx.x != 0) return;
    if (blockIdx.x == 0)
        for (int k = 0; k < 4; k++) d.counts[k] = 0;
    replay_replica(d, blockIdx.x, fused, dtd);
}

// ---------------------------------------------------------------------------
// Binning of a flat atom list as the sequence of putAtomInBox calls
// (src-flat/domains.c:237-291): wrap once into [0,L), cell =
// floor(x/boxsize), append.  Stable counting sort: atomic tickets per cell,
// then each cell's entries are ordered by input index.
__device__ static inline bool wrap_bin(const Grid &g, double &x, double &y, double &z, int &cell)
{
    if (x < 0.0) x += g.L0; else if (x >= g.L0) x -= g.L0;
    if (y < 0.0) y += g.L1; else if (y >= g.L1) y -= g.L1;
    if (z < 0.0) z += g.L2; else if (z >= g.L2) z -= g.L2;
    const int ix = (int)floor(x / g.bs0);
    const int iy = (int)floor(y / g.bs1);
    const int iz = (int)floor(z / g.bs2);
    if (ix < 0 || ix >= g.nbx0 || iy < 0 || iy >= g.nbx1 || iz < 0 || iz >= g.nbx2) return false;
    cell = g.cell_base + ix + g.nbx0 * iy + g.nbx0 * g.nbx1 * iz;
    return true;
}

__global__ void k_bin_key(DevState d, Grid g, int n, const double *xyz, int *cnt, int *tmp)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    int cell;
    if (!wrap_bin(g, x, y, z, cell)) {
        atomicOr(d.flags, (unsigned)CM_FLAG_OUTSIDE);
        return;
    }
    const int t = atomicAdd(&cnt[cell], 1);
    if (t < CM_SLOTS) tmp[cell * CM_SLOTS + t] = i;
    else atomicOr(d.flags, (unsigned)CM_FLAG_OVERFLOW);
}

__global__ __launch_bounds__(64) void k_bin_place(DevState d, Grid g, const double *xyz, const double *pxyz,
                                                  int itype, const int *cnt, const int *tmp)
{
    __shared__ int sidx[CM_SLOTS];
    const int c = g.cell_base + blockIdx.x;
    const int t = threadIdx.x;
    int n = cnt[c];
    if (n > CM_SLOTS) n = CM_SLOTS;
    if (t < n) sidx[t] = tmp[c * CM_SLOTS + t];
    __syncthreads();
    if (t == 0) d.natoms[c] = n;
    if (t >= n) return;
    const int me = sidx[t];
    int rank = 0;
    for (int u = 0; u < n; u++) rank += (sidx[u] < me);
    double x = xyz[3 * me], y = xyz[3 * me + 1], z = xyz[3 * me + 2];
    int cell;
    wrap_bin(g, x, y, z, cell);
    double cx, cy, cz;
    cell_corner(g, c, cx, cy, cz);
    const int s = c * CM_SLOTS + rank;
    d.id[s] = me;
    d.itype[s] = itype;
    d.rx[s] = x - cx;
    d.ry[s] = y - cy;
    d.rz[s] = z - cz;
    d.px[s] = pxyz ? pxyz[3 * me] : 0.0;
    d.py[s] = pxyz ? pxyz[3 * me + 1] : 0.0;
    d.pz[s] = pxyz ? pxyz[3 * me + 2] : 0.0;
}

__global__ void k_fill_int(int *p, int v, long n)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// ---------------------------------------------------------------------------
// host launchers

template <int TWO>
static void launch_move(const DevState &d, hipStream_t st, double dtk, double dtd, int kick, int drift, int rebin)
{
    if (d.ngrids == 1 && d.g0.cell_base == 0) {
        const dim3 grid((unsigned)((d.g0.nbx0 + 3) / 4), (unsigned)d.g0.nbx1, (unsigned)d.g0.nbx2);
        hipLaunchKernelGGL(k_move4<TWO>, grid, dim3(64), 0, st, d, dtk, dtd, kick, drift, rebin);
    } else {
        hipLaunchKernelGGL(k_move<TWO>, dim3((d.ncells + 3) / 4), dim3(64), 0, st, d, dtk, dtd, kick, drift, rebin);
    }
}

void cm_launch_move(const DevState &d, hipStream_t st, double dtk, double dtd, int kick, int drift, int rebin)
{
    launch_move<0>(d, st, dtk, dtd, kick, drift, rebin);
}

static int scan_blocks(const DevState &d) { return d.ncells < 8192 ? d.ncells : 8192; }
static int gather_blocks(const DevState &d) { return d.ncells < 4096 ? d.ncells : 4096; }

void cm_launch_rebox(const DevState &d, hipStream_t st)
{
    hipLaunchKernelGGL(k_rebox_scan, dim3(scan_blocks(d)), dim3(64), 0, st, d, d.ra, 0);
    hipLaunchKernelGGL(k_rebox_gather<0>, dim3(gather_blocks(d)), dim3(64), 0, st, d, d.ra, 0);
    hipLaunchKernelGGL(k_rebox_serial, dim3((unsigned)d.ngrids), dim3(64), 0, st, d, 0, 0.0);
}

void cm_launch_move_two(const DevState &d, hipStream_t st, double dtk, double dtd, int serial)
{
    launch_move<1>(d, st, dtk, dtd, 1, 1, 1);
    hipLaunchKernelGGL(k_rebox_scan, dim3(scan_blocks(d)), dim3(64), 0, st, d, d.ra, 0);
    hipLaunchKernelGGL(k_rebox_gather<1>, dim3(gather_blocks(d)), dim3(64), 0, st, d, d.ra, 0);
    hipLaunchKernelGGL(k_rebox_scan, dim3(scan_blocks(d)), dim3(64), 0, st, d, d.rb, 1);
    hipLaunchKernelGGL(k_rebox_gather<0>, dim3(gather_blocks(d)), dim3(64), 0, st, d, d.rb, 1);
    if (serial) hipLaunchKernelGGL(k_rebox_serial, dim3((unsigned)d.ngrids), dim3(64), 0, st, d, 1, dtd);
}

void cm_launch_fill_int(int *p, int v, long n, hipStream_t st)
{
    long blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_fill_int, dim3((unsigned)blocks), dim3(256), 0, st, p, v, n);
}

void cm_launch_bin(const DevState &d, const Grid &g, hipStream_t st, int n, const double *xyz, const double *pxyz,
                   int itype, int *cnt, int *tmp)
{
    cm_launch_fill_int(cnt + g.cell_base, 0, g.ncells, st);
    if (n > 0) hipLaunchKernelGGL(k_bin_key, dim3((n + 255) / 256), dim3(256), 0, st, d, g, n, xyz, cnt, tmp);
    hipLaunchKernelGGL(k_bin_place, dim3(g.ncells), dim3(64), 0, st, d, g, xyz, pxyz, itype, cnt, tmp);
}
