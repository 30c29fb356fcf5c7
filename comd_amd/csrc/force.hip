// force.hip -- link-cell force kernels for gfx950: EAM density + pair force
// + embedding (passes 1 and 2 of src-flat/eam.c:438-660, fused), EAM
// embedding force (pass 3), and Lennard-Jones (src-flat/ljForce.c:89-224).
//
// Compiled with floating-point contraction: the pair sums may differ from
// the reference in the last bits (the parity bar is 1e-10 relative), unlike
// the integrator and the binning, which round exactly as the reference does.
//
// Every kernel is full-shell: each atom sums over all of its neighbours, so
// no atom is written by two waves and nothing needs atomics; the reference's
// half-shell loops (jBox >= iBox, eam.c:494,609) count each pair once and add
// to both atoms, which gives the same sums.
//
// Work mapping.  Each wave owns one home cell at a time (persistent grid,
// cells of a z-slab per XCD so that neighbouring cells are processed under
// the same L2).  The atoms of the 27 stencil cells (the reference's order,
// src-flat/domains.c:419-426, with the duplicates it keeps when a dimension
// has fewer than 3 cells) are staged in the wave's LDS, shifted into the home
// cell's frame.  The lanes are split into S = 64/n_home groups; lane (a, s)
// tests home atom a against halo atoms s, s+S, ... and pushes the accepted
// ones into its own LDS queue.  The queues of one atom are then drained
// round-robin by that atom's S lanes, so the pair arithmetic runs on dense,
// balanced lanes rather than on the ~15% of candidates inside the cutoff.
// The S partial sums of each home atom are added in a fixed order
// (deterministic results).
#include "comd_internal.h"
#include "pair_cell.h"

template <int KIND, int EVAL, int MIXED>
__global__ __launch_bounds__(256) void k_pair(DevState d, PotDev P)
{
    // the neighbour-list kernels did this pass unless their lists are invalid
    if (d.cell_gate && !(*d.cell_gate & CM_NL_INVALID)) return;
    extern __shared__ __align__(16) char lds[];
    const int W = blockDim.x >> 6;
    const int wv = threadIdx.x >> 6;
    const int L = threadIdx.x & 63;
    WaveLds w = carve(lds + wv * wave_lds_bytes(KIND), KIND);

    // ---- cells of this wave: a slab of consecutive cells per XCD (blocks are
    // dispatched round-robin over the 8 XCDs)
    const int nxcd = gridDim.x < 8 ? (int)gridDim.x : 8;
    const int xcd = blockIdx.x % nxcd;
    const int blocks_here = ((int)gridDim.x - xcd + nxcd - 1) / nxcd;
    const int workers = blocks_here * W;
    const int worker = (blockIdx.x / nxcd) * W + wv;
    const int c_begin = (int)((long)d.ncells * xcd / nxcd);
    const int c_end = (int)((long)d.ncells * (xcd + 1) / nxcd);
    for (int c = c_begin + worker; c < c_end; c += workers) pair_cell<KIND, EVAL, MIXED>(d, d.g0, P, w, c, L);
}

// Many replicas in one launch: the cells of all replicas are dealt to the
// waves with a global stride (replicas of different cost are spread evenly
// over the waves); each cell uses its replica's grid and potential.  PASS 1
// runs the EAM density pass or Lennard-Jones, PASS 3 the EAM embedding-force
// pass (Lennard-Jones cells have none).
template <int PASS, int MIXED>
__global__ __launch_bounds__(64) void k_pair_batch(DevState d, const PotDev *pots)
{
    // beside valid neighbour lists there is nothing to do
    if (d.cell_gate && !(*d.cell_gate & CM_NL_INVALID)) return;
    extern __shared__ __align__(16) char lds[];
    const int L = threadIdx.x;
    WaveLds w = carve(lds, PASS == 1 ? CM_KIND_EAM1 : CM_KIND_EAM3);
    for (int c = blockIdx.x; c < d.ncells; c += gridDim.x) {
        const Grid g = d.grids[d.cell_grid[c]];
        const PotDev P = pots[g.pot];
        if (PASS == 1) {
            if (P.kind == COMD_POT_LJ) pair_cell<CM_KIND_LJ, COMD_EVAL_TABLE, MIXED>(d, g, P, w, c, L);
            else if (P.eval == COMD_EVAL_CHEB) pair_cell<CM_KIND_EAM1, COMD_EVAL_CHEB, MIXED>(d, g, P, w, c, L);
            else pair_cell<CM_KIND_EAM1, COMD_EVAL_TABLE, MIXED>(d, g, P, w, c, L);
        } else if (P.kind != COMD_POT_LJ) {
            if (P.eval == COMD_EVAL_CHEB) pair_cell<CM_KIND_EAM3, COMD_EVAL_CHEB, MIXED>(d, g, P, w, c, L);
            else pair_cell<CM_KIND_EAM3, COMD_EVAL_TABLE, MIXED>(d, g, P, w, c, L);
        }
    }
}

// Persistent grids never exceed the blocks that can be resident at once (or
// the last ones would start only when others finish).  The occupancy query
// is made once per kernel and block shape, so that launches made while a
// step is captured into a graph issue nothing else.
template <typename K>
static int resident_blocks(K kern, int threads, size_t lds, int ncu, int *cache)
{
    if (*cache == 0) {
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, lds) != hipSuccess || per_cu < 1)
            per_cu = -1;
        *cache = per_cu;
    }
    return *cache > 0 && ncu > 0 ? *cache * ncu : 1 << 30;
}

template <int KIND, int EVAL, int MIXED>
static void launch3(const DevState &d, const PotDev &P, const ForceCfg &cfg, hipStream_t st)
{
    static int occ[5] = {0, 0, 0, 0, 0};
    const int W = cfg.waves;
    const size_t lds = (size_t)W * wave_lds_bytes(KIND);
    auto kern = k_pair<KIND, EVAL, MIXED>;
    const int cap = resident_blocks(kern, 64 * W, lds, cfg.ncu, &occ[W < 5 ? W : 4]);
    const int blocks = cfg.blocks < cap ? cfg.blocks : cap;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * W), lds, st, d, P);
}

template <int KIND, int EVAL>
static void launch2(const DevState &d, const PotDev &P, int mixed, const ForceCfg &cfg, hipStream_t st)
{
    if (mixed) launch3<KIND, EVAL, 1>(d, P, cfg, st);
    else launch3<KIND, EVAL, 0>(d, P, cfg, st);
}

int cm_force_lds_bytes(const PotDev &P, int kind, int mixed, int waves, int tab_lds)
{
    (void)P;
    (void)mixed;
    (void)tab_lds;
    return waves * wave_lds_bytes(kind);
}

template <int PASS, int MIXED>
static void launch_batch(const DevState &d, const PotDev *pots, const ForceCfg &cfg, hipStream_t st)
{
    static int occ = 0;
    const size_t lds = wave_lds_bytes(PASS == 1 ? CM_KIND_EAM1 : CM_KIND_EAM3);
    auto kern = k_pair_batch<PASS, MIXED>;
    const int cap = resident_blocks(kern, 64, lds, cfg.ncu, &occ);
    const int blocks = cfg.blocks < cap ? cfg.blocks : cap;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64), lds, st, d, pots);
}

void cm_launch_force_batch(const DevState &d, const PotDev *pots, int pass, int mixed, const ForceCfg &cfg,
                           hipStream_t st)
{
    if (pass == 1) {
        if (mixed) launch_batch<1, 1>(d, pots, cfg, st);
        else launch_batch<1, 0>(d, pots, cfg, st);
    } else {
        if (mixed) launch_batch<3, 1>(d, pots, cfg, st);
        else launch_batch<3, 0>(d, pots, cfg, st);
    }
}

void cm_launch_force(const DevState &d, const PotDev &P, int kind, int mixed, const ForceCfg &cfg, hipStream_t st)
{
    if (kind == CM_KIND_LJ) {
        launch2<CM_KIND_LJ, COMD_EVAL_TABLE>(d, P, mixed, cfg, st);
    } else if (P.eval == COMD_EVAL_CHEB) {
        if (kind == CM_KIND_EAM1) launch2<CM_KIND_EAM1, COMD_EVAL_CHEB>(d, P, mixed, cfg, st);
        else launch2<CM_KIND_EAM3, COMD_EVAL_CHEB>(d, P, mixed, cfg, st);
    } else {
        if (kind == CM_KIND_EAM1) launch2<CM_KIND_EAM1, COMD_EVAL_TABLE>(d, P, mixed, cfg, st);
        else launch2<CM_KIND_EAM3, COMD_EVAL_TABLE>(d, P, mixed, cfg, st);
    }
}
