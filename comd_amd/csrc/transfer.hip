// transfer.hip -- the device's structure-of-arrays state to and from the
// reference's slot arrays (r, p: 3 doubles per slot, f: 4), interleaved on
// the device.
//
// Bound by PCIe (57 GB/s from pinned memory on this part's host), then by
// the host's own copy out of the staging buffer.  The kernels read and write
// the pinned staging buffer directly: one launch packs every field of a
// chunk of cells, with no device copy of the interleaved form and one
// synchronisation per chunk.  Before, each component was copied to pageable
// memory by itself and interleaved by a strided loop on the host: r, p and
// ids of 2 048 000 atoms (12.5 M slots, 650 MB) took 128 ms, of 864 atoms
// 0.23 ms; now 13.4 ms and 0.03 ms (api.hip, transfer).
#include "comd_internal.h"

#define XF_BLOCK 256

template <int N>
__device__ __forceinline__ const double *comp(const double *a, const double *b, const double *c, const double *d, int k)
{
    return k == 0 ? a : k == 1 ? b : (N == 3 || k == 2) ? c : d;
}

// N interleaved components: lane q writes value q of the field, so that the
// stores over PCIe are whole lines.
template <int N>
__device__ __forceinline__ void pack_field(double *out, const double *a, const double *b, const double *c,
                                           const double *d, long s0, int ns)
{
    const int n = ns * N;  // at most a chunk's 8 MB
    for (int q = blockIdx.x * XF_BLOCK + threadIdx.x; q < n; q += gridDim.x * XF_BLOCK)
        out[q] = comp<N>(a, b, c, d, q % N)[s0 + q / N];
}

template <class T>
__device__ __forceinline__ void copy_field(T *out, const T *in, int n)
{
    for (int q = blockIdx.x * XF_BLOCK + threadIdx.x; q < n; q += gridDim.x * XF_BLOCK) out[q] = in[q];
}

__global__ __launch_bounds__(XF_BLOCK) void k_pack(DevState d, CmSlots h, int c0, int nc)
{
    const long s0 = (long)c0 * CM_SLOTS;
    const int ns = nc * CM_SLOTS;
    if (h.natoms) copy_field(h.natoms, (const int *)d.natoms + c0, nc);
    if (h.id) copy_field(h.id, (const int *)d.id + s0, ns);
    if (h.itype) copy_field(h.itype, (const int *)d.itype + s0, ns);
    if (h.r) pack_field<3>(h.r, d.rx, d.ry, d.rz, nullptr, s0, ns);
    if (h.p) pack_field<3>(h.p, d.px, d.py, d.pz, nullptr, s0, ns);
    if (h.f) pack_field<4>(h.f, d.fx, d.fy, d.fz, d.fe, s0, ns);
    if (h.rho) copy_field(h.rho, (const double *)d.rho + s0, ns);
    if (h.fi) copy_field(h.fi, (const double *)d.fi + s0, ns);
}

// A chunk of slots into the moving state; a field not given (itype, p) is
// set to zero.
__global__ __launch_bounds__(XF_BLOCK) void k_unpack(DevState d, CmSlots h, int c0, int nc)
{
    const long s0 = (long)c0 * CM_SLOTS;
    const int ns = nc * CM_SLOTS;
    copy_field(d.natoms + c0, (const int *)h.natoms, nc);
    copy_field(d.id + s0, (const int *)h.id, ns);
    for (int q = blockIdx.x * XF_BLOCK + threadIdx.x; q < ns; q += gridDim.x * XF_BLOCK)
        d.itype[s0 + q] = h.itype ? h.itype[q] : 0;
    for (int q = blockIdx.x * XF_BLOCK + threadIdx.x; q < 3 * ns; q += gridDim.x * XF_BLOCK) {
        const int k = q % 3;
        const long s = s0 + q / 3;
        (k == 0 ? d.rx : k == 1 ? d.ry : d.rz)[s] = h.r[q];
        (k == 0 ? d.px : k == 1 ? d.py : d.pz)[s] = h.p ? h.p[q] : 0.0;
    }
}

// Blocks of a chunk: a few waves per CU keep the link busy; no more blocks
// than the widest field has work for.
static unsigned xfer_blocks(int nc)
{
    const int b = (nc * CM_SLOTS * 3 + XF_BLOCK - 1) / XF_BLOCK;
    return (unsigned)(b < 512 ? b : 512);
}

void cm_launch_pack(const DevState &d, const CmSlots &h, int c0, int nc, hipStream_t st)
{
    hipLaunchKernelGGL(k_pack, dim3(xfer_blocks(nc)), dim3(XF_BLOCK), 0, st, d, h, c0, nc);
}

void cm_launch_unpack(const DevState &d, const CmSlots &h, int c0, int nc, hipStream_t st)
{
    hipLaunchKernelGGL(k_unpack, dim3(xfer_blocks(nc)), dim3(XF_BLOCK), 0, st, d, h, c0, nc);
}
