// ws_ghost.h -- index arithmetic of the ghosted box, the periodic face halo and the RHS's
// inputs, shared by the helper kernels and the one-launch RHS.
#pragma once

#include <hip/hip_runtime.h>

#include "ws_device.h"

namespace ws {

namespace {

struct FieldList {
    ws_field f[8];
};

// Cell i of nx x ny x nz cells, x fastest.  A 64-bit division by a run-time extent costs an
// order more instructions than a 32-bit one, enough to keep these kernels from the memory's
// rate, and only a box past 2^32 cells needs it (a uniform branch on `total`, its cells).
__device__ __forceinline__ void cell_xyz(long i, long total, int nx, int ny, int &x, int &y, int &z)
{
    if (total <= 0xffffffffL) {
        const uint32_t q = (uint32_t)i / (uint32_t)nx;
        x = (int)((uint32_t)i - q * (uint32_t)nx);
        z = (int)(q / (uint32_t)ny);
        y = (int)(q - (uint32_t)z * (uint32_t)ny);
    } else {
        x = (int)(i % nx);
        y = (int)((i / nx) % ny);
        z = (int)(i / ((long)nx * ny));
    }
}

// Periodic LAP-deep face halo of the periodic directions.  Linear index over the face
// slabs of one field:
// x slabs (2*LAP*ny*nz), y slabs (2*LAP*nx*nz), z slabs (2*LAP*nx*ny).
// Ghost points read only interior points, so the three directions need no ordering.
// The ghost point dst of index i and the interior point src it copies; false: none.
struct GhostPoint {
    int dx, dy, dz, sx, sy, sz;
};

__device__ __forceinline__ bool ghost_point(int nx, int ny, int nz, bool px, bool py, bool pz, long i, GhostPoint &q)
{
    // slabs of non-periodic directions are left to the caller
    const long nxs = px ? 2L * LAP * ny * nz : 0, nys = py ? 2L * LAP * nx * nz : 0;
    const long nzs = pz ? 2L * LAP * nx * ny : 0;
    const long total = nxs + nys + nzs;
    if (i < nxs) {
        int g, y, z;
        cell_xyz(i, total, 2 * LAP, ny, g, y, z);      // g: 0..3 left ghosts, 4..7 right ghosts
        q.dy = q.sy = y + LAP; q.dz = q.sz = z + LAP;
        if (g < LAP) { q.dx = g;                q.sx = nx + g; }           // [0,4) <- [nx, nx+4)
        else         { q.dx = nx + LAP + g - LAP; q.sx = g; }               // [nx+4, nx+8) <- [4, 8)
    } else if ((i -= nxs) < nys) {
        int x, g, z;
        cell_xyz(i, total, nx, 2 * LAP, x, g, z);
        q.dx = q.sx = x + LAP; q.dz = q.sz = z + LAP;
        if (g < LAP) { q.dy = g;                q.sy = ny + g; }
        else         { q.dy = ny + g;           q.sy = g; }
    } else if ((i -= nys) < nzs) {
        int x, y, g;
        cell_xyz(i, total, nx, ny, x, y, g);
        q.dx = q.sx = x + LAP; q.dy = q.sy = y + LAP;
        if (g < LAP) { q.dz = g;                q.sz = nz + g; }
        else         { q.dz = nz + g;           q.sz = g; }
    } else {
        return false;
    }
    return true;
}

// The ghost point of n fields (at most NF): every field's load goes out before the first store.
template <int NF>
__device__ __forceinline__ void ghost_copy(const ws_field *f, int n, int nyg, const GhostPoint &q, double (&val)[NF])
{
#pragma unroll
    for (int j = 0; j < NF; ++j)
        if (j < n) val[j] = f[j].ptr[fidx(f[j].pitch, nyg, q.sx, q.sy, q.sz)];
#pragma unroll
    for (int j = 0; j < NF; ++j)
        if (j < n) f[j].ptr[fidx(f[j].pitch, nyg, q.dx, q.dy, q.dz)] = val[j];
}

// The RHS's inputs from the interior primitives, PER points of the ghosted box per thread, i0,
// i0 + NT, ...:
// beside a periodic face the ghost point of d, u, v, w and T (as k_ghost_fill), and
// everywhere the sound speed of the T that the point then holds (as k_sound_speed).  Writes no
// point it reads, so one launch does what a ghost fill and a pass over T did.
template <int PER, int NT>
__device__ __forceinline__ void prepare_points(const FieldList &fl, const ws_field &cc, int nx, int ny, int nz, int px,
                                               int py, int pz, double ama, long i0)
{
#pragma clang fp contract(off)
    const int nxg = nx + 2 * LAP, nyg = ny + 2 * LAP;
    const long total = (long)nxg * nyg * (nz + 2 * LAP);
    const ws_field &fT = fl.f[4];
    GhostPoint q[PER];
    bool ghost[PER];
    double T[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        // past the end: the last point again, not written
        GhostPoint &p = q[r];
        cell_xyz(min(i0 + r * NT, total - 1), total, nxg, nyg, p.dx, p.dy, p.dz);
        const bool ox = p.dx < LAP || p.dx >= nx + LAP, oy = p.dy < LAP || p.dy >= ny + LAP,
                   oz = p.dz < LAP || p.dz >= nz + LAP;
        ghost[r] = ox + oy + oz == 1 && (ox ? px : oy ? py : pz);
        // ghost g < LAP holds interior n + g, ghost n + LAP + g holds interior LAP + g
        p.sx = p.dx + (!ghost[r] || !ox ? 0 : p.dx < LAP ? nx : -nx);
        p.sy = p.dy + (!ghost[r] || !oy ? 0 : p.dy < LAP ? ny : -ny);
        p.sz = p.dz + (!ghost[r] || !oz ? 0 : p.dz < LAP ? nz : -nz);
        T[r] = fT.ptr[fidx(fT.pitch, nyg, p.sx, p.sy, p.sz)];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        if (i0 + r * NT >= total) break;
        const GhostPoint &p = q[r];
        if (ghost[r]) {
            double val[4];
            ghost_copy<4>(fl.f, 4, nyg, p, val);
            fT.ptr[fidx(fT.pitch, nyg, p.dx, p.dy, p.dz)] = T[r];
        }
        cc.ptr[fidx(cc.pitch, nyg, p.dx, p.dy, p.dz)] = sqrt(T[r]) / ama;
    }
}

}  // namespace

}  // namespace ws
