// k_viscous.hip -- viscous terms of the RHS (the reference's du_vis_Jacobian3d path).
//
// The tiled kernel family runs one fused kernel, k_vis_fused (below), whose fluxes never
// leave the chip.  The anchor family runs two kernels around a ghost fill, each marching
// column tiles along z:
//   k_vis_flux: per interior cell, Sutherland viscosity, the twelve central-difference
//               gradients (u, v, w, T along x, y, z), the stress tensor and heat flux, and
//               the four viscous fluxes of each of the three directions (twelve ghosted
//               scratch fields, interior written);
//   ghost fill of the twelve flux fields (periodic faces);
//   k_vis_div:  per interior cell, du[1..4] += Ajac * (central derivative of the direction's
//               fluxes), directions x, y, z in turn.
// The reference runs 12 derivative launches, three flux launches, three exchanges, twelve
// more derivative launches and twelve update launches per RHS, with the gradients and the
// fluxes' derivatives round-tripping through HBM; here the gradients never leave
// registers.
//
// The two kernels evaluate every expression in the reference's order with contraction off
// and divide as the reference does ((stencil / 60) / h): bit-identical to the CPU
// restatement.  The fused kernel weights the differences f(c + q) - f(c - q) instead, which
// moves a derivative by a few units in the last place.
#include <hip/hip_runtime.h>

#include "ws_device.h"

namespace ws {

namespace {

// A work-group owns a TX x TY column tile of up to ZC consecutive planes and marches it
// along z.  Each thread keeps the z-stencil of its column in registers, so every plane is
// read from HBM once per tile; the x and y stencils of a plane come from an LDS copy of
// the plane's tile and its halo (double-buffered: one barrier per plane).  The loads of
// plane z + 1 are issued before plane z is computed.
constexpr int TX = 32, TY = 8, NT = TX * TY;
constexpr int ZC = 32;

struct VisParams {
    int nx, ny, nz, nyg;
    double h[3];
    double amu_c0, tsb, vis_c;
    double metric[10];       // constant Akx..Asz, Ajac
    int bnd[6];              // closed faces (D0_bound): x-, x+, y-, y+, z-, z+
    int per[3];              // periodic directions
};

// the twelve flux fields (flux m of direction d at f[4*d + m]), one ghosted layout
struct EvFields {
    double *f[12];
    uint32_t pitch;
};

__device__ __forceinline__ double cd_stencil6(const double *s)
{
#pragma clang fp contract(off)
    return (45.0 * (s[4] - s[2]) - 9.0 * (s[5] - s[1]) + (s[6] - s[0])) / 60.0;
}

__device__ __forceinline__ double cd_stencil8(const double *s)
{
#pragma clang fp contract(off)
    return (672.0 * (s[5] - s[3]) - 168.0 * (s[6] - s[2]) + 32.0 * (s[7] - s[1]) - 3.0 * (s[8] - s[0])) / 840.0;
}

// central derivative along direction d of the stencil values s[0 .. ORDER]
template <int ORDER>
__device__ __forceinline__ double cd_dir(const double *s, const VisParams &p, int d)
{
#pragma clang fp contract(off)
    const double tmp = ORDER == 8 ? cd_stencil8(s) : cd_stencil6(s);
    return tmp / p.h[d];
}

// The forms of the four cells next to a closed face (the reference's D0_bound,
// OCFD_D0bound_scheme_kernel, src/boundary/OCFD_bound_Scheme.cpp:82-263, consulted by
// OCFD_CD6_kernel / OCFD_CD8_kernel before the central form, src/kernels/OCFD_Schemes.cpp:106-160):
// at distance 0 a one-sided first-order difference, at 1 a second-order, at 2 a fourth-order
// and at 3 a sixth-order central difference, the low face checked first; the reference's
// expression order, contraction off.  s[q] = f(c - R + q); none reads a point past the face.
// True and the undivided derivative in tmp when a form covers cell c of n.
template <int R>
__device__ __forceinline__ bool cd_closure(const double *s0, int c, int n, bool lo, bool hi, double &tmp)
{
#pragma clang fp contract(off)
    const double *s = s0 + R;
    if (lo && c <= 3) {
        if (c == 0) tmp = (s[1] - s[0]);
        else if (c == 1) tmp = (s[1] - s[-1]) * 0.5;
        else if (c == 2) tmp = (s[-2] - 8.0 * s[-1] + 8.0 * s[1] - s[2]) / 12.0;
        else tmp = (s[3] - s[-3] - 9.0 * (s[2] - s[-2]) + 45.0 * (s[1] - s[-1])) / 60.0;
        return true;
    }
    if (hi && c >= n - 4) {
        if (c == n - 1) tmp = (s[0] - s[-1]);
        else if (c == n - 2) tmp = (s[1] - s[-1]) * 0.5;
        else if (c == n - 3) tmp = (s[-2] - 8.0 * s[-1] + 8.0 * s[1] - s[2]) / 12.0;
        else tmp = (s[3] - s[-3] - 9.0 * (s[2] - s[-2]) + 45.0 * (s[1] - s[-1])) / 60.0;
        return true;
    }
    return false;
}

// Derivative along direction d at interior index c: a closure form next to a closed face
// (BND), else the central form; either is divided by h as the reference does (put_d0_kernel).
template <int ORDER, bool BND>
__device__ __forceinline__ double cd_at(const double *s, const VisParams &p, int d, int c)
{
#pragma clang fp contract(off)
    if constexpr (BND) {
        const int n = d == 0 ? p.nx : d == 1 ? p.ny : p.nz;
        double tmp;
        if (cd_closure<ORDER / 2>(s, c, n, p.bnd[2 * d] != 0, p.bnd[2 * d + 1] != 0, tmp)) return tmp / p.h[d];
    }
    return cd_dir<ORDER>(s, p, d);
}

// Plane tile with an R-deep halo in x and y (no corners): tile coordinates (px, py),
// px in [0, TX + 2R), py in [0, TY + 2R); the cells are px, py in [R, R + T).
template <int R>
struct Plane {
    static constexpr int PX = TX + 2 * R, PY = TY + 2 * R;
    static constexpr int NH = 2 * R * (TX + TY);       // halo points
    static constexpr int HPT = (NH + NT - 1) / NT;     // halo points per thread
    __device__ static bool xhalo(int h) { return h < 2 * R * TY; }
    __device__ static void halo(int h, int &px, int &py)
    {
        if (xhalo(h)) {
            const int side = h / (R * TY), r = h % (R * TY);
            py = R + r / R;
            px = side ? R + TX + r % R : r % R;
        } else {
            h -= 2 * R * TY;
            const int side = h / (R * TX), r = h % (R * TX);
            px = R + r % TX;
            py = side ? R + TY + r / TX : r / TX;
        }
    }
};

// Work-group -> tile.  The grid has 8 * per work-groups; work-group b runs tile
// (b % 8) * per + b / 8, so the tiles one XCD receives under round-robin dispatch form a
// contiguous range (neighbouring rows of one z-chunk), whose halos share that XCD's L2.
struct March {
    int x0, y0, z0, z1;      // tile origin (interior coordinates) and plane range
    int tx, ty;              // this thread's column in the tile
    bool tile_ok;            // the tile exists
    bool act;                // the column is inside the box: its cells are computed
    bool in;                 // the column is inside the ghosted box: its values are loaded
                             // (columns past the box are the ghosts of the cells near it)
};

__device__ __forceinline__ March march_tile(const VisParams &p)
{
    const int gx = (p.nx + TX - 1) / TX, gy = (p.ny + TY - 1) / TY, gz = (p.nz + ZC - 1) / ZC;
    const int ntiles = gx * gy * gz;
    const int per = (ntiles + 7) / 8;
    const int b = blockIdx.x;
    const int tile = (b % 8) * per + b / 8;
    const int bx = tile % gx, by = (tile / gx) % gy, bz = tile / (gx * gy);
    March m;
    m.x0 = bx * TX; m.y0 = by * TY;
    m.z0 = bz * ZC; m.z1 = min(m.z0 + ZC, p.nz);
    m.tx = (int)threadIdx.x % TX; m.ty = (int)threadIdx.x / TX;
    m.tile_ok = tile < ntiles;
    m.act = m.x0 + m.tx < p.nx && m.y0 + m.ty < p.ny;
    m.in = m.x0 + m.tx < p.nx + LAP && m.y0 + m.ty < p.ny + LAP;
    return m;
}

inline unsigned march_blocks(int nx, int ny, int nz)
{
    const long ntiles = (long)((nx + TX - 1) / TX) * ((ny + TY - 1) / TY) * ((nz + ZC - 1) / ZC);
    return (unsigned)(8 * ((ntiles + 7) / 8));
}

// This thread's halo points of the plane tile: tile coordinates and whether the point
// lies inside the ghosted box (points outside are only read by the stencils of cells
// outside the box)
template <int R>
struct HaloPts {
    int px[Plane<R>::HPT], py[Plane<R>::HPT];
    bool ok[Plane<R>::HPT];
};

template <int R>
__device__ __forceinline__ HaloPts<R> halo_points(const March &t, const VisParams &p)
{
    HaloPts<R> hp;
#pragma unroll
    for (int s = 0; s < Plane<R>::HPT; ++s) {
        const int h = (int)threadIdx.x + s * NT;
        hp.px[s] = hp.py[s] = 0;
        hp.ok[s] = false;
        if (h < Plane<R>::NH) {
            Plane<R>::halo(h, hp.px[s], hp.py[s]);
            const int gx = t.x0 + LAP - R + hp.px[s], gy = t.y0 + LAP - R + hp.py[s];
            hp.ok[s] = gx < p.nx + 2 * LAP && gy < p.nyg;
        }
    }
    return hp;
}

// z-column of a ghosted field through (x, y): element of ghosted plane zg at col.p[zg * col.s]
struct Col {
    const double *p;
    size_t s;
};

__device__ __forceinline__ Col column(const double *ptr, uint32_t pitch, int nyg, int x, int y)
{
    return Col{ptr + fidx(pitch, nyg, x, y, 0), (size_t)pitch * (size_t)nyg};
}

template <int ORDER, bool FIELDS, bool BND>
__global__ void __launch_bounds__(NT) k_vis_flux(VisParams p, ws_field u, ws_field v, ws_field w, ws_field T,
                                                 ws_metric_fields mf, EvFields ev)
{
#pragma clang fp contract(off)
    constexpr int R = ORDER / 2, Q = 2 * R + 1;
    using PL = Plane<R>;
    __shared__ double lds[2][4][PL::PY][PL::PX];
    const March t = march_tile(p);
    if (!t.tile_ok) return;
    const int nyg = p.nyg;
    const int x = t.x0 + t.tx + LAP, y = t.y0 + t.ty + LAP;
    const ws_field fl[4] = {u, v, w, T};
    const HaloPts<R> hp = halo_points<R>(t, p);
    // slot q of column f holds ghosted plane zg - R + q of the current plane zg
    Col k[4];
    double c[4][Q];
    const int zb = t.z0 + LAP, ze = t.z1 + LAP;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        k[f] = column(fl[f].ptr, fl[f].pitch, nyg, x, y);
#pragma unroll
        for (int q = 0; q < Q - 1; ++q) c[f][q] = t.in ? k[f].p[(size_t)(zb - R + q) * k[f].s] : 0.0;
    }
    // plane zg + 1: its new column slot and its halo points
    double nq[4], hv[PL::HPT][4];
    auto fetch = [&](int zg) {
#pragma unroll
        for (int f = 0; f < 4; ++f) nq[f] = t.in ? k[f].p[(size_t)(zg + R) * k[f].s] : 0.0;
#pragma unroll
        for (int s = 0; s < PL::HPT; ++s) {
            const int gx = t.x0 + LAP - R + hp.px[s], gy = t.y0 + LAP - R + hp.py[s];
#pragma unroll
            for (int f = 0; f < 4; ++f) hv[s][f] = hp.ok[s] ? fl[f].ptr[fidx(fl[f].pitch, nyg, gx, gy, zg)] : 0.0;
        }
    };
    fetch(zb);
    size_t o = fidx(ev.pitch, nyg, x, y, zb);             // output offset of plane zg
    const size_t oplane = (size_t)ev.pitch * nyg;
    for (int zg = zb; zg < ze; ++zg, o += oplane) {
        const int b = zg & 1;
#pragma unroll
        for (int f = 0; f < 4; ++f) c[f][Q - 1] = nq[f];
#pragma unroll
        for (int s = 0; s < PL::HPT; ++s) {
            if ((int)threadIdx.x + s * NT >= PL::NH) break;
#pragma unroll
            for (int f = 0; f < 4; ++f) lds[b][f][hp.py[s]][hp.px[s]] = hv[s][f];
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) lds[b][f][R + t.ty][R + t.tx] = c[f][R];
        if (zg + 1 < ze) fetch(zg + 1);
        __syncthreads();
        if (t.act) {
            auto met = [&](int m) -> double {
                if (FIELDS) {
                    const ws_field &g = m < 9 ? mf.A[m] : mf.ajac;
                    return g.ptr[fidx(g.pitch, nyg, x, y, zg)];
                }
                return p.metric[m];
            };
            // gradients along the computational directions (k, i, s = x, y, z)
            const int cx = x - LAP, cy = y - LAP, cz = zg - LAP;
            auto dx = [&](int f) {
                double s[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) s[q] = lds[b][f][R + t.ty][t.tx + q];
                return cd_at<ORDER, BND>(s, p, 0, cx);
            };
            auto dy = [&](int f) {
                double s[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) s[q] = lds[b][f][t.ty + q][R + t.tx];
                return cd_at<ORDER, BND>(s, p, 1, cy);
            };
            const double uk = dx(0), vk = dx(1), wk = dx(2), Tk = dx(3);
            const double ui = dy(0), vi = dy(1), wi = dy(2), Ti = dy(3);
            const double us = cd_at<ORDER, BND>(c[0], p, 2, cz), vs = cd_at<ORDER, BND>(c[1], p, 2, cz);
            const double ws = cd_at<ORDER, BND>(c[2], p, 2, cz), Ts = cd_at<ORDER, BND>(c[3], p, 2, cz);
            const double Akx = met(0), Aky = met(1), Akz = met(2), Aix = met(3), Aiy = met(4), Aiz = met(5);
            const double Asx = met(6), Asy = met(7), Asz = met(8), aj1 = met(9);
            // viscosity (get_Amu_kernal) and the stress tensor (vis_flux_ker)
            const double tc = c[3][R];
            const double amu = p.amu_c0 * sqrt(tc * tc * tc) / (p.tsb + tc);
            const double ux = uk * Akx + ui * Aix + us * Asx, vx = vk * Akx + vi * Aix + vs * Asx;
            const double wx = wk * Akx + wi * Aix + ws * Asx;
            const double uy = uk * Aky + ui * Aiy + us * Asy, vy = vk * Aky + vi * Aiy + vs * Asy;
            const double wy = wk * Aky + wi * Aiy + ws * Asy;
            const double uz = uk * Akz + ui * Aiz + us * Asz, vz = vk * Akz + vi * Aiz + vs * Asz;
            const double wz = wk * Akz + wi * Aiz + ws * Asz;
            const double div = ux + vy + wz;
            const double s11 = (2.0 * ux - 2.0 / 3.0 * div) * amu;
            const double s22 = (2.0 * vy - 2.0 / 3.0 * div) * amu;
            const double s33 = (2.0 * wz - 2.0 / 3.0 * div) * amu;
            const double s12 = (uy + vx) * amu, s13 = (uz + wx) * amu, s23 = (vz + wy) * amu;
            const double amuk = amu * p.vis_c;
            const double Tx = Tk * Akx + Ti * Aix + Ts * Asx;
            const double Ty = Tk * Aky + Ti * Aiy + Ts * Asy;
            const double Tz = Tk * Akz + Ti * Aiz + Ts * Asz;
            const double uc = c[0][R], vc = c[1][R], wc = c[2][R];
            const double E1 = uc * s11 + vc * s12 + wc * s13 + amuk * Tx;
            const double E2 = uc * s12 + vc * s22 + wc * s23 + amuk * Ty;
            const double E3 = uc * s13 + vc * s23 + wc * s33 + amuk * Tz;
            const double Am[9] = {Akx, Aky, Akz, Aix, Aiy, Aiz, Asx, Asy, Asz};
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double akx = Am[3 * d] * aj1, aky = Am[3 * d + 1] * aj1, akz = Am[3 * d + 2] * aj1;
                ev.f[4 * d + 0][o] = akx * s11 + aky * s12 + akz * s13;
                ev.f[4 * d + 1][o] = akx * s12 + aky * s22 + akz * s23;
                ev.f[4 * d + 2][o] = akx * s13 + aky * s23 + akz * s33;
                ev.f[4 * d + 3][o] = akx * E1 + aky * E2 + akz * E3;
            }
        }
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int q = 0; q < Q - 1; ++q) c[f][q] = c[f][q + 1];
    }
}

template <int ORDER, bool FIELDS, bool BND>
__global__ void __launch_bounds__(NT) k_vis_div(VisParams p, EvFields ev, ws_field ajac, ws_soa du)
{
#pragma clang fp contract(off)
    constexpr int R = ORDER / 2, Q = 2 * R + 1;
    using PL = Plane<R>;
    // x-direction fluxes with their x-halo, y-direction fluxes with their y-halo
    __shared__ double lx[2][4][TY][PL::PX];
    __shared__ double ly[2][4][PL::PY][TX];
    const March t = march_tile(p);
    if (!t.tile_ok) return;
    const int nyg = p.nyg;
    const int x = t.x0 + t.tx + LAP, y = t.y0 + t.ty + LAP;
    const HaloPts<R> hp = halo_points<R>(t, p);
    const size_t oplane = (size_t)ev.pitch * nyg;
    const size_t o0 = fidx(ev.pitch, nyg, x, y, 0);       // this column's offset in plane 0
    // z-columns of the four z-direction fluxes (slot q: ghosted plane zg - R + q)
    double cz[4][Q];
    const int zb = t.z0 + LAP, ze = t.z1 + LAP;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < Q - 1; ++q) cz[m][q] = t.in ? ev.f[8 + m][o0 + (size_t)(zb - R + q) * oplane] : 0.0;
    const size_t vstride = (size_t)du.pitch * p.ny * p.nz;
    const size_t dplane = (size_t)du.pitch * p.ny;
    double *dp = du.ptr + (size_t)(x - LAP) + (size_t)du.pitch * ((size_t)(y - LAP) + (size_t)p.ny * (size_t)t.z0);
    // plane zg + 1: new z-column slots, the column's x and y fluxes, du, the halo points
    double nz_[4], nx_[4], ny_[4], dn[4], hv[PL::HPT][4];
    auto fetch = [&](int zg, const double *q) {
        const size_t oz = o0 + (size_t)zg * oplane;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            nz_[m] = t.in ? ev.f[8 + m][oz + (size_t)R * oplane] : 0.0;
            nx_[m] = t.in ? ev.f[m][oz] : 0.0;
            ny_[m] = t.in ? ev.f[4 + m][oz] : 0.0;
            dn[m] = t.act ? q[(m + 1) * vstride] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < PL::HPT; ++s) {
            const int h = (int)threadIdx.x + s * NT;
            const int gx = t.x0 + LAP - R + hp.px[s], gy = t.y0 + LAP - R + hp.py[s];
            const size_t oh = fidx(ev.pitch, nyg, gx, gy, zg);
            const int d = PL::xhalo(h) ? 0 : 1;
#pragma unroll
            for (int m = 0; m < 4; ++m) hv[s][m] = hp.ok[s] ? ev.f[4 * d + m][oh] : 0.0;
        }
    };
    fetch(zb, dp);
    for (int zg = zb; zg < ze; ++zg, dp += dplane) {
        const int b = zg & 1;
        double acc[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            cz[m][Q - 1] = nz_[m];
            lx[b][m][t.ty][R + t.tx] = nx_[m];
            ly[b][m][R + t.ty][t.tx] = ny_[m];
            acc[m] = dn[m];
        }
#pragma unroll
        for (int s = 0; s < PL::HPT; ++s) {
            const int h = (int)threadIdx.x + s * NT;
            if (h >= PL::NH) break;
            if (PL::xhalo(h)) {
#pragma unroll
                for (int m = 0; m < 4; ++m) lx[b][m][hp.py[s] - R][hp.px[s]] = hv[s][m];
            } else {
#pragma unroll
                for (int m = 0; m < 4; ++m) ly[b][m][hp.py[s]][hp.px[s] - R] = hv[s][m];
            }
        }
        if (zg + 1 < ze) fetch(zg + 1, dp + dplane);
        __syncthreads();
        if (t.act) {
            const double aj = FIELDS ? ajac.ptr[fidx(ajac.pitch, nyg, x, y, zg)] : p.metric[9];
            const int cx = x - LAP, cy = y - LAP, ck = zg - LAP;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                double s[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) s[q] = lx[b][m][t.ty][t.tx + q];
                acc[m] = acc[m] + aj * cd_at<ORDER, BND>(s, p, 0, cx);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                double s[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) s[q] = ly[b][m][t.ty + q][t.tx];
                acc[m] = acc[m] + aj * cd_at<ORDER, BND>(s, p, 1, cy);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[m] = acc[m] + aj * cd_at<ORDER, BND>(cz[m], p, 2, ck);
#pragma unroll
            for (int m = 0; m < 4; ++m) dp[(m + 1) * vstride] = acc[m];
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int q = 0; q < Q - 1; ++q) cz[m][q] = cz[m][q + 1];
    }
}

// ---- fused form (fast family) ------------------------------------------------------------
//
// One kernel for the whole viscous update: no flux field goes through memory.  A work-group
// of FX x FY = 32 x 16 threads owns the flux points of a (FX - 2R) x (FY - 2R) cell tile plus
// an R-deep ring around it and marches a chunk of planes along z.  At each flux plane every
// thread computes the twelve gradients at its point (x and y stencils from an LDS copy of
// the plane with a further R-deep border, the z stencil from its column's register window)
// and the fluxes its point contributes: x fluxes on the tile's rows, y fluxes on its columns,
// z fluxes inside the tile.  The x and y fluxes go to LDS and are differentiated one plane
// later; a z flux is added at once, by its increment over the plane before, to the 2R cells of
// its column whose derivative the two enter on either side (register accumulators of the cells
// zf - R .. zf + R - 1), so a cell is complete R planes after its own flux plane.  With W_j = the
// sum of the coefficients c_q, q >= max(j, 1 - j),
//   sum_q c_q (F(c + q) - F(c - q)) = sum_j W_j (F(c + j) - F(c + j - 1)),  j = 1 - R .. R:
// differences of the flux as along x and y, so a flux that does not change along z adds
// nothing (its weighted values one by one would leave their rounding).
//
// Both LDS arrays are double-buffered: a step computes plane zf's fluxes from one copy,
// writes the copy of plane zf + 1, and differentiates the fluxes of plane zf - 1, with one
// barrier between steps; the loads of the next step are issued at its top.  The window and
// the accumulators turn by one slot per plane, so the loop is unrolled over one turn (2R + 1
// steps) and no slot is ever moved.
//
// Data points are addressed in interior coordinates: a periodic direction wraps them onto the
// interior (the flux at a point past the face is the one of its periodic image, bit for bit),
// so neither the fields' ghost layers nor any scratch is touched.  At a closed face the
// derivative forms (cd_closure) are all weights on f(c + q) - f(c - q), q <= 3, if the points
// past the face repeat the face cell's value: the first-order one-sided difference is q = 1
// with weight 1.  Points past the face therefore are the face point itself (its data, its
// flux), the weights come from a table by the distance to the face, and a difference whose
// weight is zero reads the cell itself on both sides.
//
// MODE: constant metrics without off-diagonal terms (a Cartesian box; the weights carry the
// metric terms), constant metrics, or metric fields read per flux point.  LAYOUT (the
// launcher chooses): with one pitch and planes within 32-bit byte offsets one offset per thread
// addresses every field (VL_ONE); with several pitches (VL_PITCHES) each load forms its own
// from the thread's column and row, two instructions, rather than hold up to eighteen of them;
// planes of 4 GB and more (VL_BIG) take 64-bit addresses.
//
// Algorithmic traffic 96 B per cell (constant metrics): u, v, w, T in and du[1..4] read and
// written.  512 threads of up to 256 VGPRs: one work-group per compute unit.  Sixth order and
// periodic eighth order spill nothing with one pitch; scratch per lane of the others: eighth order
// with closed faces 36-72 bytes, over metric fields 140-144; eighth order with several pitches
// 8-52 (closed faces 64, over metric fields 156); planes of 4 GB 36-380.
//
// What bounds it: a step moves 84 values per thread through LDS at 128 B per cycle (3,100 of
// about 5,300 cycles), and the eight wavefronts read LDS and compute in the same phases, so
// the two add up; issuing each stage's reads under the stage before it, and letting half the
// wavefronts run half a step behind, were tried and measured no faster.  Before this form (z
// fluxes and xy sums in LDS rings, closure forms branched per derivative, fixed 64-plane
// chunks) and now, alone: 600x128x128 sixth order 640 -> 466 us, eighth 943 -> 696;
// 157x111x75 193 -> 69 and 227 -> 125; x faces closed 211x93x67 459 -> 98 and 458 -> 178, all
// faces closed 521 -> 151 and 523 -> 197; metric fields 256x160x96 (two kernels around a ghost
// fill of twelve flux fields before) 446 -> 320 and 450 -> 358.
// Rounding against 64-bit-mantissa arithmetic, before and now: vortices 5.29e-16 -> 5.03e-16
// (sixth order) and 6.18e-16 -> 5.91e-16, rough flow 1.87e-16 -> 1.87e-16 and 2.54e-16 ->
// 2.54e-16.
constexpr int FX = 32, FY = 16, FNT = FX * FY;
enum { VM_DIAG, VM_CONST, VM_FIELDS };
enum { VC_NONE, VC_XY, VC_ALL };
enum { VL_ONE, VL_PITCHES, VL_BIG };

// Weights of the differences f(c + q) - f(c - q), q = 1..4 at index q - 1: whole numbers over one
// denominator (60, or 840 for the eighth order), so that they carry no rounding, and what that
// denominator, the spacing and the constant metric terms make of a derivative.
struct VisWeights {
    double row[5][4];        // numerators at distance 0..3 from a closed face, and the central ones
    double rz[5][4];         // of the W_j = W_(1-j), j = 1..4, of each row
    double gs[3], fs[3];     // VM_DIAG: of a gradient along d and of a flux derivative; VM_FIELDS: gs alone, on the terms
    double gA[9], fA[9];     // VM_CONST: the metric terms of the gradients and of the fluxes, times them
};

template <int R>
struct Fused {
    static constexpr int TX = FX - 2 * R, TY = FY - 2 * R;     // cells of the tile
    static constexpr int PX = FX + 2 * R, PY = FY + 2 * R;     // plane copy: flux points + border
    static constexpr int PN = PX * PY;
    static constexpr int NBX = 2 * R * FY;                     // border points left and right
    static constexpr int NB = NBX + 2 * R * FX;                // and below and above (no corners)
    static_assert(NB <= FNT, "one border point per thread");
    // border point h -> plane-copy coordinates
    __device__ static void border(int h, int &px, int &py)
    {
        if (h < NBX) {
            const int side = h / (R * FY), r = h % (R * FY);
            py = R + r / R;
            px = side ? R + FX + r % R : r % R;
        } else {
            h -= NBX;
            const int side = h / (R * FX), r = h % (R * FX);
            px = R + r % FX;
            py = side ? R + FY + r / FX : r / FX;
        }
    }
};

// a coordinate of the data onto the interior [0, n): periodic images, or clamped
__device__ __forceinline__ int wrap_coord(int c, int n, bool periodic)
{
    if (periodic) {
        c %= n;
        return c < 0 ? c + n : c;
    }
    return c < 0 ? 0 : (c >= n ? n - 1 : c);
}

// Byte offsets of consecutive planes of a ghosted field (uniform across the work-group):
// wrap_coord of planes z, z + 1, ...; PER: every direction is periodic
template <bool PER>
struct PlaneWalk {
    int raw, n;              // periodic: the wrapped plane
    bool periodic;
    size_t bytes, off;       // bytes per plane; offset of the current plane
    __device__ PlaneWalk(int z, int n_, bool per, size_t bytes_) : n(n_), periodic(PER || per), bytes(bytes_)
    {
        const int at = wrap_coord(z, n, periodic);
        raw = periodic ? at : z;
        off = bytes * (size_t)(at + LAP);
    }
    __device__ int plane() const { return periodic ? raw : min(max(raw, 0), n - 1); }
    __device__ void next()
    {
        ++raw;
        if (PER || periodic) {
            const bool turn = raw == n;
            off = turn ? bytes * LAP : off + bytes;
            raw = turn ? 0 : raw;
        } else {
            off = raw > 0 && raw < n ? off + bytes : off;
        }
    }
};

// row of VisWeights::row of cell c, and how many differences that row has
__device__ __forceinline__ int closure_row(int c, int n, bool lo, bool hi)
{
    return lo && c <= 3 ? c : hi && c >= n - 4 ? n - 1 - c : 4;
}

template <int R>
__device__ __forceinline__ int closure_reach(int row)
{
    return row == 0 ? 1 : row == 4 ? R : row;
}

template <int P>
struct Phase {
    static constexpr int value = P;
};

template <int ORDER, int MODE, int CLOSED, int LAYOUT>
__global__ void __launch_bounds__(FNT) k_vis_fused(VisParams p, VisWeights wt, ws_field u, ws_field v, ws_field w,
                                                   ws_field T, ws_metric_fields mf, ws_soa du, int zc)
{
    // Every fused multiply-add is written out: the step is compiled 2R + 1 times, and left to the
    // compiler each of them could fuse differently, so that a flux would depend on the plane its
    // chunk starts at.  So the flux at a point past a periodic face equals the one at its image
    // bit for bit, and neither the chunks nor the tile a cell falls in change its bits.
#pragma clang fp contract(off)
    constexpr int R = ORDER / 2, Q = 2 * R + 1;
    using FZ = Fused<R>;
    constexpr int PX = FZ::PX, PN = FZ::PN, XN = FZ::TY * FX, YN = FY * PX;
    constexpr bool FLD = MODE == VM_FIELDS, BND = CLOSED != VC_NONE, BNDZ = CLOSED == VC_ALL;
    __shared__ double pl[2][4][PN];      // u, v, w, T of a plane: flux points and border
    __shared__ double fxa[2][4][XN];     // x fluxes on the tile's rows (rows of FX)
    __shared__ double fya[2][4][YN];     // y fluxes on the tile's columns (rows of PX, as the plane copy)
    const int gx = (p.nx + FZ::TX - 1) / FZ::TX, gy = (p.ny + FZ::TY - 1) / FZ::TY, gz = (p.nz + zc - 1) / zc;
    const int ntiles = gx * gy * gz;
    const int per = (ntiles + 7) / 8;
    const int tile = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
    if (tile >= ntiles) return;
    const int x0 = (tile % gx) * FZ::TX, y0 = ((tile / gx) % gy) * FZ::TY;
    const int z0 = (tile / (gx * gy)) * zc, z1 = min(z0 + zc, p.nz);
    // the tile's rows go to the first wavefronts, the ring's to the last ones, which then have
    // no flux derivatives to take
    constexpr int TY = FZ::TY;
    const int tx = (int)threadIdx.x % FX, ti = (int)threadIdx.x / FX;
    const int ty = ti < TY ? ti + R : ti < TY + R ? ti - TY : ti;
    const bool perx = p.per[0] != 0, pery = p.per[1] != 0, perz = p.per[2] != 0;
    // this thread's flux point and (inside the tile) cell
    const int fx = x0 - R + tx, fy = y0 - R + ty;
    const bool xrow = ty >= R && ty < FY - R, ycol = tx >= R && tx < FX - R;   // x / y fluxes needed
    const bool cell = xrow && ycol && fx < p.nx && fy < p.ny;
    const int nyg = p.nyg;
    const ws_field fl[4] = {u, v, w, T};
    // the column of this flux point, and this thread's border point of the plane copy (threads
    // without one load their own point again)
    const int cxw = wrap_coord(fx, p.nx, perx), cyw = wrap_coord(fy, p.ny, pery);
    const int bi = FNT - 1 - (int)threadIdx.x;     // the last threads first: ring wavefronts
    const bool bord = bi < FZ::NB;
    int bpx = 0, bpy = 0, bxw = cxw, byw = cyw;
    if (bord) {
        FZ::border(bi, bpx, bpy);
        bxw = wrap_coord(x0 - 2 * R + bpx, p.nx, perx);
        byw = wrap_coord(y0 - 2 * R + bpy, p.ny, pery);
    }
    // VL_ONE: byte offsets within a plane of the fields (they share u's pitch); VL_PITCHES: the
    // column and row they come from; of du (threads without a cell point at its first)
    uint32_t off = 8u * ((uint32_t)(cxw + LAP) + u.pitch * (uint32_t)(cyw + LAP));
    uint32_t boff = 8u * ((uint32_t)(bxw + LAP) + u.pitch * (uint32_t)(byw + LAP));
    uint32_t cx = 8u * (uint32_t)(cxw + LAP), cy = (uint32_t)(cyw + LAP);
    uint32_t bx = 8u * (uint32_t)(bxw + LAP), by = (uint32_t)(byw + LAP);
    uint32_t doff = cell ? 8u * ((uint32_t)fx + du.pitch * (uint32_t)fy) : 0u;
    const size_t vstride = (size_t)du.pitch * p.ny * p.nz, dplane = 8 * (size_t)du.pitch * p.ny;
    const size_t fplane = 8 * (size_t)u.pitch * nyg;          // VL_ONE: bytes of a field's plane
    // VL_ONE; with closed z faces formed from the plane: the four running offsets would not fit the
    // scalar registers, and what spills takes vector ones (eighth order over metric fields 368 ->
    // 132 bytes of scratch per lane; all faces closed 211x93x67 sixth order 157 -> 143 us)
    auto plane_off = [&](const PlaneWalk<!BNDZ> &z) { return BNDZ ? fplane * (size_t)(z.plane() + LAP) : z.off; };
    auto plane_of = [&](const ws_field &f, const PlaneWalk<!BNDZ> &z) {
        return (const char *)f.ptr + 8 * (size_t)f.pitch * (size_t)nyg * (size_t)(z.plane() + LAP);
    };
    // element of field f at this thread's point of the plane a walk stands on
    auto at = [&](const ws_field &f, const PlaneWalk<!BNDZ> &z) -> double {
        if constexpr (LAYOUT == VL_ONE) return *(const double *)((const char *)f.ptr + plane_off(z) + off);
        else if constexpr (LAYOUT == VL_PITCHES) return *(const double *)(plane_of(f, z) + (cx + 8u * f.pitch * cy));
        else return f.ptr[fidx(f.pitch, nyg, cxw + LAP, cyw + LAP, z.plane() + LAP)];
    };
    auto at_border = [&](const ws_field &f, const PlaneWalk<!BNDZ> &z) -> double {
        if constexpr (LAYOUT == VL_ONE) return *(const double *)((const char *)f.ptr + plane_off(z) + boff);
        else if constexpr (LAYOUT == VL_PITCHES) return *(const double *)(plane_of(f, z) + (bx + 8u * f.pitch * by));
        else return f.ptr[fidx(f.pitch, nyg, bxw + LAP, byw + LAP, z.plane() + LAP)];
    };
    double *const dm[4] = {du.ptr + vstride, du.ptr + 2 * vstride, du.ptr + 3 * vstride, du.ptr + 4 * vstride};
    // du[m + 1] of this thread's cell at plane offset z (bytes)
    auto du_at = [&](int m, size_t z) -> double & {
        if constexpr (LAYOUT != VL_BIG) return *(double *)((char *)dm[m] + z + doff);
        else return *(double *)((char *)dm[m] + z + 8 * (cell ? (size_t)fx + (size_t)du.pitch * fy : 0));
    };
    // where this thread reads the plane copy; past a closed face the face point (BND), with the
    // weights and the reach (0 where the weight is) of the differences along x and y
    int own = (ty + R) * PX + tx + R;
    const int mine = own;
    __shared__ double wxl[BND ? R : 1][FX], wyl[BND ? R : 1][FY];
    int ox[BND ? R : 1], oy[BND ? R : 1];
    const bool zlo = BNDZ && p.bnd[4], zhi = BNDZ && p.bnd[5];
    if constexpr (BND) {
        const int px = perx ? fx : cxw, py = pery ? fy : cyw;
        own = (py - (y0 - 2 * R)) * PX + px - (x0 - 2 * R);
        const int rx = closure_row(cxw, p.nx, p.bnd[0] != 0, p.bnd[1] != 0);
        const int ry = closure_row(cyw, p.ny, p.bnd[2] != 0, p.bnd[3] != 0);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (ty == 0) wxl[q][tx] = wt.row[rx][q];
            if (tx == 0) wyl[q][ty] = wt.row[ry][q];
            ox[q] = q < closure_reach<R>(rx) ? q + 1 : 0;
            oy[q] = (q < closure_reach<R>(ry) ? q + 1 : 0) * PX;
        }
    }
    // Undivided derivatives along x and y (rows of PX) at element e of an LDS array: the smallest
    // difference's weight is one in the sixth-order central form.
    constexpr double CD[4] = {ORDER == 8 ? 672.0 : 45.0, ORDER == 8 ? -168.0 : -9.0, ORDER == 8 ? 32.0 : 1.0, -3.0};
    constexpr double CZ[4] = {ORDER == 8 ? 533.0 : 37.0, ORDER == 8 ? -139.0 : -8.0, ORDER == 8 ? 29.0 : 1.0, -3.0};
    int wtx = tx, wty = ty;
    auto ddx = [&](const double *e) {
        double t = 0.0;
#pragma unroll
        for (int q = R - 1; q >= 0; --q) {
            const double d = BND ? e[ox[q]] - e[-ox[q]] : e[q + 1] - e[-q - 1], a = BND ? wxl[q][wtx] : CD[q];
            t = q == R - 1 ? a * d : fma(a, d, t);
        }
        return t;
    };
    auto ddy = [&](const double *e) {
        double t = 0.0;
#pragma unroll
        for (int q = R - 1; q >= 0; --q) {
            const double d = BND ? e[oy[q]] - e[-oy[q]] : e[(q + 1) * PX] - e[-(q + 1) * PX];
            const double a = BND ? wyl[q][wty] : CD[q];
            t = q == R - 1 ? a * d : fma(a, d, t);
        }
        return t;
    };
    // flux planes zf0 .. zf1 - 1 produce the chunk's cells z0 .. z1 - 1
    const int zf0 = z0 - R, zf1 = z1 + R;
    // slot (P + R + k) % Q at the step of phase P: plane zf + k of the column (c), and the
    // derivative sum of cell zf + k (acc)
    double c[4][Q], acc[4][Q];
    // the z flux of plane zf - 1: in registers, but in instances that have none to spare in LDS,
    // which costs less than the scratch they would take (eighth order, x closed 211x93x67 198 ->
    // 178 us, all faces 220 -> 200, metric fields 256x160x96 394 -> 388; sixth order, x closed 101
    // -> 98)
    constexpr bool FZL = BND || (ORDER == 8 && FLD);
    __shared__ double fzl[4][FZL ? FNT : 1];
    double fzr[4];
    auto last = [&](int m) -> double & {
        if constexpr (FZL) return fzl[m][threadIdx.x];
        else return fzr[m];
    };
    // loaded for the coming step: the newest column plane, the border of the plane after its
    // flux plane, du of the cell it writes, and with metric fields that cell's Jacobian
    double nq[4], hb[4], dn[4], jn = 0.0;
    size_t dz = dplane * (size_t)z0;               // du plane of the cell the coming step writes
    PlaneWalk<!BNDZ> wq(zf0 - R, p.nz, perz, fplane), wb(zf0, p.nz, perz, fplane), wm(zf0, p.nz, perz, fplane),
        wj(z0, p.nz, perz, fplane);
#pragma unroll
    for (int q = 0; q < Q - 1; ++q, wq.next())
#pragma unroll
        for (int f = 0; f < 4; ++f) c[f][q] = at(fl[f], wq);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[f][q] = 0.0;
        pl[0][f][mine] = c[f][R];
        hb[f] = at_border(fl[f], wb);
        dn[f] = last(f) = 0.0;    // the first increment reaches no cell of the chunk
    }
    wb.next();
    if (bord)
#pragma unroll
        for (int f = 0; f < 4; ++f) pl[0][f][bpy * PX + bpx] = hb[f];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        nq[f] = at(fl[f], wq);
        hb[f] = at_border(fl[f], wb);
    }
    wq.next();
    wb.next();
    __syncthreads();
    int zf = zf0, cur = 0;
    // one step; false when the march is complete
    auto step = [&](auto phase) __attribute__((always_inline)) -> bool {
        constexpr int P = decltype(phase)::value;
        auto slot = [](int k) constexpr { return (P + R + k + 2 * Q) % Q; };
        const int nxt = cur ^ 1;
        // keeps the plane offsets scalar: the loads take them as their scalar base
        asm volatile("" : "+v"(off), "+v"(boff), "+v"(doff));
        // and the fields' own offsets from being formed once for all steps and kept
        if constexpr (LAYOUT == VL_PITCHES) asm volatile("" : "+v"(cx), "+v"(cy), "+v"(bx), "+v"(by));
        // the cell that the last step completed (its slot is the coming cell's)
        if (cell && zf - R - 1 >= z0)
#pragma unroll
            for (int m = 0; m < 4; ++m)
                du_at(m, dz) = FLD ? fma(jn, acc[m][slot(-R - 1)], dn[m]) : dn[m] + acc[m][slot(-R - 1)];
        if (zf == zf1) return false;
        // the newest plane of the column, and the copy of the next plane
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            c[f][slot(R)] = nq[f];
            pl[nxt][f][mine] = c[f][slot(1)];
        }
        if (bord)
#pragma unroll
            for (int f = 0; f < 4; ++f) pl[nxt][f][bpy * PX + bpx] = hb[f];
        // the loads of the coming step
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            nq[f] = at(fl[f], wq);
            hb[f] = at_border(fl[f], wb);
        }
        wq.next();
        wb.next();
        __builtin_amdgcn_sched_barrier(0);
        // gradients and fluxes at this thread's flux point of plane zf
        if (BND) asm volatile("" : "+v"(wtx), "+v"(wty));    // the weights are read where they are used
        const double *pc = &pl[cur][0][own];
        double gk[4], gi[4], gs[4], met[FLD ? 10 : 1];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if constexpr (FLD) {
                // this plane's metric terms, used once the gradients are complete
                if (f == 2) {
#pragma unroll
                    for (int q = 0; q < 10; ++q) met[q] = at(q < 9 ? mf.A[q] : mf.ajac, wm);
                    wm.next();
                }
            }
            gk[f] = ddx(pc + f * PN);
            gi[f] = ddy(pc + f * PN);
            if constexpr (!BNDZ) {
#pragma unroll
                for (int q = R; q >= 1; --q) {
                    const double d = c[f][slot(q)] - c[f][slot(-q)];
                    gs[f] = q == R ? CD[q - 1] * d : fma(CD[q - 1], d, gs[f]);
                }
            }
            if constexpr (MODE == VM_DIAG) { gk[f] *= wt.gs[0]; gi[f] *= wt.gs[1]; if (!BNDZ) gs[f] *= wt.gs[2]; }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (BNDZ) {
            // selects and not branches: the arrays stay in registers without copies at joins
            const int row = closure_row(min(max(zf, 0), p.nz - 1), p.nz, zlo, zhi), reach = closure_reach<R>(row);
#pragma unroll
            for (int q = R; q >= 1; --q)
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    const double d = q <= reach ? c[f][slot(q)] - c[f][slot(-q)] : 0.0;
                    gs[f] = q == R ? wt.row[row][q - 1] * d : fma(wt.row[row][q - 1], d, gs[f]);
                    if (MODE == VM_DIAG && q == 1) gs[f] *= wt.gs[2];
                }
        }
        if constexpr (FLD)
#pragma unroll
            for (int q = 0; q < 9; ++q) met[q] *= wt.gs[q / 3];
        const double uc = c[0][slot(0)], vc = c[1][slot(0)], wc = c[2][slot(0)], tc = c[3][slot(0)];
        // T^3 with a summand below its last bit, except for T = 0, of which sqrt_nr is not defined
        const double amu = p.amu_c0 * sqrt_nr(fma(tc * tc, tc, 0x1p-1000)) * recip_nr(p.tsb + tc);
        auto A = [&](int q) {
            if constexpr (FLD) return met[q];
            else return wt.gA[q];
        };
        // physical derivatives from the computational ones (the metric terms, or in VM_DIAG the
        // scale before, carry the spacing)
        auto dot = [](double a, double x, double b, double y, double c, double z) { return fma(c, z, fma(b, y, a * x)); };
        auto px = [&](int f) { return MODE == VM_DIAG ? gk[f] : dot(gk[f], A(0), gi[f], A(3), gs[f], A(6)); };
        auto py = [&](int f) { return MODE == VM_DIAG ? gi[f] : dot(gk[f], A(1), gi[f], A(4), gs[f], A(7)); };
        auto pz = [&](int f) { return MODE == VM_DIAG ? gs[f] : dot(gk[f], A(2), gi[f], A(5), gs[f], A(8)); };
        const double ux = px(0), vx = px(1), wx_ = px(2), Tx = px(3);
        const double uy = py(0), vy = py(1), wy_ = py(2), Ty = py(3);
        const double uz = pz(0), vz = pz(1), wz = pz(2), Tz = pz(3);
        const double div23 = -2.0 / 3.0 * (ux + vy + wz);
        const double s11 = fma(2.0, ux, div23) * amu;
        const double s22 = fma(2.0, vy, div23) * amu;
        const double s33 = fma(2.0, wz, div23) * amu;
        const double s12 = (uy + vx) * amu, s13 = (uz + wx_) * amu, s23 = (vz + wy_) * amu;
        const double amuk = amu * p.vis_c;
        const double E1 = fma(amuk, Tx, dot(uc, s11, vc, s12, wc, s13));
        const double E2 = fma(amuk, Ty, dot(uc, s12, vc, s22, wc, s23));
        const double E3 = fma(amuk, Tz, dot(uc, s13, vc, s23, wc, s33));
        // flux of direction d (its metric terms, or in VM_DIAG the scale of its derivative, carry the
        // spacing and the constant factors)
        auto flux = [&](int d, double out[4]) {
            if constexpr (MODE == VM_DIAG) {
                out[0] = d == 0 ? s11 : d == 1 ? s12 : s13;
                out[1] = d == 0 ? s12 : d == 1 ? s22 : s23;
                out[2] = d == 0 ? s13 : d == 1 ? s23 : s33;
                out[3] = d == 0 ? E1 : d == 1 ? E2 : E3;
            } else {
                double a1 = wt.fA[3 * d], a2 = wt.fA[3 * d + 1], a3 = wt.fA[3 * d + 2];
                if constexpr (FLD) { a1 = A(3 * d) * met[9]; a2 = A(3 * d + 1) * met[9]; a3 = A(3 * d + 2) * met[9]; }
                out[0] = dot(a1, s11, a2, s12, a3, s13);
                out[1] = dot(a1, s12, a2, s22, a3, s23);
                out[2] = dot(a1, s13, a2, s23, a3, s33);
                out[3] = dot(a1, E1, a2, E2, a3, E3);
            }
        };
        double F[4];
        if (xrow) {
            flux(0, F);
#pragma unroll
            for (int m = 0; m < 4; ++m) fxa[cur][m][(ty - R) * FX + tx] = F[m];
        }
        if (ycol) {
            flux(1, F);
#pragma unroll
            for (int m = 0; m < 4; ++m) fya[cur][m][ty * PX + tx] = F[m];
        }
        flux(2, F);
        double G[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            G[m] = F[m] - last(m);
            if (MODE == VM_DIAG) G[m] *= wt.fs[2];
            last(m) = F[m];
        }
        if constexpr (BNDZ) {
            // no flux changes past a closed z face
            const bool zin = perz || (zf > 0 && zf < p.nz);
#pragma unroll
            for (int q = 1; q <= R; ++q) {
                const int zl = zf - q, zh = zf + q - 1;
                const int lo = closure_row(min(max(zl, 0), p.nz - 1), p.nz, zlo, zhi);
                const int hi = closure_row(min(max(zh, 0), p.nz - 1), p.nz, zlo, zhi);
                const bool ul = zin && (perz || zl >= 0) && q <= closure_reach<R>(lo);
                const bool uh = zin && (perz || zh < p.nz) && q <= closure_reach<R>(hi);
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const double Gl = ul ? G[m] : 0.0, Gh = uh ? G[m] : 0.0;
                    acc[m][slot(-q)] = fma(wt.rz[lo][q - 1], Gl, acc[m][slot(-q)]);
                    acc[m][slot(q - 1)] =
                        q == R ? wt.rz[hi][q - 1] * Gh : fma(wt.rz[hi][q - 1], Gh, acc[m][slot(q - 1)]);
                }
            }
        } else {
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 1; q <= R; ++q) {
                    acc[m][slot(-q)] = fma(CZ[q - 1], G[m], acc[m][slot(-q)]);
                    acc[m][slot(q - 1)] = q == R ? CZ[q - 1] * G[m] : fma(CZ[q - 1], G[m], acc[m][slot(q - 1)]);
                }
        }
        // du of the cell the coming step writes: here rather than with the other loads, whose
        // registers the gradients need
        if (zf - R > z0) {
            dz += dplane;
            if constexpr (FLD) wj.next();
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) dn[m] = du_at(m, dz);
        if constexpr (FLD) jn = at(mf.ajac, wj);
        __builtin_amdgcn_sched_barrier(0);
        // x and y derivatives of the previous plane's fluxes
        if (cell)
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const double fx_x = ddx(&fxa[nxt][m][(ty - R) * FX + tx]), fy_y = ddy(&fya[nxt][m][ty * PX + tx]);
                if constexpr (MODE == VM_DIAG) acc[m][slot(-1)] += fma(fx_x, wt.fs[0], fy_y * wt.fs[1]);
                else acc[m][slot(-1)] += fx_x + fy_y;
                __builtin_amdgcn_sched_barrier(0);
            }
        // the sums are formed here: used only where a cell is written, they would otherwise be
        // sunk there, with every flux of the last 2R planes kept alive for them
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int q = -R; q < R; ++q) asm volatile("" : "+v"(acc[m][slot(q)]));
        ++zf;
        __syncthreads();
        cur = nxt;
        return true;
    };
    auto turn = [&](auto... phase) __attribute__((always_inline)) { return (step(phase) && ...); };
    if constexpr (Q == 7) {
        while (turn(Phase<0>{}, Phase<1>{}, Phase<2>{}, Phase<3>{}, Phase<4>{}, Phase<5>{}, Phase<6>{})) {}
    } else {
        while (turn(Phase<0>{}, Phase<1>{}, Phase<2>{}, Phase<3>{}, Phase<4>{}, Phase<5>{}, Phase<6>{}, Phase<7>{},
                    Phase<8>{})) {}
    }
}

// Planes per work-group of the fused form: its work-groups hold a compute unit each, so a
// launch takes about (rounds of work-groups) x (planes each marches, the 2R of its halo
// included) plane steps; the chunk length with the smallest product is taken.  Runs on every
// call: only the chunk counts at which the length changes are looked at, about 2 sqrt(nz) of nz
// (nz = 4000: 1.6 us, 21 over every count).
inline int fused_chunk(long columns, int nz, int R, int cus)
{
    int best = nz;
    long cost = 0;
    for (int n = 1; n <= nz;) {
        const int zc = (nz + n - 1) / n;
        const long groups = columns * ((nz + zc - 1) / zc);
        const long t = (groups + cus - 1) / cus * (zc + 2 * R);
        if (n == 1 || t < cost) { cost = t; best = zc; }
        if (zc == 1) break;
        n = (nz + zc - 2) / (zc - 1);      // the first count with shorter chunks
    }
    return best;
}

template <int ORDER, int MODE>
void launch_fused(const VisParams &vp, ws_field u, ws_field v, ws_field w, ws_field T, const ws_metric_fields &mf,
                  ws_soa du, int cus, hipStream_t s)
{
    constexpr int R = ORDER / 2;
    using FZ = Fused<R>;
    // the four rows beside a closed face and the central form, over 60 (sixth order) or 840
    constexpr double C = ORDER == 8 ? 14.0 : 1.0;
    const double num[5][4] = {{60 * C, 0, 0, 0}, {30 * C, 0, 0, 0}, {40 * C, -5 * C, 0, 0}, {45 * C, -9 * C, C, 0},
                              {ORDER == 8 ? 672.0 : 45.0, ORDER == 8 ? -168.0 : -9.0, ORDER == 8 ? 32.0 : 1.0,
                               ORDER == 8 ? -3.0 : 0.0}};
    VisWeights wt{};
    const double aj = vp.metric[9];
    for (int d = 0; d < 3; ++d) {
        const double A = MODE == VM_DIAG ? vp.metric[4 * d] : 1.0, h = 60.0 * C * vp.h[d];
        wt.gs[d] = A / h;
        wt.fs[d] = aj * (A * aj) / h;
        for (int q = 3 * d; q < 3 * d + 3; ++q) {
            wt.gA[q] = vp.metric[q] / h;
            wt.fA[q] = aj * (vp.metric[q] * aj) / h;
        }
    }
    for (int r = 0; r < 5; ++r) {
        double sum = 0.0;
        for (int q = 3; q >= 0; --q) {
            sum += num[r][q];
            wt.row[r][q] = num[r][q];
            wt.rz[r][q] = sum;
        }
    }
    const bool bnd_xy = vp.bnd[0] || vp.bnd[1] || vp.bnd[2] || vp.bnd[3], bnd_z = vp.bnd[4] || vp.bnd[5];
    // the layout: shared pitch, planes of fewer than 2^32 bytes
    bool one = true, small = (uint64_t)du.pitch * (uint64_t)vp.ny < (1ull << 29);
    auto look = [&](const ws_field &f) {
        one = one && f.pitch == u.pitch;
        small = small && (uint64_t)f.pitch * (uint64_t)vp.nyg < (1ull << 29);
    };
    for (const ws_field &f : {u, v, w, T}) look(f);
    if (MODE == VM_FIELDS) {
        for (int q = 0; q < 9; ++q) look(mf.A[q]);
        look(mf.ajac);
    }
    const long columns = (long)((vp.nx + FZ::TX - 1) / FZ::TX) * ((vp.ny + FZ::TY - 1) / FZ::TY);
    const int zc = fused_chunk(columns, vp.nz, R, cus);
    const long ntiles = columns * ((vp.nz + zc - 1) / zc);
    const dim3 g((unsigned)(8 * ((ntiles + 7) / 8)));
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, g, dim3(FNT), 0, s, vp, wt, u, v, w, T, mf, du, zc); };
    // the closure form's table holds the central weights too: it also serves the largest planes,
    // and with several pitches any closed face.  T's pitch its own, with 64-bit addresses in the
    // closure form for every such layout / now / one pitch: 256x160x96 sixth order 467 / 179 / 177
    // us, eighth 927 / 287 / 275; x faces closed 157x111x75 184 / 129 and 362 / 239, metric fields
    // 237 / 107 and 680 / 168 before and now
    if (!small) go(k_vis_fused<ORDER, MODE, VC_ALL, VL_BIG>);
    else if (!one && (bnd_z || bnd_xy)) go(k_vis_fused<ORDER, MODE, VC_ALL, VL_PITCHES>);
    else if (!one) go(k_vis_fused<ORDER, MODE, VC_NONE, VL_PITCHES>);
    else if (bnd_z) go(k_vis_fused<ORDER, MODE, VC_ALL, VL_ONE>);
    else if (bnd_xy) go(k_vis_fused<ORDER, MODE, VC_XY, VL_ONE>);
    else go(k_vis_fused<ORDER, MODE, VC_NONE, VL_ONE>);
}

template <int ORDER, bool FIELDS, bool BND>
void launch_order_b(const VisParams &vp, ws_field u, ws_field v, ws_field w, ws_field T, const ws_metric_fields &mf,
                    const EvFields &ev, ws_soa du, const Ctx &c, hipStream_t s, int &r)
{
    const unsigned g = march_blocks(vp.nx, vp.ny, vp.nz);
    hipLaunchKernelGGL((k_vis_flux<ORDER, FIELDS, BND>), dim3(g), dim3(NT), 0, s, vp, u, v, w, T, mf, ev);
    // periodic directions only: the closure forms read no flux past a closed face
    ws_field fl[12];
    for (int q = 0; q < 12; ++q) fl[q] = ws_field{ev.f[q], ev.pitch, 0};
    if ((r = launch_ghost_fill(c, fl, 12, s))) return;
    hipLaunchKernelGGL((k_vis_div<ORDER, FIELDS, BND>), dim3(g), dim3(NT), 0, s, vp, ev, mf.ajac, du);
}

template <int ORDER, bool FIELDS>
void launch_order(const VisParams &vp, ws_field u, ws_field v, ws_field w, ws_field T, const ws_metric_fields &mf,
                  const EvFields &ev, ws_soa du, const Ctx &c, hipStream_t s, int &r)
{
    bool bnd = false;
    for (int q = 0; q < 6; ++q) bnd = bnd || vp.bnd[q];
    if (bnd) launch_order_b<ORDER, FIELDS, true>(vp, u, v, w, T, mf, ev, du, c, s, r);
    else launch_order_b<ORDER, FIELDS, false>(vp, u, v, w, T, mf, ev, du, c, s, r);
}

template <int ORDER>
void launch_fields(const VisParams &vp, ws_field u, ws_field v, ws_field w, ws_field T, const ws_metric_fields *m,
                   const EvFields &ev, ws_soa du, const Ctx &c, hipStream_t s, int &r)
{
    ws_metric_fields mf{};
    if (m) {
        mf = *m;
        launch_order<ORDER, true>(vp, u, v, w, T, mf, ev, du, c, s, r);
    } else {
        launch_order<ORDER, false>(vp, u, v, w, T, mf, ev, du, c, s, r);
    }
}

}  // namespace

int launch_viscous(Ctx &c, ws_field u, ws_field v, ws_field w, ws_field T, const ws_metric_fields *m, ws_soa du,
                   hipStream_t s)
{
    const ws_config &cfg = c.cfg;
    if (cfg.viscous != 6 && cfg.viscous != 8) return set_error(WS_ERR_INVALID, "viscous terms are off (cfg.viscous)");
    VisParams vp{};
    vp.nx = cfg.nx; vp.ny = cfg.ny; vp.nz = cfg.nz; vp.nyg = cfg.ny + 2 * LAP;
    vp.h[0] = cfg.hx; vp.h[1] = cfg.hy; vp.h[2] = cfg.hz;
    for (int q = 0; q < 6; ++q) vp.bnd[q] = cfg.d0_bound[q] ? 1 : 0;
    for (int q = 0; q < 3; ++q) vp.per[q] = cfg.periodic[q] ? 1 : 0;
    // constants as the reference's opencfd_para_init forms them (src/runtime/OCFD_init.cpp:379-396)
    vp.tsb = 110.4 / cfg.ref_t;
    vp.amu_c0 = 1.0 / cfg.re * (1.0 + 110.4 / cfg.ref_t);
    const double cp = 1.0 / ((cfg.gamma - 1.0) * cfg.ama * cfg.ama);
    vp.vis_c = cp / cfg.pr;
    for (int q = 0; q < 10; ++q) vp.metric[q] = cfg.metric[q];
    // the anchor kernel family keeps the reference's arithmetic bit for bit
    const bool exact = cfg.kernel == WS_KERNEL_ANCHOR;
    if (!exact) {
        // the fast family: one fused kernel, no scratch
        const double *A = cfg.metric;
        const bool diag = A[1] == 0.0 && A[2] == 0.0 && A[3] == 0.0 && A[5] == 0.0 && A[6] == 0.0 && A[7] == 0.0;
        const ws_metric_fields mf = m ? *m : ws_metric_fields{};
        const int mode = m ? VM_FIELDS : diag ? VM_DIAG : VM_CONST;
        auto go = [&](auto launch) { launch(vp, u, v, w, T, mf, du, c.compute_units, s); };
        if (cfg.viscous == 8) {
            // no VM_DIAG form: with the eighth order's longer windows its instance spills (the
            // general one keeps fewer values across the flux stage and does not), which costs
            // more than the general metric products (157x111x75: 190 us against 133)
            if (mode == VM_FIELDS) go(launch_fused<8, VM_FIELDS>);
            else go(launch_fused<8, VM_CONST>);
        } else {
            if (mode == VM_FIELDS) go(launch_fused<6, VM_FIELDS>);
            else if (mode == VM_DIAG) go(launch_fused<6, VM_DIAG>);
            else go(launch_fused<6, VM_CONST>);
        }
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? WS_OK : hip_error(e, "fused viscous launch");
    }
    // the two-kernel form: twelve ghosted flux fields of scratch, allocated at the first call
    const uint32_t pitch = (uint32_t)((cfg.nx + 2 * LAP + 31) / 32 * 32);
    const size_t per = (size_t)pitch * (cfg.ny + 2 * LAP) * (cfg.nz + 2 * LAP);
    if (!c.vis_scratch || c.vis_scratch_elems < 12 * per) {
        if (c.vis_scratch) (void)hipFree(c.vis_scratch);
        c.vis_scratch = nullptr;
        c.vis_scratch_elems = 0;
        hipError_t e = hipMalloc(&c.vis_scratch, 12 * per * sizeof(double));
        if (e != hipSuccess) { c.vis_scratch = nullptr; return set_error(WS_ERR_NOMEM, "viscous scratch allocation"); }
        c.vis_scratch_elems = 12 * per;
    }
    EvFields ev;
    for (int q = 0; q < 12; ++q) ev.f[q] = c.vis_scratch + q * per;
    ev.pitch = pitch;
    int r = WS_OK;
    if (cfg.viscous == 8) {
        launch_fields<8>(vp, u, v, w, T, m, ev, du, c, s, r);
    } else {
        launch_fields<6>(vp, u, v, w, T, m, ev, du, c, s, r);
    }
    if (r) return r;
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? WS_OK : hip_error(e, "viscous launch");
}

}  // namespace ws
