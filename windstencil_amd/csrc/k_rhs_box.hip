// k_rhs_box.hip -- LDS-tiled inviscid RHS of small jobs, FP64 and mixed: one launch for all
// three directions.
//
// The directional launches of rhs_tile.h want some thousand tiles in flight: a grid of
// 64x32x16 cells gives each of them about 100 work-groups for 256 compute units, so a launch
// takes as long as one work-group does and the three follow one another.  Here a work-group
// owns a cube of 4^3 cells and does the three directions together, so a small grid spreads
// over the chip, every cell's flux differences meet in registers, and du is written once (or
// the RK3 stage applied at once).
// Faces and cells are computed by the expressions of rhs_tile.h and summed in the same order
// (dir_order), so du has the bits of the directional launches.
#include "rhs_tile.h"
#include "ws_ghost.h"

namespace ws {

namespace {

constexpr int B = 4;                           // edge of the cube
constexpr int BOX_NT = 256;
constexpr int BOX_NL = B + 2 * LAP;            // points per line
constexpr int BOX_F = B + 1;                   // faces per line
constexpr int BOX_LINES = B * B;               // lines per direction
constexpr int BOX_LT = 3 * BOX_LINES;          // lines of the three directions
constexpr int BOX_CELLS = B * B * B;
constexpr int BOX_DPTS = BOX_LINES * BOX_NL;   // points per direction
constexpr int BOX_NPTS = 3 * BOX_DPTS;
constexpr int BOX_ROUNDS = (BOX_NPTS + BOX_NT - 1) / BOX_NT;
static_assert(BOX_DPTS % 64 == 0, "a wavefront's points lie in one direction");
static_assert(BOX_LT * 5 <= BOX_NT && BOX_CELLS <= BOX_NT, "a thread per line and variable, and per cell");

// LDS index of quantity q (P 0..4, M 5..9) at point p of line l (directions one after the
// other): consecutive lines are consecutive doubles, which the threads of a wavefront read
// and, in y and z, write together
__device__ constexpr int box_pidx(int q, int p, int l) { return (q * BOX_NL + p) * BOX_LT + l; }
// the face fluxes reuse the buffer, line-major: with an odd number of faces per line both the
// writes (consecutive lines) and the reads (consecutive cells) spread over the banks
__device__ constexpr int box_fidx(int m, int l, int f) { return (m * BOX_LT + l) * BOX_F + f; }

// the helper kernels' sound speed
__device__ __forceinline__ double sound_speed(double T, double ama)
{
#pragma clang fp contract(off)
    return sqrt(T) / ama;
}

// this thread's point of round r: direction (the same for a whole wavefront), line and point;
// false: none (a valid point all the same).  Along x consecutive threads take 4 points of 16
// lines: loads of 32-byte runs, LDS writes two to a bank.
__device__ __forceinline__ bool box_point(int r, int &dir, int &l, int &p)
{
    const int g = (int)threadIdx.x + r * BOX_NT;
    const bool in = g < BOX_NPTS;
    int q = min(g, BOX_NPTS - 1);
    dir = __builtin_amdgcn_readfirstlane(q / BOX_DPTS);
    q -= dir * BOX_DPTS;
    if (dir == 0) { p = (q & 3) + q / (4 * BOX_LINES) * 4; l = (q >> 2) % BOX_LINES; }
    else          { l = q % BOX_LINES; p = q / BOX_LINES; }
    return in;
}

// What bounds it: on a small grid the chain load - split - reconstruct - store of one cube,
// with one to three cubes per compute unit to overlap it; on a larger one the FP64 issue.
// Both want few operations, so one thread reconstructs all five faces of one line and
// variable, which share the window's differences: 135 FP64 operations per face (with a thread
// per face 64x32x16 took 9.5 us, 100x60x40 52).  Cubes of 8^3 cells through the three
// directions in turn took 19-23 us on a grid of any small size.
// FP64 RHS, the directional launches and this kernel: 64x32x16 24.0 / 8.9 us, 48x48x48 35.0 /
// 20.5 us, 100x60x40 52.6 / 39.1; an RK3 step of 64x32x16 77.7 / 34.9 us.
// PREP: the launch also prepares its inputs: these work-groups read the interior primitives, by
// their periodic images past a periodic face, and take the sound speed of the T they read;
// the work-groups after them write the ghost points and the sound speed (prepare_points),
// which nothing in the launch reads (du_comput of 64x32x16 12.9 -> 9.6 us against preparing in a
// launch before, of 100x60x40 47.2 -> 44.0).
template <bool FIELDS, bool MIX, bool STG, bool PREP>
__global__ void __launch_bounds__(BOX_NT, 3)
k_rhs_box(KParams k, ws_field d, ws_field u, ws_field v, ws_field w, ws_field cc, ws_metric_fields mf, ws_soa du,
          Box box, int gx, int gy, int ntiles, int order, int accumulate, StageArgs sa, BoxPrep pr)
{
    static_assert(!(STG && PREP), "a stage's inputs are prepared by the stage before it");
    constexpr int K = BOX_F;
    __shared__ double sp[10 * BOX_NPTS];
    // cubes in x-fastest order, a contiguous range of them per XCD (as k_rhs_tile)
    const int per = (ntiles + 7) / 8;
    if (PREP && (int)blockIdx.x >= 8 * per) {
        prepare_points<1, BOX_NT>(FieldList{{d, u, v, w, pr.T}}, cc, k.nx, k.ny, k.nz, pr.per[0], pr.per[1], pr.per[2],
                                  k.ama, (long)((int)blockIdx.x - 8 * per) * BOX_NT + threadIdx.x);
        return;
    }
    const int tile = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
    if (tile >= ntiles) return;
    const int trow = tile / gx;
    const int x0 = box.s[0] + (tile - trow * gx) * B, y0 = box.s[1] + trow % gy * B, z0 = box.s[2] + trow / gy * B;
    // cells of the cube inside the box
    const int lx = min(B, box.e[0] - x0), ly = min(B, box.e[1] - y0), lz = min(B, box.e[2] - z0);
    const int t = threadIdx.x;

    // ---- loads: primitives (and metric terms) of this thread's points; points that no face
    // inside the box reaches repeat one that does (their values go to no stored face)
    double ld[BOX_ROUNDS][FIELDS ? 8 : 5];
#pragma unroll
    for (int r = 0; r < BOX_ROUNDS; ++r) {
        int dir, l, p;
        box_point(r, dir, l, p);
        const int a = min(l % B, (dir == 0 ? ly : lx) - 1), b = min(l / B, (dir == 2 ? ly : lz) - 1);
        const int c = min(p, (dir == 0 ? lx : dir == 1 ? ly : lz) + 2 * LAP - 1);
        // from the first point of the direction's lines
        const int bx = x0 - (dir == 0 ? LAP : 0), by = y0 - (dir == 1 ? LAP : 0), bz = z0 - (dir == 2 ? LAP : 0);
        const uint32_t px = dir == 0 ? c : a, py = dir == 1 ? c : dir == 0 ? a : b, pz = dir == 2 ? c : b;
        auto off = [&](const ws_field &f) { return 8u * (px + f.pitch * (py + (uint32_t)k.nyg * pz)); };
        auto base = [&](const ws_field &f) { return f.ptr + origin(f.pitch, k.nyg, bx, by, bz); };
        const ws_field in[5] = {d, u, v, w, PREP ? pr.T : cc};
        if constexpr (PREP) {
            // a halo point's image inside the box
            auto image = [](int g, int n, int periodic) {
                return !periodic ? g : g < LAP ? g + n : g >= n + LAP ? g - n : g;
            };
            const int ix = image(bx + (int)px, k.nx, pr.per[0]), iy = image(by + (int)py, k.ny, pr.per[1]),
                      iz = image(bz + (int)pz, k.nz, pr.per[2]);
#pragma unroll
            for (int q = 0; q < 5; ++q) ld[r][q] = in[q].ptr[fidx(in[q].pitch, k.nyg, ix, iy, iz)];
        } else if (k.same_pitch) {
            const uint32_t o = off(d);
#pragma unroll
            for (int q = 0; q < 5; ++q) ld[r][q] = elem(base(in[q]), o);
        } else {
#pragma unroll
            for (int q = 0; q < 5; ++q) ld[r][q] = elem(base(in[q]), off(in[q]));
        }
        if constexpr (FIELDS) {
#pragma unroll
            for (int q = 0; q < 3; ++q) ld[r][5 + q] = elem(base(mf.A[3 * dir + q]), off(mf.A[3 * dir + q]));
        }
    }

    // this thread's cell (threads past the last cell, and cells past the box: none)
    const int ix = t % B, iy = t / B % B, iz = t / (B * B);
    const bool cell = t < BOX_CELLS && ix < lx && iy < ly && iz < lz;
    auto ghosted = [&](const ws_field &f) -> double & {
        return elem(f.ptr + origin(f.pitch, k.nyg, x0, y0, z0),
                    8u * ((uint32_t)ix + f.pitch * ((uint32_t)iy + (uint32_t)k.nyg * (uint32_t)iz)));
    };
    auto state = [&](const ws_soa &f, int m) -> double & {
        return elem(f.ptr + (size_t)m * f.pitch * k.ny * k.nz + origin(f.pitch, k.ny, x0 - LAP, y0 - LAP, z0 - LAP),
                    8u * ((uint32_t)ix + f.pitch * ((uint32_t)iy + (uint32_t)k.ny * (uint32_t)iz)));
    };
    double acc[5] = {}, fnv[5] = {}, fvv[5] = {};
    double aj = k.ajac;
    if (cell) {
        if (FIELDS) aj = ghosted(mf.ajac);
        if (STG) {
#pragma unroll
            for (int m = 0; m < 5; ++m) fnv[m] = state(sa.fn, m);
            if (sa.krk != 1)
#pragma unroll
                for (int m = 0; m < 5; ++m) fvv[m] = state(sa.f, m);
        } else if (accumulate) {
#pragma unroll
            for (int m = 0; m < 5; ++m) acc[m] = state(du, m);
        }
    }

    // ---- split every point into LDS ----------------------------------------------------------
#pragma unroll
    for (int r = 0; r < BOX_ROUNDS; ++r) {
        int dir, l, p;
        if (!box_point(r, dir, l, p)) continue;
        const double dd = ld[r][0], uu = ld[r][1], vv = ld[r][2], ww = ld[r][3];
        const double c = PREP ? sound_speed(ld[r][4], k.ama) : ld[r][4];
        double fp[5], fm[5];
        if (FIELDS) {
            const double A1 = ld[r][FIELDS ? 5 : 0], A2 = ld[r][FIELDS ? 6 : 0], A3 = ld[r][FIELDS ? 7 : 0];
            if (MIX) {
                const double sn = sqrt(fma(A3, A3, fma(A2, A2, A1 * A1)));
                const double rs = 1.0 / sn;
                split_mixed(k, dd, uu, vv, ww, c, A1, A2, A3, sn, A1 * rs, A2 * rs, A3 * rs, fp, fm);
            } else {
                double sn, rs;
                sqrt_rsqrt_h(fma(A3, A3, fma(A2, A2, A1 * A1)), sn, rs);
                split_fast(k, dd, uu, vv, ww, c, A1, A2, A3, sn, rs, fp, fm);
            }
        } else {
            const double A1 = k.A[3 * dir], A2 = k.A[3 * dir + 1], A3 = k.A[3 * dir + 2];
            if (MIX)
                split_mixed(k, dd, uu, vv, ww, c, A1, A2, A3, k.Anorm[dir], k.Ak[3 * dir], k.Ak[3 * dir + 1],
                            k.Ak[3 * dir + 2], fp, fm);
            else
                split_fast(k, dd, uu, vv, ww, c, A1, A2, A3, k.Anorm[dir], k.Arnorm[dir], fp, fm);
        }
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            sp[box_pidx(m, p, dir * BOX_LINES + l)] = fp[m];
            sp[box_pidx(5 + m, p, dir * BOX_LINES + l)] = fm[m];
        }
    }
    __syncthreads();

    // ---- reconstruct: the faces of line tl, variable m ------------------------------------------
    const int tl = t % BOX_LT, var = t / BOX_LT;
    double Fv[K];
    if (var < 5) {
        const double *qp = sp + box_pidx(var, 0, tl), *qm = sp + box_pidx(5 + var, 0, tl);
        if (MIX) {
            double bP[K], bM[K];
            float cP[K], cM[K];
            unsigned badP, badM;
            weno_k_mixed<false, K>([&](int j) { return qp[j * BOX_LT]; }, bP, cP, badP);
            weno_k_mixed<true, K>([&](int j) { return qm[j * BOX_LT]; }, bM, cM, badM);
#pragma unroll
            for (int j = 0; j < K; ++j) Fv[j] = (bP[j] + bM[j]) + (double)(cP[j] + cM[j]);
            // FP32 weights out of FP32's range: both halves again in FP64 (as in rhs_tile.h)
            const unsigned bad = badP | badM;
            if (bad) {
#pragma unroll 1
                for (int j = 0; j < K; ++j) {
                    if (!((bad >> j) & 1u)) continue;
                    double nP[1], dP[1], cP1[1], nM[1], dM[1], cM1[1];
                    weno_k<false, 1>([&](int i) { return qp[(i + j) * BOX_LT]; }, nP, dP, cP1);
                    weno_k<true, 1>([&](int i) { return qm[(i + j) * BOX_LT]; }, nM, dM, cM1);
                    const double val = face_merge(nP[0], dP[0], cP1[0], nM[0], dM[0], cM1[0]);
#pragma unroll
                    for (int q = 0; q < K; ++q)
                        if (q == j) Fv[q] = val;
                }
            }
        } else {
            double nP[K], dP[K], nM[K], dM[K], bP[K], bM[K];
            weno_k<false, K>([&](int j) { return qp[j * BOX_LT]; }, nP, dP, bP);
            weno_k<true, K>([&](int j) { return qm[j * BOX_LT]; }, nM, dM, bM);
#pragma unroll
            for (int j = 0; j < K; ++j) Fv[j] = face_merge(nP[j], dP[j], bP[j], nM[j], dM[j], bM[j]);
        }
        // finished here (the compiler would otherwise carry the parts to the store below)
#pragma unroll
        for (int j = 0; j < K; ++j) asm volatile("" : "+v"(Fv[j]));
    }
    __syncthreads();
    if (var < 5)
#pragma unroll
        for (int j = 0; j < K; ++j) sp[box_fidx(var, tl, j)] = Fv[j];
    __syncthreads();

    // ---- flux differences of this thread's cell, summed in the order of the directional launches
    double cmax = 0.0;
    if (cell) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int dir = order == WS_ORDER_ZYX ? 2 - q : q;
            const int i = dir == 0 ? ix : dir == 1 ? iy : iz;
            const int line = dir * BOX_LINES + (dir == 0 ? iy : ix) + B * (dir == 2 ? iy : iz);
            const double scale = aj * -k.rh[dir];
#pragma unroll
            for (int m = 0; m < 5; ++m) {
                const double val = scale * (sp[box_fidx(m, line, i + 1)] - sp[box_fidx(m, line, i)]);
                acc[m] = q == 0 && !accumulate ? val : acc_sum(acc[m], val);
            }
        }
        if (STG)
            cmax = stage_cell(k, sa, x0 + ix, y0 + iy, z0 + iz, ghosted, fnv, fvv, sa.dt_dev ? *sa.dt_dev : sa.dt, acc);
        const ws_soa &out = STG ? sa.f : du;
#pragma unroll
        for (int m = 0; m < 5; ++m) state(out, m) = acc[m];
    }
    if (STG && sa.cfl_part) {
        // the cells are the first wavefront's, so its lanes hold every maximum
        if (t < 64) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) cmax = fmax(cmax, __shfl_xor(cmax, o));
            if (t == 0) sa.cfl_part[tile] = cmax;
        }
    }
}

dim3 box_grid(const Box &box)
{
    return dim3((box.e[0] - box.s[0] + B - 1) / B, (box.e[1] - box.s[1] + B - 1) / B, (box.e[2] - box.s[2] + B - 1) / B);
}

}  // namespace

bool box_serves(const Ctx &c, const ws_job &job)
{
    if (!c.box || c.kp.bnd_any[0] || c.kp.bnd_any[1] || c.kp.bnd_any[2]) return false;
    const long n = (long)(job.end.x - job.start.x) * (long)(job.end.y - job.start.y) * (long)(job.end.z - job.start.z);
    // 1400 cells per compute unit, 358 thousand on 256.  du_comput by cubes / by tiles, in us:
    //   thousand cells      196        262        319        368        409        460        589
    //   FP64             42.5/54.1  49.7/60.3  61.5/68.8  68.5/75.4  74.1/74.7  85.2/84.8  106/99.6
    //   mixed            37.6/53.9  50.3/59.5  61.6/66.7  69.6/74.2  79.6/72.9  87.5/83.1  111/98.0
    //   metric fields    45.2/54.1  55.4/59.1  66.0/68.9  77.0/77.2  83.8/76.3  94.3/90.3  117/104
    // RK3 steps cross between 368 (203/220) and 422 (255/250).  Then the tiles fill the chip, and
    // split 1.27 points per cell and direction where a cube splits 3.  Cells and not cubes are
    // counted: a job thinner than a cube leaves cubes partly empty, but tiles more so (600x256x1
    // 95/101, 300x128x1 29/39, 1x256x16 8/25).
    return n <= 1400l * c.compute_units;
}

long box_launch_tiles(const ws_job &job)
{
    const dim3 g = box_grid(job_box(job));
    return (long)g.x * g.y * g.z;
}

void launch_rhs_box(bool mixed, const KParams &k, ws_field d, ws_field u, ws_field v, ws_field w, ws_field cc,
                    const ws_metric_fields *m, ws_soa du, const ws_job &job, int order, int accumulate,
                    const StageArgs *sa, const BoxPrep *prep, hipStream_t s)
{
    const Box box = job_box(job);
    const dim3 g = box_grid(box);
    const int n = (int)(g.x * g.y * g.z);
    if (n <= 0) return;
    const ws_metric_fields mf = m ? *m : ws_metric_fields{};
    auto go = [&](auto kern) {
        const long points = prep ? (long)(k.nx + 2 * LAP) * k.nyg * k.nzg : 0;
        hipLaunchKernelGGL(kern, dim3(8 * ((n + 7) / 8) + (unsigned)((points + BOX_NT - 1) / BOX_NT)), dim3(BOX_NT), 0, s, k,
                           d, u, v, w, cc, mf, du, box, (int)g.x, (int)g.y, n, order, accumulate, sa ? *sa : StageArgs{},
                           prep ? *prep : BoxPrep{});
    };
    if (mixed) {
        if (sa) go(k_rhs_box<false, true, true, false>);
        else if (m && prep) go(k_rhs_box<true, true, false, true>);
        else if (m) go(k_rhs_box<true, true, false, false>);
        else if (prep) go(k_rhs_box<false, true, false, true>);
        else go(k_rhs_box<false, true, false, false>);
    } else {
        if (sa) go(k_rhs_box<false, false, true, false>);
        else if (m && prep) go(k_rhs_box<true, false, false, true>);
        else if (m) go(k_rhs_box<true, false, false, false>);
        else if (prep) go(k_rhs_box<false, false, false, true>);
        else go(k_rhs_box<false, false, false, false>);
    }
}

int launch_prepared_rhs(const Ctx &c, const ws_state &st, const ws_metric_fields *m, bool *done, hipStream_t s)
{
    const ws_job job = interior_job(&c);
    KParams k = c.kp;
    *done = c.cfg.kernel == WS_KERNEL_TILED && box_serves(c, job) && (!m || !plane_reach(k, *m)) &&
            !plane_reach(k, {st.d, st.u, st.v, st.w, st.T, st.cc}, {st.du});
    if (!*done) return WS_OK;
    k.same_pitch = same_pitch(st.d, st.u, st.v, st.w, st.cc) ? 1 : 0;
    const BoxPrep prep{st.T, {c.cfg.periodic[0], c.cfg.periodic[1], c.cfg.periodic[2]}};
    launch_rhs_box(c.cfg.precision == WS_PREC_MIXED, k, st.d, st.u, st.v, st.w, st.cc, m, st.du, job, c.dir_order, 0,
                   nullptr, &prep, s);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? WS_OK : hip_error(e, "one-launch du_comput");
}

}  // namespace ws
