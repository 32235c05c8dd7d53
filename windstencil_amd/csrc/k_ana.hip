// k_ana.hip -- failure detection on the device: the reference's ana_NAN_and_NT (NaN and
// negative temperature over the ghosted box, src/runtime/OCFD_ana.cpp:115-225) and
// ana_Jac (negative Jacobian, :35-56), plus negative density and the CFL number of a
// given time step.
//
// One pass over the ghosted box: each work-group reduces its counts, first offending
// cells (smallest linear ghosted index) and the largest max(|u|,|v|,|w|) + c of its
// interior cells in LDS and writes one partial record; one work-group reduces the
// records.  No atomics: the report is reproducible.
#include <hip/hip_runtime.h>

#include <mutex>

#include "ws_device.h"

namespace ws {

namespace {

constexpr int AT = 256;
constexpr int ABLOCKS = 512;
constexpr int AU = 4;           // points in flight per thread
constexpr int FT = 512;         // threads of the final reduction
constexpr long long NONE = 0x7fffffffffffffffLL;

// per-quantity count and first offending ghosted index
struct AnaRec {
    long long count[4];      // NaN T, T < 0, d < 0, Ajac < 0
    long long first[4];
    double smax;             // largest max(|u|,|v|,|w|) + c over interior cells
};

__device__ __forceinline__ void rec_merge(AnaRec &a, const AnaRec &b)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        a.count[q] += b.count[q];
        a.first[q] = min(a.first[q], b.first[q]);
    }
    a.smax = fmax(a.smax, b.smax);
}

// r of thread 0: the work-group's NTH records merged (every thread calls it), within each
// wavefront by lane exchanges, then over the wavefronts
template <int NTH>
__device__ __forceinline__ void rec_reduce(AnaRec &r)
{
    __shared__ AnaRec wave[NTH / 64];
    auto fold = [&](int o) {
        AnaRec b;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            b.count[q] = __shfl_xor(r.count[q], o);
            b.first[q] = __shfl_xor(r.first[q], o);
        }
        b.smax = __shfl_xor(r.smax, o);
        rec_merge(r, b);
    };
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) fold(o);
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = r;
    __syncthreads();
    if (threadIdx.x < 64) {
        r = wave[threadIdx.x & (NTH / 64 - 1)];
#pragma unroll
        for (int o = NTH / 128; o > 0; o >>= 1) fold(o);
    }
}

__global__ void __launch_bounds__(AT) k_ana_partial(KParams k, ws_field d, ws_field u, ws_field v, ws_field w,
                                                    ws_field T, ws_field ajac, AnaRec *partial)
{
    AnaRec r;
#pragma unroll
    for (int q = 0; q < 4; ++q) { r.count[q] = 0; r.first[q] = NONE; }
    r.smax = 0.0;
    const int nxg = k.nx + 2 * LAP;
    const long long total = (long long)nxg * k.nyg * k.nzg;
    const long long stride = (long long)gridDim.x * AT;
    for (long long i0 = (long long)blockIdx.x * AT + threadIdx.x; i0 < total; i0 += AU * stride) {
        // the loads of AU points go out together; points past the end repeat the last one and
        // are not counted, and ghost points read the velocities of the nearest interior cell,
        // which are not used
        double tv[AU], dv[AU], jv[AU], uv[AU], vv[AU], wv[AU];
        bool interior[AU];
#pragma unroll
        for (int q = 0; q < AU; ++q) {
            const long long i = min(i0 + q * stride, total - 1);
            int x, y, z;
            if (total <= 0xffffffffLL) {   // a 32-bit division costs a tenth of a 64-bit one
                const uint32_t row = (uint32_t)i / (uint32_t)nxg;
                x = (int)((uint32_t)i - row * (uint32_t)nxg);
                z = (int)(row / (uint32_t)k.nyg);
                y = (int)(row - (uint32_t)z * (uint32_t)k.nyg);
            } else {
                x = (int)(i % nxg); y = (int)((i / nxg) % k.nyg); z = (int)(i / ((long long)nxg * k.nyg));
            }
            tv[q] = T.ptr[fidx(T.pitch, k.nyg, x, y, z)];
            dv[q] = d.ptr[fidx(d.pitch, k.nyg, x, y, z)];
            jv[q] = ajac.ptr ? ajac.ptr[fidx(ajac.pitch, k.nyg, x, y, z)] : k.ajac;
            const int cx = min(max(x, LAP), LAP + k.nx - 1), cy = min(max(y, LAP), LAP + k.ny - 1),
                      cz = min(max(z, LAP), LAP + k.nz - 1);
            interior[q] = cx == x && cy == y && cz == z;
            uv[q] = u.ptr[fidx(u.pitch, k.nyg, cx, cy, cz)];
            vv[q] = v.ptr[fidx(v.pitch, k.nyg, cx, cy, cz)];
            wv[q] = w.ptr[fidx(w.pitch, k.nyg, cx, cy, cz)];
        }
#pragma unroll
        for (int q = 0; q < AU; ++q) {
            const long long i = i0 + q * stride;
            if (i >= total) break;
            const bool bad[4] = {isnan(tv[q]), tv[q] < 0.0, dv[q] < 0.0, jv[q] < 0.0};
#pragma unroll
            for (int n = 0; n < 4; ++n)
                if (bad[n]) {
                    ++r.count[n];
                    r.first[n] = min(r.first[n], i);
                }
            if (interior[q] && tv[q] >= 0.0) {
                const double c = sqrt(tv[q]) / k.ama;
                r.smax = fmax(r.smax, fmax(fabs(uv[q]), fmax(fabs(vv[q]), fabs(wv[q]))) + c);
            }
        }
    }
    rec_reduce<AT>(r);
    if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

__global__ void __launch_bounds__(FT) k_ana_final(const AnaRec *partial, int n, AnaRec *out)
{
    AnaRec r;
#pragma unroll
    for (int q = 0; q < 4; ++q) { r.count[q] = 0; r.first[q] = NONE; }
    r.smax = 0.0;
    for (int i = threadIdx.x; i < n; i += FT) rec_merge(r, partial[i]);
    rec_reduce<FT>(r);
    if (threadIdx.x == 0) *out = r;
}

// Device scratch of ws_ana_state_noalloc: the partial records of k_ana_partial and the
// final record.  Fixed size (ABLOCKS + 1 records of 72 bytes, about 37 KB) whatever the
// box, since the pass is grid-strided over ABLOCKS work-groups; each device holds its own
// copy until the process ends.  In host code `scratch` names the host-side shadow, not the
// device array: kernels get the address hipGetSymbolAddress returns for the current
// device (ana_scratch_ptr), never `scratch` itself.
constexpr int ANA_SCRATCH_RECS = ABLOCKS + 1;
static __device__ __align__(256) AnaRec scratch[ANA_SCRATCH_RECS];
// The same for ws_ana_state, one call per device at a time (held under g_ana_busy until the
// call's last work has ended; a call that finds it taken allocates its own): an allocation
// and a free on every call cost more than the pass over a middling box.
static __device__ __align__(256) AnaRec scratch_state[ANA_SCRATCH_RECS];

constexpr int ANA_MAX_DEVICES = 64;
std::mutex g_ana_mutex;
AnaRec *g_ana_scratch[ANA_MAX_DEVICES][2] = {};
std::mutex g_ana_busy[ANA_MAX_DEVICES];
AnaRec *g_ana_host[ANA_MAX_DEVICES] = {};    // pinned result of ws_ana_state, under g_ana_busy

// The device address of `scratch` (which 0) or `scratch_state` (which 1) on the current device
// `dev`, looked up once per device.
int ana_scratch_ptr(int dev, int which, AnaRec **out)
{
    if (dev < 0 || dev >= ANA_MAX_DEVICES) return set_error(WS_ERR_UNSUPPORTED, "device index beyond 64");
    std::lock_guard<std::mutex> lock(g_ana_mutex);
    AnaRec *&at = g_ana_scratch[dev][which];
    if (!at) {
        void *ptr = nullptr;
        hipError_t e = which ? hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch_state))
                             : hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) return hip_error(e, "analysis scratch: hipGetSymbolAddress");
        at = static_cast<AnaRec *>(ptr);
    }
    *out = at;
    return WS_OK;
}

// The pass and its report; buf holds ABLOCKS + 1 records of device memory.  Every record
// is written before it is read, so buf needs no clearing between calls.  host: pinned memory
// the result is written to by the kernel itself (null: a copy from buf's last record).
int ana_run(ws_ctx *c, const ws_state *st, const ws_metric_fields *metrics, double dt, ws_ana_report *rep,
            hipStream_t s, AnaRec *buf, AnaRec *host = nullptr)
{
    const KParams &k = c->kp;
    const ws_field aj = metrics ? metrics->ajac : ws_field{};
    hipLaunchKernelGGL(k_ana_partial, dim3(ABLOCKS), dim3(AT), 0, s, k, st->d, st->u, st->v, st->w, st->T, aj, buf);
    hipLaunchKernelGGL(k_ana_final, dim3(1), dim3(FT), 0, s, (const AnaRec *)buf, ABLOCKS, host ? host : buf + ABLOCKS);
    AnaRec r{};
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && !host) e = hipMemcpyAsync(&r, buf + ABLOCKS, sizeof(AnaRec), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return hip_error(e, "state analysis");
    if (host) r = *host;
    const long long nxg = k.nx + 2 * LAP, nyg = k.nyg;
    int64_t *cnt[4] = {&rep->nan_T, &rep->neg_T, &rep->neg_d, &rep->neg_jac};
    int32_t *first[4] = {rep->first_nan_T, rep->first_neg_T, rep->first_neg_d, rep->first_neg_jac};
    for (int q = 0; q < 4; ++q) {
        *cnt[q] = r.count[q];
        if (r.first[q] == NONE) {
            first[q][0] = first[q][1] = first[q][2] = WS_ANA_NONE;
        } else {
            const long long i = r.first[q];
            first[q][0] = (int32_t)(i % nxg) - LAP;
            first[q][1] = (int32_t)((i / nxg) % nyg) - LAP;
            first[q][2] = (int32_t)(i / (nxg * nyg)) - LAP;
        }
    }
    const double hmin = fmin(k.h[0], fmin(k.h[1], k.h[2]));
    rep->cfl = dt > 0.0 ? dt * r.smax / hmin : 0.0;
    rep->fatal = (rep->nan_T > 0 || rep->neg_T > 10) ? 1 : 0;
    return WS_OK;
}

int ana_check(ws_ctx *c, const ws_state *st, const ws_metric_fields *metrics, ws_ana_report *rep)
{
    if (!c || !st || !rep) return set_error(WS_ERR_INVALID, "null argument");
    if (!st->d.ptr || !st->u.ptr || !st->v.ptr || !st->w.ptr || !st->T.ptr)
        return set_error(WS_ERR_INVALID, "state primitives not allocated");
    if (metrics && !metrics->ajac.ptr) return set_error(WS_ERR_INVALID, "metric fields without Ajac");
    // the ghosted linear index of the pass and of the first offending cells is 64-bit
    const long long cells = (long long)(c->kp.nx + 2 * LAP) * c->kp.nyg * c->kp.nzg;
    if (cells <= 0 || cells > (1LL << 40)) return set_error(WS_ERR_INVALID, "ghosted box too large for the analysis pass");
    return WS_OK;
}

}  // namespace

}  // namespace ws

using namespace ws;

extern "C" int ws_ana_state(ws_ctx *c, const ws_state *st, const ws_metric_fields *metrics, double dt,
                            ws_ana_report *rep, hipStream_t s)
{
    int r = ana_check(c, st, metrics, rep);
    if (r) return r;
    int dev = 0;
    AnaRec *buf = nullptr;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < ANA_MAX_DEVICES) {
        std::unique_lock<std::mutex> busy(g_ana_busy[dev], std::try_to_lock);
        if (busy.owns_lock() && ana_scratch_ptr(dev, 1, &buf) == WS_OK) {
            AnaRec *&host = g_ana_host[dev];
            if (!host && hipHostMalloc((void **)&host, sizeof(AnaRec), hipHostMallocDefault) != hipSuccess) {
                host = nullptr;
                (void)hipGetLastError();
            }
            r = ana_run(c, st, metrics, dt, rep, s, buf, host);
            if (r) (void)hipStreamSynchronize(s);   // nothing of a failed call still writes it
            return r;
        }
    }
    hipError_t e = hipMalloc(&buf, sizeof(AnaRec) * ANA_SCRATCH_RECS);
    if (e != hipSuccess) return hip_error(e, "analysis scratch");
    r = ana_run(c, st, metrics, dt, rep, s, buf);
    (void)hipFree(buf);
    return r;
}

extern "C" int ws_ana_state_noalloc(ws_ctx *c, const ws_state *st, const ws_metric_fields *metrics, double dt,
                                    ws_ana_report *rep, hipStream_t s)
{
    int r = ana_check(c, st, metrics, rep);
    if (r) return r;
    AnaRec *buf = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_error(e, "hipGetDevice");
    if ((r = ana_scratch_ptr(dev, 0, &buf))) return r;
    return ana_run(c, st, metrics, dt, rep, s, buf);
}
