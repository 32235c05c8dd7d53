"""The work a program has this framework do, as cases that can be timed and compared.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the inputs, context, state and tuning a program holds before the call
    run(state)          one pass through the public entry points, and its outputs
    work(case)          bytes and operations of one pass that no implementation can do without
    exact(case, seed)   the outputs of a first pass in plain 64-bit torch

A case's "kind" says what is called:

    rhs      ws_du_comput of one box: ghost fill, sound speed, inviscid RHS and, with "viscous"
             6 or 8, the viscous terms; "metrics": per-cell metric fields; "closed": the x faces
             are domain faces with the one-sided closures instead of periodic ones
    rk3      ws_rk3_run: "steps" SSP-RK3 steps at CFL 0.5, the step captured in a graph
    batch    "blocks" blocks of uneven size advanced together: ws_batch_du_comput, or with
             "steps" ws_batch_rk3_run
    monitor  the state check of a solver loop: the CFL step and the failure detection

"tuned": the program calls the autotuner once before its loop, as one that keeps a large box or
a batch for thousands of steps does; the others run a context as it is created.
"""
import ctypes
import math
import random

import torch

import windstencil_amd as W

GAMMA = 1.4
CFL = 0.5
RE, PR, REF_T = 1000.0, 0.72, 288.15
EPSL = 1e-3
MONITOR_DT = 1e-4
LAP = W.LAP

# algorithmic operations per cell: the inviscid RHS, and the viscous terms by order
FLOPS_RHS = 7431
FLOPS_VISCOUS = {0: 0, 6: 621, 8: 693}

MOST_CELL_RHS = 12 * 600 * 128 * 128      # cells times RHS evaluations of the largest listed case
MOST_CELLS = 600 * 256 * 128


def listed():
    return [
        # the CPU-path workload: one evaluation and a short run of a small Mach 2 box, where
        # launches and latency count
        {"name": "rhs_64x32x16", "kind": "rhs", "nx": 64, "ny": 32, "nz": 16, "flow": "blobs"},
        {"name": "rk3_64x32x16", "kind": "rk3", "nx": 64, "ny": 32, "nz": 16, "flow": "blobs", "steps": 10},
        # the headline box in both precisions: a program that evaluates the RHS inside its own
        # time integrator
        {"name": "rhs_600x256x128", "kind": "rhs", "nx": 600, "ny": 256, "nz": 128, "flow": "sod", "tuned": True},
        {"name": "rhs_600x256x128_mixed", "kind": "rhs", "nx": 600, "ny": 256, "nz": 128, "flow": "sod",
         "mixed": True, "tuned": True},
        # Navier-Stokes of a middle-sized box, sixth-order viscous terms
        {"name": "ns6_600x128x128", "kind": "rhs", "nx": 600, "ny": 128, "nz": 128, "flow": "vortex", "viscous": 6},
        # an odd box between two domain faces, sixth-order viscous terms
        {"name": "closed_ns6_211x93x67", "kind": "rhs", "nx": 211, "ny": 93, "nz": 67, "flow": "vortex",
         "viscous": 6, "closed": True},
        # a curvilinear mesh: metric terms read per cell, eighth-order viscous terms
        {"name": "curv_ns8_256x160x96", "kind": "rhs", "nx": 256, "ny": 160, "nz": 96, "flow": "vortex",
         "viscous": 8, "metrics": True},
        # the drop-in time integration
        {"name": "rk3_600x128x128", "kind": "rk3", "nx": 600, "ny": 128, "nz": 128, "flow": "vortex", "steps": 4,
         "tuned": True},
        # Navier-Stokes time steps of an odd box, eighth-order viscous terms
        {"name": "rk3_ns8_157x111x75", "kind": "rk3", "nx": 157, "ny": 111, "nz": 75, "flow": "vortex", "steps": 3,
         "viscous": 8},
        # many uneven blocks: one evaluation, and mixed-precision time steps
        {"name": "batch_rhs_16", "kind": "batch", "blocks": 16, "lo": 32, "hi": 160, "extents_seed": 1,
         "tuned": True},
        {"name": "batch_rk3_12_mixed", "kind": "batch", "blocks": 12, "lo": 24, "hi": 112, "extents_seed": 2,
         "steps": 3, "mixed": True, "tuned": True},
        # the check a solver loop makes between its steps
        {"name": "monitor_600x128x128", "kind": "monitor", "nx": 600, "ny": 128, "nz": 128, "flow": "vortex"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rhs", "rhs", "rhs", "rk3", "rk3", "batch", "monitor"])
    if kind == "batch":
        c = {"kind": "batch", "blocks": rng.randint(4, 20), "lo": rng.randint(20, 40), "hi": rng.randint(64, 144),
             "extents_seed": rng.randint(3, 10 ** 6), "tuned": True}
        if rng.random() < 0.5:
            c["steps"] = rng.randint(2, 4)
        if rng.random() < 0.4:
            c["mixed"] = True
        while _evaluations(c) * _cells(c) > MOST_CELL_RHS or _cells(c) > MOST_CELLS:
            c["blocks"] -= 1
        return c
    while True:
        c = {"kind": kind, "nx": _log_int(rng, 24, 640), "ny": _log_int(rng, 16, 256), "nz": _log_int(rng, 16, 160),
             "flow": rng.choice(["blobs", "vortex", "sod"])}
        if kind == "rk3":
            c["steps"] = rng.randint(2, 8)
            c["flow"] = rng.choice(["blobs", "vortex"])
        if kind in ("rhs", "rk3"):
            style = rng.choice(["euler", "euler", "euler", "ns"] if kind == "rk3" else
                               ["euler", "euler", "ns", "ns", "closed", "curvilinear"])
            if style == "euler" and rng.random() < 0.4:
                c["mixed"] = True
            if style != "euler":
                c["viscous"] = rng.choice([6, 8])
                c["flow"] = rng.choice(["blobs", "vortex"])
            if style == "closed":
                c["closed"] = True
            if style == "curvilinear":
                c["metrics"] = True
        if _cells(c) > MOST_CELLS or _evaluations(c) * _cells(c) > MOST_CELL_RHS:
            continue
        if kind in ("rhs", "rk3") and _cells(c) > 2_000_000:
            c["tuned"] = True
        return c


def _extents(case):
    if case["kind"] != "batch":
        return [(case["nx"], case["ny"], case["nz"])]
    r = random.Random(case["extents_seed"])
    return [tuple(r.randint(case["lo"], case["hi"]) for _ in range(3)) for _ in range(case["blocks"])]


def _cells(case):
    return sum(nx * ny * nz for nx, ny, nz in _extents(case))


def _evaluations(case):
    return 3 * case["steps"] if case.get("steps") else 1


def work(case):
    n = _cells(case)
    if case["kind"] == "monitor":
        # d, u, v, w, T in
        return {"bytes": 40 * n, "flops": 8 * n}
    if case.get("steps"):
        # f in; f, d, u, v, w, T and P out
        return {"bytes": (40 + 40 + 48) * n, "flops": _evaluations(case) * n * (FLOPS_RHS + FLOPS_VISCOUS[case.get("viscous", 0)])}
    # d, u, v, w, T in (and ten metric terms); du and the sound speed out
    return {"bytes": (40 + 48 + (80 if case.get("metrics") else 0)) * n,
            "flops": n * (FLOPS_RHS + FLOPS_VISCOUS[case.get("viscous", 0)])}


# ---- inputs ------------------------------------------------------------------------------------

def _spacing(n):
    return tuple(1.0 / (v - 1) for v in n)


def _flow(flow, n, seed):
    """Primitives rho, u, v, w, T of one box as (nz, ny, nx) tensors on the GPU, made from the seed."""
    nx, ny, nz = n
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    host = random.Random(seed)
    dev = dict(device="cuda", dtype=torch.float64)
    x = torch.arange(nx, **dev)[None, None, :]
    y = torch.arange(ny, **dev)[None, :, None]
    z = torch.arange(nz, **dev)[:, None, None]
    one = torch.ones((nz, ny, nx), **dev)

    def periodic(a, c, length):
        d = a - c
        return d - length * torch.round(d / length)

    def noise(size):
        return 1.0 + size * (2.0 * torch.rand((nz, ny, nx), generator=g, **dev) - 1.0)

    if flow == "sod":
        # a planar Sod discontinuity at rest with 1 % noise
        left = (x < 0.4 * nx) & (one > 0)
        rho = torch.where(left, 1.0, 0.125) * noise(0.01)
        p = torch.where(left, 1.0, 0.1) * noise(0.01)
        zero = torch.zeros_like(one)
        return rho, zero, zero.clone(), zero.clone(), GAMMA * p / rho
    if flow == "blobs":
        # a stream of Mach 2 along a direction in the x-y plane with Gaussian blobs
        rho, p = one.clone(), one.clone()
        for _ in range(8):
            c = [host.uniform(0, v) for v in n]
            r2 = periodic(x, c[0], nx) ** 2 + periodic(y, c[1], ny) ** 2 + periodic(z, c[2], nz) ** 2
            blob = torch.exp(-r2 / 32.0)
            rho += host.uniform(-0.1, 0.1) * blob
            p += host.uniform(-0.1, 0.1) * blob
        a = host.uniform(0, 0.5 * math.pi)
        return rho, one * 2.0 * math.cos(a), one * 2.0 * math.sin(a), torch.zeros_like(one), p / rho
    # isentropic vortices with axes along z on a Mach 0.5 stream, and a weak wave along z
    du, dv, dT = (torch.zeros((1, ny, nx), **dev) for _ in range(3))
    radius = max(4.0, min(nx, ny) / 16.0)
    beta = 3.0
    for _ in range(6):
        ex = periodic(x, host.uniform(0, nx), nx) / radius
        ey = periodic(y, host.uniform(0, ny), ny) / radius
        e = torch.exp(0.5 * (1.0 - ex * ex - ey * ey))
        du = du - beta / (2.0 * math.pi * math.sqrt(GAMMA)) * ey * e
        dv = dv + beta / (2.0 * math.pi * math.sqrt(GAMMA)) * ex * e
        dT = dT - (GAMMA - 1.0) * beta * beta / (8.0 * GAMMA * math.pi ** 2) * e * e
    T = torch.clamp(1.0 + dT, min=0.1) * one
    w = 0.1 * torch.sin(2.0 * math.pi * (z / nz + host.random())) * one
    return T ** (1.0 / (GAMMA - 1.0)), (0.5 + du) * one, dv * one, w, T


def _metric_fields(n, seed):
    """Ghosted metric terms Akx .. Asz, Ajac of a smooth periodic curvilinear mesh."""
    nx, ny, nz = n
    host = random.Random(seed)
    dev = dict(device="cuda", dtype=torch.float64)

    def wave(size):
        ph = [host.uniform(0, 2 * math.pi) for _ in range(3)]
        a = torch.sin(2 * math.pi * (torch.arange(-LAP, nx + LAP, **dev) / nx) + ph[0])[None, None, :]
        b = torch.sin(2 * math.pi * (torch.arange(-LAP, ny + LAP, **dev) / ny) + ph[1])[None, :, None]
        c = torch.sin(2 * math.pi * (torch.arange(-LAP, nz + LAP, **dev) / nz) + ph[2])[:, None, None]
        return size * (a + b + c)

    terms = [(1.0 if m % 4 == 0 else 0.0) + wave(0.05) for m in range(9)]
    return [t.contiguous() for t in terms + [1.0 + wave(0.05)]]


def _config(case, n, **more):
    kw = dict(precision=W.WS_PREC_MIXED if case.get("mixed") else W.WS_PREC_FP64, viscous=case.get("viscous", 0),
              re=RE, pr=PR, ref_t=REF_T, epsl_sw=EPSL, **more)
    if case.get("closed"):
        kw.update(periodic=(0, 1, 1), d0_bound=(1, 1, 0, 0, 0, 0))
    return W.default_config(*n, **kw)


def _state(case, n, seed):
    """A state with the primitives set and the conserved variables derived from them."""
    ctx = W.Context(_config(case, n))
    st = W.TorchState(*n)
    for k, a in zip(("d", "u", "v", "w", "T"), _flow(case.get("flow", "blobs"), n, seed)):
        st.interior(k).copy_(a)
        if case.get("closed"):
            # the caller's ghost layers beside the domain faces
            inner = st.t[k][LAP:-LAP, LAP:-LAP]
            inner[:, :, :LAP] = a[:, :, :1]
            inner[:, :, n[0] + LAP:n[0] + 2 * LAP] = a[:, :, -1:]
    W.check(W.lib().ws_pri_to_cons(ctx.handle, st.ws.f, st.ws.d, st.ws.u, st.ws.v, st.ws.w, st.ws.T,
                                   W.job((0, 0, 0), n), W.stream_handle()), "ws_pri_to_cons")
    return ctx, st


def prepare(case, seed):
    L, s = W.lib(), W.stream_handle()
    if case["kind"] == "batch":
        extents = _extents(case)
        states = [_state(case, n, 1000 * seed + i)[1] for i, n in enumerate(extents)]
        batch = W.Batch(_config(case, (8, 8, 8)), extents, states)
        if case.get("tuned"):
            W.check(L.ws_batch_du_comput(batch.handle, s), "ws_batch_du_comput")
            W.check(L.ws_batch_autotune(batch.handle, 3, None, s), "ws_batch_autotune")
        return {"case": case, "batch": batch}
    n = (case["nx"], case["ny"], case["nz"])
    ctx, st = _state(case, n, seed)
    state = {"case": case, "ctx": ctx, "st": st, "metrics": None}
    if case.get("metrics"):
        fields = _metric_fields(n, seed)
        m = W.WsMetricFields()
        for q in range(9):
            m.A[q] = W.field_of(fields[q])
        m.ajac = W.field_of(fields[9])
        state.update(metrics=m, metric_tensors=fields)
    if case["kind"] == "monitor":
        state["dt"] = torch.zeros(1, dtype=torch.float64, device="cuda")
    if case.get("tuned"):
        W.check(L.ws_du_comput(ctx.handle, ctypes.byref(st.ws), None, s), "ws_du_comput")
        W.check(L.ws_autotune(ctx.handle, ctypes.byref(st.ws), 3, None, s), "ws_autotune")
    return state


# ---- one pass ----------------------------------------------------------------------------------

def run(state):
    L, s, case = W.lib(), W.stream_handle(), state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        if case.get("steps"):
            W.check(L.ws_batch_rk3_run(b.handle, case["steps"], CFL, 1, s), "ws_batch_rk3_run")
            b.sync_states()
            return {"f": [st.interior("f") for st in b.states], "T": [st.interior("T") for st in b.states]}
        W.check(L.ws_batch_du_comput(b.handle, s), "ws_batch_du_comput")
        return {"du": [st.interior("du") for st in b.states]}
    ctx, st = state["ctx"], state["st"]
    if case["kind"] == "monitor":
        W.check(L.ws_cfl_dt(ctx.handle, ctypes.byref(st.ws), CFL, state["dt"].data_ptr(), s), "ws_cfl_dt")
        rep = W.WsAnaReport()
        W.check(L.ws_ana_state(ctx.handle, ctypes.byref(st.ws), None, MONITOR_DT, ctypes.byref(rep), s), "ws_ana_state")
        return {"dt": state["dt"], "cfl": rep.cfl, "fatal": rep.fatal,
                "counts": [rep.nan_T, rep.neg_T, rep.neg_d, rep.neg_jac]}
    if case["kind"] == "rk3":
        W.check(L.ws_rk3_run(ctx.handle, ctypes.byref(st.ws), case["steps"], CFL, 1, s), "ws_rk3_run")
        st.sync_from_ws()
        return {k: st.interior(k) for k in ("f", "d", "u", "v", "w", "T", "P")}
    m = ctypes.byref(state["metrics"]) if state["metrics"] is not None else None
    W.check(L.ws_du_comput(ctx.handle, ctypes.byref(st.ws), m, s), "ws_du_comput")
    return {"du": st.interior("du"), "cc": st.interior("cc")}


# ---- the same in plain 64-bit torch --------------------------------------------------------------

_FIRST = ((-2, 9, -18, 11), (1, -6, 3, 2), (-2, -3, 6, -1), (-11, 18, -9, 2), (-26, 57, -42, 11))
_SECOND = ((-6, 24, -30, 12), (0, 6, -12, 6), (0, 6, -12, 6), (12, -30, 24, -6), (18, -48, 42, -12))
_THIRD = (-6, 18, -18, 6)
_VALUE = ((-3, 13, -23, 25), (1, -5, 13, 3), (-1, 7, 7, -1), (3, 13, -5, 1), (25, -23, 13, -3))
_LINEAR = (0.0401954833730, 0.2493800006710, 0.4802686256260, 0.2009775476730, 0.0291783426580)


def _dot(c, s):
    out = None
    for a, v in zip(c, s):
        if a:
            out = a * v if out is None else out + a * v
    return out


def _weno(s):
    """Face value between s[3] and s[4] from the window s[0..7]."""
    S, q = [], []
    for k in range(5):
        p = s[k:k + 4]
        S.append(720.0 * _dot(_FIRST[k], p) ** 2 + 780.0 * _dot(_SECOND[k], p) ** 2 + 781.0 * _dot(_THIRD, p) ** 2)
        q.append(_dot(_VALUE[k], p) / 12.0)
    for k in range(4):
        S[4] = torch.maximum(S[4], S[k])
    w = [_LINEAR[k] / (2.592e-6 + S[k]) for k in range(5)]
    return sum(w[k] * q[k] for k in range(5)) / sum(w)


def _ghosted(a, dim, closed=False):
    """a with LAP ghost layers along dim: periodic images, or beside a domain face its value repeated."""
    n = a.shape[dim]
    if closed:
        lo, hi = (a.narrow(dim, i, 1).expand([LAP if q == dim else v for q, v in enumerate(a.shape)]) for i in (0, n - 1))
    else:
        lo, hi = a.narrow(dim, n - LAP, LAP), a.narrow(dim, 0, LAP)
    return torch.cat([lo, a, hi], dim)


def _split(d, u, v, w, c, A):
    """Steger-Warming fluxes f+, f- of five components along the metric row A."""
    norm = torch.sqrt(A[0] * A[0] + A[1] * A[1] + A[2] * A[2])
    k = [a / norm for a in A]
    V = A[0] * u + A[1] * v + A[2] * w
    E = (V, V - c * norm, V + c * norm)
    plus = [0.5 * (e + torch.sqrt(e * e + EPSL * EPSL)) for e in E]
    t = d / (2.0 * GAMMA)
    lo = (u - c * k[0], v - c * k[1], w - c * k[2])
    hi = (u + c * k[0], v + c * k[1], w + c * k[2])
    lo2, hi2 = (0.5 * sum(x * x for x in p) for p in (lo, hi))
    q2 = (GAMMA - 1.0) * (u * u + v * v + w * w)
    W2 = (3.0 - GAMMA) / (2.0 * (GAMMA - 1.0)) * c * c

    def flux(e):
        a = 2.0 * (GAMMA - 1.0) * e[0]
        return [t * (a + e[1] + e[2])] + [t * (a * x + e[1] * l + e[2] * h) for x, l, h in zip((u, v, w), lo, hi)] + \
               [t * (e[0] * q2 + e[1] * lo2 + e[2] * hi2 + W2 * (e[1] + e[2]))]
    return flux(plus), flux([e - p for e, p in zip(E, plus)])


def _closed_faces(cells, faces):
    """The one-sided forms of an upwind-from-the-left flux on the faces next to both domain faces.
    cells: the n values along the last axis; faces (n + 1): overwritten there."""
    n = cells.shape[-1]
    c = lambda i: cells[..., i]
    S0 = lambda a, b, d: 13 * (a - 2 * b + d) ** 2 + 3 * (3 * a - 4 * b + d) ** 2
    S1 = lambda a, b, d: 13 * (a - 2 * b + d) ** 2 + 3 * (a - d) ** 2
    S2 = lambda a, b, d: 13 * (a - 2 * b + d) ** 2 + 3 * (a - 4 * b + 3 * d) ** 2
    q0 = lambda a, b, d: 2 * a + 5 * b - d
    q1 = lambda a, b, d: -a + 5 * b + 2 * d
    q2 = lambda a, b, d: 2 * a - 7 * b + 11 * d
    wt = lambda S: 1.0 / (1.2e-5 + S) ** 2

    def mean(pairs):
        return sum(w * q for w, q in pairs) / (6.0 * sum(w for w, _ in pairs))

    def full(f, left):
        s = [c(f - 3 + i) if left else c(f + 2 - i) for i in range(5)]
        A, B, C = S0(*s[2:5]), S1(*s[1:4]), S2(*s[0:3])
        if left:
            # the left form's first two products take indicators that are still zero
            e = 1.2e-5
            w = (e ** 4 * torch.ones_like(A), (e + A) ** 2 * e ** 2, (e + A) ** 2 * (e + B) ** 2)
        else:
            w = (wt(A), wt(B), wt(C))
        return mean(list(zip(w, (q0(*s[2:5]), q1(*s[1:4]), q2(*s[0:3])))))

    def left_form():
        faces[..., 0] = c(0)
        faces[..., 1] = q0(c(0), c(1), c(2)) / 6.0
        a, b = (c(1), c(2), c(3)), (c(0), c(1), c(2))
        faces[..., 2] = mean([(wt(S0(*a)), q0(*a)), (wt(S1(*b)), q1(*b))])
        faces[..., 3] = full(3, True)
        faces[..., n - 2] = full(n - 2, True)
        a, b = (c(n - 3), c(n - 2), c(n - 1)), (c(n - 4), c(n - 3), c(n - 2))
        faces[..., n - 1] = mean([(wt(S1(*a)), q1(*a)), (wt(S2(*b)), q2(*b))])
        faces[..., n] = 1.5 * c(n - 1) - 0.5 * c(n - 2)
        return faces

    def right_form():
        faces[..., 0] = q2(c(2), c(1), c(0)) / 6.0
        a, b = (c(2), c(1), c(0)), (c(3), c(2), c(1))
        faces[..., 1] = mean([(wt(S1(*a)), q1(*a)), (wt(S2(*b)), q2(*b))])
        for f in (2, 3):
            faces[..., f] = full(f, False)
        faces[..., n - 3] = full(n - 3, False)
        a, b = (c(n - 2), c(n - 3), c(n - 4)), (c(n - 1), c(n - 2), c(n - 3))
        faces[..., n - 2] = mean([(wt(S0(*a)), q0(*a)), (wt(S1(*b)), q1(*b))])
        faces[..., n - 1] = 0.5 * (c(n - 1) + c(n - 2))
        faces[..., n] = c(n - 1)
        return faces
    return left_form, right_form


def _rhs(prims, c, h, A, jac, closed):
    """Inviscid RHS (5, nz, ny, nx); A: the nine metric terms, jac: the Jacobian factor."""
    shape = prims[0].shape
    du = torch.zeros((5,) + tuple(shape), device=prims[0].device, dtype=torch.float64)
    for d in range(3):
        dim = 2 - d
        n = shape[dim]
        plus, minus = _split(*prims, c, A[3 * d:3 * d + 3])
        for m in range(5):
            P, M = (_ghosted(x[m], dim, closed and d == 0) for x in (plus, minus))
            fp = _weno([P.narrow(dim, j, n + 1) for j in range(8)])
            fm = _weno([M.narrow(dim, 7 - j, n + 1) for j in range(8)])
            if closed and d == 0:
                fp = _closed_faces(plus[m], fp)[0]()
                fm = _closed_faces(minus[m], fm)[1]()
            face = fp + fm
            du[m] -= jac * (face.narrow(dim, 1, n) - face.narrow(dim, 0, n)) / h[d]
    return du


_CENTRAL = {6: (45.0 / 60.0, -9.0 / 60.0, 1.0 / 60.0), 8: (672.0 / 840.0, -168.0 / 840.0, 32.0 / 840.0, -3.0 / 840.0)}


def _deriv(a, dim, h, order, closed):
    out = torch.zeros_like(a)
    for q, w in enumerate(_CENTRAL[order], start=1):
        out += w * (torch.roll(a, -q, dim) - torch.roll(a, q, dim))
    if closed and dim == 2:
        n = a.shape[2]
        s = lambda i: a[..., i]
        four = lambda i: (s(i - 2) - 8.0 * s(i - 1) + 8.0 * s(i + 1) - s(i + 2)) / 12.0
        six = lambda i: (s(i + 3) - s(i - 3) - 9.0 * (s(i + 2) - s(i - 2)) + 45.0 * (s(i + 1) - s(i - 1))) / 60.0
        forms = {0: s(1) - s(0), 1: 0.5 * (s(2) - s(0)), 2: four(2), 3: six(3), n - 1: s(n - 1) - s(n - 2),
                 n - 2: 0.5 * (s(n - 1) - s(n - 3)), n - 3: four(n - 3), n - 4: six(n - 4)}
        for i, v in forms.items():
            out[..., i] = v
    return out / h


def _viscous(prims, T, h, A, jac, order, closed):
    _, u, v, w = prims
    vel = (u, v, w)
    tsb = 110.4 / REF_T
    mu = (1.0 + tsb) / RE * torch.sqrt(T * T * T) / (tsb + T)
    heat = mu / (GAMMA - 1.0) / PR
    comp = [[_deriv(f, 2 - d, h[d], order, closed) for d in range(3)] for f in vel + (T,)]
    grad = [[sum(A[3 * d + j] * g[d] for d in range(3)) for j in range(3)] for g in comp]
    div = grad[0][0] + grad[1][1] + grad[2][2]
    tau = [[mu * (grad[i][j] + grad[j][i] - (2.0 / 3.0 * div if i == j else 0.0)) for j in range(3)] for i in range(3)]
    en = [sum(vel[i] * tau[i][j] for i in range(3)) + heat * grad[3][j] for j in range(3)]
    out = torch.zeros((5,) + tuple(u.shape), device=u.device, dtype=torch.float64)
    for d in range(3):
        a = [A[3 * d + j] * jac for j in range(3)]
        for m, row in enumerate(tau + [en]):
            out[m + 1] += jac * _deriv(sum(a[j] * row[j] for j in range(3)), 2 - d, h[d], order, closed)
    return out


def _evaluate(case, n, prims, T, A, jac):
    c = torch.sqrt(T)
    du = _rhs(prims, c, _spacing(n), A, jac, case.get("closed", False))
    if case.get("viscous"):
        du += _viscous(prims, T, _spacing(n), A, jac, case["viscous"], case.get("closed", False))
    return du


def _cartesian():
    one, zero = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in (1.0, 0.0))
    return [one if m % 4 == 0 else zero for m in range(9)], one


def _primitives(f):
    rho = f[0]
    u, v, w = (f[m] / rho for m in (1, 2, 3))
    e = f[4] - 0.5 * rho * (u * u + v * v + w * w)
    return (rho, u, v, w), e * GAMMA * (GAMMA - 1.0) / rho, e / rho * (GAMMA - 1.0)


def _conserved(prims, T):
    rho, u, v, w = prims
    return torch.stack([rho, rho * u, rho * v, rho * w,
                        rho * (0.5 * (u * u + v * v + w * w) + T / (GAMMA * (GAMMA - 1.0)))])


def _speed(prims, T):
    c = torch.sqrt(T)
    return max(float((torch.abs(x) + c).max()) for x in prims[1:])


def _advance(case, extents, f):
    """RK3 steps of every block with the smallest of the blocks' CFL steps."""
    A, jac = _cartesian()
    for _ in range(case["steps"]):
        now = [_primitives(x) for x in f]
        dt = min(CFL * min(_spacing(n)) / _speed(p, T) for n, (p, T, _) in zip(extents, now))
        for i, n in enumerate(extents):
            start, x = f[i], f[i]
            for a, b in ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)):
                p, T, _ = _primitives(x)
                x = a * start + b * (x + dt * _evaluate(case, n, p, T, A, jac))
            f[i] = x
    return f


def exact(case, seed):
    extents = _extents(case)
    if case["kind"] == "batch":
        flows = [_flow("blobs", n, 1000 * seed + i) for i, n in enumerate(extents)]
        if case.get("steps"):
            f = _advance(case, extents, [_conserved(p[:4], p[4]) for p in flows])
            return {"f": f, "T": [_primitives(x)[1] for x in f]}
        A, jac = _cartesian()
        return {"du": [_evaluate(case, n, p[:4], p[4], A, jac) for n, p in zip(extents, flows)]}
    n = extents[0]
    flow = _flow(case["flow"], n, seed)
    prims, T = flow[:4], flow[4]
    if case["kind"] == "monitor":
        speed, h = _speed(prims, T), min(_spacing(n))
        return {"dt": torch.tensor([CFL * h / speed], dtype=torch.float64), "cfl": MONITOR_DT * speed / h,
                "fatal": None, "counts": [None] * 4}
    if case["kind"] == "rk3":
        f = _advance(case, extents, [_conserved(prims, T)])[0]
        (d, u, v, w), T, P = _primitives(f)
        return {"f": f, "d": d, "u": u, "v": v, "w": w, "T": T, "P": P}
    if case.get("metrics"):
        fields = [t[LAP:-LAP, LAP:-LAP, LAP:-LAP] for t in _metric_fields(n, seed)]
        A, jac = fields[:9], fields[9]
    else:
        A, jac = _cartesian()
    return {"du": _evaluate(case, n, prims, T, A, jac), "cc": torch.sqrt(T)}
