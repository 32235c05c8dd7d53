"""The memory-bound kernels around the RHS at the edges of their index arithmetic."""
import ctypes

import numpy as np
import pytest

import windstencil_amd as W
from tests.gpu_util import make_ctx, upload_state
from tests.helpers import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [W.WS_PREC_FP64, W.WS_PREC_MIXED])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 1, 1), (1, 0, 0), (0, 0, 0)])
@pytest.mark.parametrize("shape", [(4, 4, 4), (9, 6, 5), (70, 65, 66)])
def test_rhs_inputs_in_one_launch(ws, shape, periodic, precision):
    """The RHS's inputs, prepared alone (one point per thread up to 2^18 ghosted points, two
    above) and by a small grid's du_comput in the launch that computes the RHS, against a
    ghost fill, a pass over T and the RHS: every point of the ghosted box and du bit for bit, the
    caller's ghost layers and corners included, with a sound speed of another pitch and with
    metric fields."""
    import torch
    nx, ny, nz = shape
    L, sh = W.lib(), W.stream_handle()
    ctx = make_ctx(nx, ny, nz, periodic=periodic, precision=precision)
    rng = np.random.default_rng(41)
    tens = [torch.from_numpy(0.7 + 0.6 * rng.random((nz + 8, ny + 8, nx + 8))).cuda() for _ in range(10)]
    mf = W.WsMetricFields()
    for i in range(9):
        mf.A[i] = W.field_of(tens[i])
    mf.ajac = W.field_of(tens[9])
    states = []
    for _ in range(4):
        st = upload_state(random_state(nx, ny, nz, 3, "blobs"))
        st.t["cc"] = W.ghosted_tensor(nx, ny, nz, pad=3)
        st.refresh()
        gen = torch.Generator(device="cuda").manual_seed(7)
        for k in ("d", "u", "v", "w", "T"):
            inner = st.interior(k).clone()
            st.t[k].copy_(1.0 + 0.2 * torch.rand(st.t[k].shape, dtype=torch.float64, device="cuda", generator=gen))
            st.interior(k).copy_(inner)
        states.append(st)
    a, am, p, b = states
    W.check(L.ws_du_comput(ctx.handle, ctypes.byref(a.ws), None, sh))
    W.check(L.ws_du_comput(ctx.handle, ctypes.byref(am.ws), ctypes.byref(mf), sh))
    W.check(L.ws_prepare_rhs_inputs(ctx.handle, ctypes.byref(p.ws), sh))
    fl = (W.WsField * 5)(b.ws.d, b.ws.u, b.ws.v, b.ws.w, b.ws.T)
    W.check(L.ws_ghost_fill_periodic(ctx.handle, fl, 5, sh))
    W.check(L.ws_sound_speed(ctx.handle, b.ws.T, b.ws.cc, W.job((0, 0, 0), (nx + 8, ny + 8, nz + 8)), sh))
    for k in ("d", "u", "v", "w", "T", "cc"):
        for st in (a, am, p):
            assert torch.equal(st.t[k][..., :nx + 8], b.t[k][..., :nx + 8]), k
    job = W.interior_job(nx, ny, nz)
    for st, m in ((a, None), (am, ctypes.byref(mf))):
        W.check(L.ws_inviscid_rhs(ctx.handle, b.ws.d, b.ws.u, b.ws.v, b.ws.w, b.ws.cc, m, b.ws.du, job, 0, sh))
        assert torch.equal(st.interior("du"), b.interior("du"))


@pytest.mark.parametrize("shape", [(4, 4, 4), (33, 17, 9), (129, 127, 131)])
def test_reductions_over_ragged_boxes(ws, shape):
    """The CFL step and the state analysis take four points per thread and round: the largest
    speed and each bad cell count wherever they lie, the last cell and the ends of a round
    included, and points past the end are not counted twice."""
    import torch
    nx, ny, nz = shape
    L, sh = W.lib(), W.stream_handle()
    ctx = make_ctx(nx, ny, nz)
    dt = torch.zeros(1, dtype=torch.float64, device="cuda")
    hmin = min(ctx.cfg.hx, ctx.cfg.hy, ctx.cfg.hz)
    n = nx * ny * nz
    for at in sorted({0, n - 1, n // 2, min(n - 1, 4 * 1024 * 256), min(n - 1, 1024 * 256 - 1)}):
        st = upload_state(random_state(nx, ny, nz, 3, "blobs"))
        z, y, x = np.unravel_index(at, (nz, ny, nx))
        st.interior("v")[z, y, x] = -50.0
        W.check(L.ws_cfl_dt(ctx.handle, ctypes.byref(st.ws), 0.5, dt.data_ptr(), sh))
        c = np.sqrt(st.interior("T")[z, y, x].item()) / ctx.cfg.ama
        want = 0.5 * hmin / (50.0 + c)
        assert abs(dt.item() - want) <= 4 * np.finfo(float).eps * want
        for k in ("d", "u", "v", "w", "T"):
            full = st.t[k]
            inner = st.interior(k).clone()
            full.fill_(1.0)
            st.interior(k).copy_(inner)
        st.interior("T")[z, y, x] = float("nan")
        st.t["d"][-1, -1, nx + 7] = -1.0      # the last ghosted point
        rep = W.WsAnaReport()
        W.check(L.ws_ana_state(ctx.handle, ctypes.byref(st.ws), None, 0.1, ctypes.byref(rep), sh))
        assert (rep.nan_T, rep.neg_T, rep.neg_d, rep.neg_jac) == (1, 0, 1, 0)
        assert tuple(rep.first_nan_T) == (x, y, z)
        assert tuple(rep.first_neg_d) == (nx + 3, ny + 3, nz + 3)


@pytest.mark.parametrize("viscous", [0, 6])
@pytest.mark.parametrize("steps", [1, 2, 4, 5, 6, 8])
def test_runs_replaying_pairs_of_steps(ws, steps, viscous):
    """ws_rk3_run and ws_batch_rk3_run replay a graph of two steps where there are at least two
    pairs after the first step: any number of steps gives the eager run bit for bit."""
    n = (20, 13, 11)
    L, sh = W.lib(), W.stream_handle()
    got = []
    for graph in (0, 1):
        out = []
        for batch in (False, True):
            st = upload_state(random_state(*n, 3, "blobs"))
            ctx = make_ctx(*n, viscous=viscous)
            W.check(L.ws_pri_to_cons(ctx.handle, st.ws.f, st.ws.d, st.ws.u, st.ws.v, st.ws.w, st.ws.T,
                                     W.job((0, 0, 0), n), sh))
            if batch:
                b = W.Batch(W.default_config(8, 8, 8, viscous=viscous), [n], [st])
                W.check(L.ws_batch_rk3_run(b.handle, steps, 0.5, graph, sh))
                b.sync_states()
            else:
                W.check(L.ws_rk3_run(ctx.handle, ctypes.byref(st.ws), steps, 0.5, graph, sh))
                st.sync_from_ws()
            out += [st.interior(k).cpu().numpy().copy() for k in ("f", "d", "u", "v", "w", "T")]
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_state_analyses_that_overlap(ws):
    """ws_ana_state's fixed records serve one call per GPU at a time and a call that finds them
    taken allocates its own: four threads on streams of their own each get their state's counts."""
    import threading

    import torch
    L = W.lib()
    n = (70, 33, 29)
    bad = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            ctx = make_ctx(*n)
            st = upload_state(random_state(*n, 3 + i, "blobs"))
            st.interior("T")[:i + 1, 0, 0] = float("nan")
            stream.synchronize()
            rep = W.WsAnaReport()
            for _ in range(20):
                W.check(L.ws_ana_state(ctx.handle, ctypes.byref(st.ws), None, 0.1, ctypes.byref(rep), W.stream_handle(stream)))
                if (rep.nan_T, tuple(rep.first_nan_T)) != (i + 1, (0, 0, 0)):
                    bad.append((i, rep.nan_T))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
