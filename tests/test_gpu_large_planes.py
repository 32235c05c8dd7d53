"""Boxes whose planes or rows are beyond the tiles' 32-bit offsets (13.1 million points): the
tile shape, schedule, stage order and stage fusion that the caller chose apply there as
elsewhere, with the bits of the same box in short rows."""
import ctypes

import numpy as np
import pytest

import windstencil_amd as W
from tests.gpu_util import log, make_ctx, upload_state
from tests.helpers import random_state

pytestmark = pytest.mark.gpu

LIMIT = (1 << 29) // 41
N = (9, 5, 6)
KEYS = ("f", "du", "d", "u", "v", "w", "T", "P", "cc")


def _roomy(gib):
    import torch
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < gib << 30:
        pytest.skip(f"needs {gib} GiB of device memory")


def _load(st, prims):
    """prims into a state used before: ghost layers zero, f from them."""
    for k in ("d", "u", "v", "w", "T", "P", "cc"):
        st.t[k][:, :, :N[0] + 8].zero_()
    st.set_prims(*prims)
    ctx = make_ctx(*N)
    W.check(W.lib().ws_pri_to_cons(ctx.handle, st.ws.f, st.ws.d, st.ws.u, st.ws.v, st.ws.w, st.ws.T,
                                   W.job((0, 0, 0), N), W.stream_handle()))


def _out(st):
    import torch
    st.sync_from_ws()
    torch.cuda.synchronize()
    return {k: (st.t[k][..., :N[0]] if k in ("f", "du") else st.t[k][..., :N[0] + 8]).cpu().numpy() for k in KEYS}


def _runs(st, prims, precision, tiles):
    """RHS in every tile shape and schedule, RK3 runs in every shape and stage order."""
    L = W.lib()
    s = W.stream_handle()
    for tile in tiles:
        for sched in W.SCHEDULES:
            _load(st, prims)
            ctx = make_ctx(*N, precision=precision)
            ctx.set_tile_shape(tile)
            ctx.set_schedule(sched)
            W.check(L.ws_du_comput(ctx.handle, ctypes.byref(st.ws), None, s))
            yield ("rhs", tile, sched), _out(st)
        for order in W.ORDERS:
            for fusion in (1, 2, 3):
                _load(st, prims)
                ctx = make_ctx(*N, precision=precision)
                ctx.set_tile_shape(tile)
                ctx.set_stage_order(order)
                ctx.set_stage_fusion(fusion)
                W.check(L.ws_rk3_run(ctx.handle, ctypes.byref(st.ws), 2, 0.5, 0, s))
                yield ("rk3", tile, order, fusion), _out(st)


@pytest.mark.parametrize("precision", [W.WS_PREC_FP64, W.WS_PREC_MIXED])
def test_large_planes_keep_the_callers_choices(ws, precision):
    """du tells the routes apart: a fused stage leaves partial sums there, the separate stage
    kernel the complete RHS."""
    _roomy(24)
    prims = random_state(*N, 29, "blobs")
    short, long_ = upload_state(prims), upload_state(prims, pad=1_100_000)
    assert short.ws.d.pitch * (N[1] + 8) < LIMIT <= long_.ws.d.pitch * (N[1] + 8) and long_.ws.d.pitch < LIMIT
    for (what, a), (_, b) in zip(_runs(short, prims, precision, W.TILE_SHAPES),
                                 _runs(long_, prims, precision, W.TILE_SHAPES)):
        for k in KEYS:
            assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k]), (what, k)


@pytest.mark.parametrize("precision", [W.WS_PREC_FP64, W.WS_PREC_MIXED])
def test_rows_beyond_32_bit_offsets(ws, precision):
    """One field (T) with rows of 13.2 million points: one tile shape serves them, in every
    schedule, stage order and fusion level."""
    import torch
    _roomy(24)
    prims = random_state(*N, 29, "blobs")
    short, long_ = upload_state(prims), upload_state(prims)
    long_.t["T"] = torch.empty((N[2] + 8, N[1] + 8, LIMIT + 100_000), dtype=torch.float64, device="cuda")
    long_.refresh()
    tiles = [W.WS_TILE_30x16_K2]
    for (what, a), (_, b) in zip(_runs(short, prims, precision, tiles), _runs(long_, prims, precision, tiles)):
        for k in KEYS:
            assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k]), (what, k)


@pytest.mark.parametrize("precision", [W.WS_PREC_FP64, W.WS_PREC_MIXED])
def test_batch_with_a_block_of_large_planes(ws, precision):
    """A batch with one such block, against the same batch in short rows: shape, schedule and
    fused steps, bit for bit."""
    import torch
    _roomy(24)
    L = W.lib()
    s = W.stream_handle()
    prims = [random_state(*N, 31 + i, "blobs") for i in range(2)]
    base = W.default_config(8, 8, 8, precision=precision)
    got = []
    for pad in (0, 1_100_000):
        out = []
        sts = [upload_state(prims[0], pad=pad), upload_state(prims[1])]
        for tile, sched in ((W.WS_TILE_126x2_K2, W.WS_SCHED_PREFETCH), (W.WS_TILE_15x16_K1, W.WS_SCHED_GRID)):
            for p, st in zip(prims, sts):
                _load(st, p)
            b = W.Batch(base, [N, N], sts)
            W.check(L.ws_batch_set_tile_shape(b.handle, tile))
            W.check(L.ws_batch_set_schedule(b.handle, sched))
            W.check(L.ws_batch_du_comput(b.handle, s))
            torch.cuda.synchronize()
            out += [st.interior("du").cpu().numpy() for st in sts]
            W.check(L.ws_batch_rk3_run(b.handle, 2, 0.5, 0, s))
            b.sync_states()
            out += [_out(st) for st in sts]
            b.close()
        got.append(out)
        log(f"  batch precision {precision} pad {pad} done")
    for a, b in zip(*got):
        if isinstance(a, dict):
            for k in KEYS:
                assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k]), k
        else:
            assert np.array_equal(a, b)
