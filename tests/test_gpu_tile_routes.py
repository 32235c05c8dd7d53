"""The directional tiles on small grids.  A context without a tile shape runs small jobs in
one launch over cubes; these run them by the tiles, so that the launches which large grids
take (the stage applied by the last direction, its halo, P, sound speed and CFL maxima per
tile) are compared with the separate stage kernel and the oracle."""
import ctypes

import numpy as np
import pytest

import windstencil_amd as W
from tests.gpu_util import gpu_du_comput, log, make_ctx, oracle_du, upload_state
from tests.helpers import random_state, rel_l2
from tests.test_gpu_solver import _gpu_run, _oracle_run

pytestmark = pytest.mark.gpu

TILES = [W.WS_TILE_15x16_K1, W.WS_TILE_30x16_K2, W.WS_TILE_126x2_K2]
PRECISIONS = [W.WS_PREC_FP64, W.WS_PREC_MIXED]
FIELDS = ("d", "u", "v", "w", "T", "P", "cc")


def _same(a, sa, b, sb):
    assert np.isfinite(a).all()
    assert np.array_equal(a, b), rel_l2(a, b)
    for k in FIELDS:
        assert np.array_equal(sa.t[k].cpu().numpy(), sb.t[k].cpu().numpy()), k


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("fusion", [1, 2, 3])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("order", [W.WS_ORDER_XYZ, W.WS_ORDER_ZYX])
def test_tiles_apply_the_stage_as_the_stage_kernel_does(ws, precision, order, fusion, tile):
    """Every fusion level against the separate stage kernel, bit for bit, in either order."""
    prims = random_state(45, 26, 19, 13, "shock")
    run = dict(graph=False, precision=precision, order=order, tile=tile)
    _same(*_gpu_run(prims, 4, W.WS_KERNEL_TILED, fusion=fusion, stage_order=order, **run),
          *_gpu_run(prims, 4, W.WS_KERNEL_TILED, fusion=0, **run))


@pytest.mark.parametrize("nsteps", [1, 2, 3, 5, 6])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("shape", [(37, 24, 18), (64, 32, 32)])
def test_tiles_alternate_the_primitive_sets(ws, precision, graph, nsteps, shape):
    """Fusion 3 by the tiles ends as the plain steps do.  64x32x32: the stage kernel of a plain
    last step has 256 work-groups, the stage-applying launch 160 tiles, and the buffer of the
    maxima holds either."""
    prims = random_state(*shape, 17, "vortex")
    run = dict(graph=graph, precision=precision, tile=W.WS_TILE_30x16_K2)
    _same(*_gpu_run(prims, nsteps, W.WS_KERNEL_TILED, fusion=3, **run),
          *_gpu_run(prims, nsteps, W.WS_KERNEL_TILED, fusion=0, **run))


@pytest.mark.parametrize("fusion", [0, 2, 3])
@pytest.mark.parametrize("precision", PRECISIONS)
def test_tiles_leave_the_cfl_maxima(ws, precision, fusion):
    """A run's dt from the maxima per tile (fusion 3) or stage kernel, against steps driven one
    by one with a pass over the state: same bits."""
    import torch
    prims = random_state(41, 22, 17, 21, "vortex")
    tile = W.WS_TILE_30x16_K2
    a, _ = _gpu_run(prims, 4, W.WS_KERNEL_TILED, graph=True, cfl=0.45, precision=precision, fusion=fusion, tile=tile)
    nz, ny, nx = prims[0].shape
    L = W.lib()
    s = W.stream_handle()
    ctx = make_ctx(nx, ny, nz, precision=precision)
    ctx.set_tile_shape(tile)
    ctx.set_stage_fusion(fusion)
    st = upload_state(prims)
    W.check(L.ws_pri_to_cons(ctx.handle, st.ws.f, st.ws.d, st.ws.u, st.ws.v, st.ws.w, st.ws.T,
                             W.job((0, 0, 0), (nx, ny, nz)), s))
    dt = torch.zeros(1, dtype=torch.float64, device="cuda")
    for _ in range(4):
        W.check(L.ws_cfl_dt(ctx.handle, ctypes.byref(st.ws), 0.45, ctypes.c_void_p(dt.data_ptr()), s))
        W.check(L.ws_rk3_step(ctx.handle, ctypes.byref(st.ws), ctypes.c_void_p(dt.data_ptr()), s))
    st.sync_from_ws()
    torch.cuda.synchronize()
    assert np.array_equal(a, st.interior("f").cpu().numpy())


@pytest.mark.parametrize("precision,tol", [(W.WS_PREC_FP64, 1e-12), (W.WS_PREC_MIXED, 1e-6)])
@pytest.mark.parametrize("kind", ["blobs", "vortex", "shock"])
def test_rk3_by_the_tiles_matches_the_oracle(orc, ws, kind, precision, tol):
    prims = random_state(48, 32, 16, 11, kind)
    f, _ = _gpu_run(prims, 10, W.WS_KERNEL_TILED, graph=False, precision=precision, tile=W.WS_TILE_30x16_K2)
    err = rel_l2(f, _oracle_run(orc, prims, 10))
    log(f"  rk3 by the tiles {kind} precision {precision} x10: rel L2 {err:.3e}")
    assert err <= tol


@pytest.mark.parametrize("tile", W.TILE_SHAPES)
@pytest.mark.parametrize("precision", PRECISIONS)
def test_exact_properties_by_the_tiles(ws, precision, tile):
    """Uniform state -> exactly zero; a padded pitch keeps the bits; a periodic shift shifts
    them; totals conserved to summation rounding."""
    nx, ny, nz = 45, 32, 20
    ctx = make_ctx(nx, ny, nz, precision=precision)
    ctx.set_tile_shape(tile)
    uniform = [np.full((nz, ny, nx), v) for v in (1.1, 0.4, -0.3, 0.2, 1.3)]
    assert not gpu_du_comput(ctx, upload_state(uniform)).any()
    prims = random_state(nx, ny, nz, 5, "shock")
    du = gpu_du_comput(ctx, upload_state(prims))
    assert np.array_equal(gpu_du_comput(ctx, upload_state(prims, pad=7)), du)
    rolled = gpu_du_comput(ctx, upload_state([np.roll(a, (3, 5, 7), axis=(0, 1, 2)) for a in prims]))
    assert np.array_equal(rolled, np.roll(du, (3, 5, 7), axis=(1, 2, 3)))
    for m in range(5):
        assert abs(du[m].sum()) <= 1e-12 * np.abs(du[m]).sum()


@pytest.mark.parametrize("tile", W.TILE_SHAPES)
@pytest.mark.parametrize("precision,tol", [(W.WS_PREC_FP64, 1e-12), (W.WS_PREC_MIXED, 1e-6)])
def test_metric_fields_by_the_tiles(orc, ws, tile, precision, tol):
    """Curvilinear metric terms and Jacobian per cell, every tile shape."""
    import torch
    from tests.helpers import ghosted
    from tests.test_gpu_rhs import _wavy_metrics
    nx, ny, nz = 37, 21, 34
    prims = random_state(nx, ny, nz, 8, "blobs")
    g = [ghosted(a) for a in _wavy_metrics(nx, ny, nz)]
    p = orc.params(nx, ny, nz)
    for a in g:
        orc.ghost_fill_periodic(p, a)
    ref = oracle_du(orc, prims, metrics=g[:9], ajac=g[9])
    terms = [torch.from_numpy(a).cuda() for a in g]
    mf = W.WsMetricFields()
    for q in range(9):
        mf.A[q] = W.field_of(terms[q])
    mf.ajac = W.field_of(terms[9])
    ctx = make_ctx(nx, ny, nz, precision=precision)
    ctx.set_tile_shape(tile)
    err = rel_l2(gpu_du_comput(ctx, upload_state(prims), metrics=mf), ref)
    log(f"  metric fields tile {tile} precision {precision}: rel L2 {err:.3e}")
    assert err <= tol


@pytest.mark.parametrize("tile", W.TILE_SHAPES)
@pytest.mark.parametrize("order", W.ORDERS)
@pytest.mark.parametrize("precision", PRECISIONS)
def test_sub_box_and_accumulation_by_the_tiles(ws, precision, order, tile):
    """A job box updates exactly its cells, with a full run's values; accumulate adds."""
    nx, ny, nz = 40, 24, 20
    prims = random_state(nx, ny, nz, 3, "shock")
    ctx = make_ctx(nx, ny, nz, precision=precision)
    ctx.set_tile_shape(tile)
    ctx.set_direction_order(order)
    full = gpu_du_comput(ctx, upload_state(prims))
    st = upload_state(prims)
    st.t["du"].fill_(7.0)
    part = gpu_du_comput(ctx, st, job=W.job((4 + 5, 4 + 3, 4 + 2), (4 + 33, 4 + 21, 4 + 17)))
    inside = np.zeros(part.shape, dtype=bool)
    inside[:, 2:17, 3:21, 5:33] = True
    assert np.array_equal(part[inside], full[inside])
    assert (part[~inside] == 7.0).all()
    st = upload_state(prims)
    st.t["du"].fill_(2.0)
    acc = gpu_du_comput(ctx, st, accumulate=True)
    assert np.abs(acc - 2.0 - full).max() <= 1e-12 * np.abs(full).max()
