"""Accuracy of the FP64 paths where a norm over the whole box cannot see it."""
import numpy as np
import pytest

import windstencil_amd as W
from tests.gpu_util import gpu_du_comput, log, make_ctx, oracle_du, upload_state

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _planar_jump(axis, ratio, n=48, across=8, seed=3):
    """rho, u, v, w, T varying along `axis` only: cells 0 .. n/2-1 near (1, 0.3 along the
    axis, 0.1 across, 1) with 1 % noise, the others with `ratio` times the density."""
    rng = np.random.default_rng(seed)
    line = [1.0 + 0.01 * rng.uniform(-1, 1, n) for _ in range(5)]
    rho, T = line[0] * np.where(np.arange(n) < n // 2, 1.0, ratio), line[4]
    vel = [0.1 * line[1 + d] for d in range(3)]
    vel[axis] = 0.3 * line[1 + axis]
    shape = [across] * 3
    shape[2 - axis] = n
    ix = [None] * 3
    ix[2 - axis] = slice(None)
    return [np.ascontiguousarray(np.broadcast_to(a[tuple(ix)], shape)) for a in (rho, *vel, T)]


@pytest.mark.parametrize("ratio", [1e2, 1e4, 1e8])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_quiet_side_of_a_jump_keeps_its_own_accuracy(orc, ws, axis, ratio):
    """Beside a jump, the cells of the quiet side (from one cell off the jump on, where both
    faces take quiet-side values) agree with the oracle to rounding of the quiet side's own
    fluxes, whatever the jump: per component within 64 eps of its flux scale over h (two
    faces of two halves on either side of the comparison, each a few roundings of the split
    and one of the reconstruction).  Every tile shape and the one-launch kernel (None)."""
    prims = _planar_jump(axis, ratio)
    nz, ny, nx = prims[0].shape
    n = (nx, ny, nz)[axis]
    ref = oracle_du(orc, prims)
    h = 1.0 / (n - 1.0)
    wave = 0.5 + 1.0                       # largest |u| + c of the quiet side, c = sqrt(T)/Ma
    scale = np.array([wave, wave ** 2, wave ** 2, wave ** 2, 3.0 * wave ** 3]) * 1.01 / h
    quiet = [slice(None)] * 4
    quiet[3 - axis] = slice(1, n // 2 - 1)
    for tile in [None, *W.TILE_SHAPES]:
        ctx = make_ctx(nx, ny, nz)
        if tile is not None:
            ctx.set_tile_shape(tile)
        du = gpu_du_comput(ctx, upload_state(prims))
        err = np.abs(du - ref)[tuple(quiet)].max(axis=(1, 2, 3)) / scale
        log(f"  axis {axis} ratio {ratio:g} tile {tile}: {err / EPS} eps")
        assert (err <= 64 * EPS).all()


VIS = dict(re=500.0, pr=0.72, ref_t=288.15)
SHEARED = (1.0, 0.2, -0.1, 0.15, 0.9, 0.05, -0.05, 0.12, 1.1, 0.8)


def _device(a):
    """A ghosted device tensor holding the interior array `a` (ghost layers zero)."""
    import torch
    nz, ny, nx = a.shape
    t = W.ghosted_tensor(nx, ny, nz, 0)
    t[4:-4, 4:-4, 4:4 + nx] = torch.from_numpy(np.ascontiguousarray(a))
    return t


def _viscous(prims, order, metrics=None, **kw):
    """ws_viscous_rhs alone into a zero du (numpy, interior); metrics: ten interior arrays."""
    import ctypes

    import torch
    nz, ny, nx = prims[0].shape
    ctx = make_ctx(nx, ny, nz, viscous=order, **VIS, **kw)
    terms = [_device(a) for a in (*prims[1:], *(metrics or ()))]
    f = [W.field_of(t) for t in terms]
    fl = (W.WsField * len(f))(*f)
    W.check(W.lib().ws_ghost_fill_periodic(ctx.handle, fl, len(f), W.stream_handle()))
    mf = None
    if metrics:
        mf = W.WsMetricFields()
        for q in range(9):
            mf.A[q] = f[4 + q]
        mf.ajac = f[13]
    du = W.soa_tensor(nx, ny, nz)
    W.check(W.lib().ws_viscous_rhs(ctx.handle, *f[:4], ctypes.byref(mf) if mf else None, W.soa_of(du),
                                   W.stream_handle()))
    torch.cuda.synchronize()
    return du.cpu().numpy()


@pytest.mark.parametrize("mode", ["cartesian", "sheared", "fields"])
@pytest.mark.parametrize("closed", [False, True])
@pytest.mark.parametrize("order", [6, 8])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_constant_stress_exerts_no_force(ws, axis, order, closed, mode):
    """A velocity across `axis` that changes by the same power of two from cell to cell, at
    constant T: every difference is exact, so the stress is the same number at each cell and its
    derivative, a sum of differences, exactly zero; along z as along x and y."""
    n, across, step = 64, 12, 2.0 ** -4
    i = np.arange(n)
    line = step * (i if closed else np.minimum(i, n - i))
    cells = slice(12, 52) if closed else slice(10, 23)    # 2 R cells off the faces and the kinks
    shape = [across] * 3
    shape[2 - axis] = n
    ix = [None] * 3
    ix[2 - axis] = slice(None)
    prims = [np.ones(shape)] + [np.zeros(shape) for _ in range(3)] + [np.ones(shape)]
    prims[1 + (axis + 1) % 3] = np.broadcast_to(line[tuple(ix)], shape)
    kw = dict(hx=1 / 32, hy=1 / 32, hz=1 / 32, periodic=[1 - int(closed and d == axis) for d in range(3)],
              d0_bound=[int(closed and q // 2 == axis) for q in range(6)])
    metrics = None
    if mode == "sheared":
        kw["metric"] = SHEARED
    if mode == "fields":
        metrics = [np.full(shape, a) for a in SHEARED]
    du = _viscous(prims, order, metrics, **kw)
    at = [slice(None)] * 4
    at[3 - axis] = cells
    assert np.abs(du[4]).max() > 0          # the work term does vary
    assert not du[tuple(at)][1:4].any()


@pytest.mark.parametrize("order", [6, 8])
@pytest.mark.parametrize("fields", [False, True])
def test_viscous_terms_do_not_depend_on_the_chunks(ws, order, fields):
    """A flow of four equal periods along z, and one of them alone: the march starts its chunks
    at other planes, and the terms keep their bits."""
    from tests.helpers import random_state
    nx, ny, nz, reps = 53, 25, 40, 4
    prims = random_state(nx, ny, nz, 19, "rough")
    metrics = None
    if fields:
        from tests.test_gpu_rhs import _wavy_metrics
        metrics = list(_wavy_metrics(nx, ny, nz))
    h = dict(hx=0.02, hy=0.03, hz=0.025)
    one = _viscous(prims, order, metrics, **h)
    rep = lambda arrays: [np.concatenate([a] * reps) for a in arrays]
    four = _viscous(rep(prims), order, rep(metrics) if metrics else None, **h)
    for k in range(reps):
        assert np.array_equal(four[:, k * nz:(k + 1) * nz], one), k


@pytest.mark.parametrize("fields", [False, True])
def test_viscous_terms_of_a_cell_without_temperature(ws, fields):
    """T = 0 has no viscosity (Sutherland's law gives 0): the terms stay finite and agree with
    the anchor kernels."""
    from tests.helpers import random_state, rel_l2
    nx, ny, nz = 30, 20, 16
    prims = [a.copy() for a in random_state(nx, ny, nz, 4, "vortex")]
    prims[4][7, 9, 11] = 0.0
    metrics = None
    if fields:
        from tests.test_gpu_rhs import _wavy_metrics
        metrics = list(_wavy_metrics(nx, ny, nz))
    ref = _viscous(prims, 6, metrics, kernel=W.WS_KERNEL_ANCHOR)
    du = _viscous(prims, 6, metrics)
    assert np.isfinite(ref).all() and np.isfinite(du).all()
    assert rel_l2(du, ref) <= 1e-13


@pytest.mark.parametrize("flow", [(0.0, 0.0, 0.0), (0.4, 0.0, 0.0)])
@pytest.mark.parametrize("precision,tol", [(W.WS_PREC_FP64, 1e-12), (W.WS_PREC_MIXED, 1e-6)])
def test_no_smoothing_of_eigenvalues_at_rest(orc, ws, flow, precision, tol):
    """epsl_sw = 0 is accepted: gas at rest, and directions without flow, have eigenvalues of
    exactly zero, of which the split takes |0| = 0 (tiles and one-launch kernel, as the oracle)."""
    from tests.helpers import rel_l2
    rng = np.random.default_rng(11)
    nx, ny, nz = 31, 17, 19
    a = lambda: 1.0 + 0.2 * rng.random((nz, ny, nx))
    prims = [a(), *(np.full((nz, ny, nx), q) for q in flow), a()]
    ref = oracle_du(orc, prims, eps=0.0)
    for tile in [None, *W.TILE_SHAPES]:
        ctx = make_ctx(nx, ny, nz, precision=precision, epsl_sw=0.0)
        if tile is not None:
            ctx.set_tile_shape(tile)
        err = rel_l2(gpu_du_comput(ctx, upload_state(prims)), ref)
        log(f"  flow {flow} precision {precision} tile {tile}: rel L2 {err:.3e}")
        assert err <= tol
