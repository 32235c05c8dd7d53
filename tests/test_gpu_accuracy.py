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
