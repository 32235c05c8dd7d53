"""Storage layouts of the tiled family's viscous terms: fields that share a pitch, fields
that do not, and planes beyond 32-bit byte offsets."""
import ctypes

import numpy as np
import pytest

import windstencil_amd as W
from tests.helpers import ghosted, random_state, rel_l2

pytestmark = pytest.mark.gpu

VIS = dict(re=500.0, pr=0.72, ref_t=288.15)


def _fields(prims, pads, pitch=None):
    """u, v, w, T on the device with filled periodic ghosts, field q padded by pads[q]; pitch: of
    T, whose unused columns are never touched."""
    import torch
    nz, ny, nx = prims[0].shape
    out = []
    for q, a in enumerate(prims[1:]):
        t = W.ghosted_tensor(nx, ny, nz, pads[q])
        if pitch and q == 3:
            t = torch.empty((nz + 8, ny + 8, pitch), dtype=torch.float64, device="cuda")
        t[:, :, :nx + 8] = torch.from_numpy(np.pad(a, 4, mode="wrap"))
        out.append(t)
    return out


def _viscous(fields, n, order, metrics=None, **kw):
    import torch
    ctx = W.Context(W.default_config(*n, viscous=order, **VIS, **kw))
    mf = None
    if metrics:
        mf = W.WsMetricFields()
        for q in range(9):
            mf.A[q] = W.field_of(metrics[q])
        mf.ajac = W.field_of(metrics[9])
    du = W.soa_tensor(*n)
    W.check(W.lib().ws_viscous_rhs(ctx.handle, *[W.field_of(t) for t in fields], ctypes.byref(mf) if mf else None,
                                   W.soa_of(du), W.stream_handle()))
    torch.cuda.synchronize()
    return du.cpu().numpy()


@pytest.mark.parametrize("faces", [((1, 1, 1), (0,) * 6), ((0, 1, 1), (1, 1, 0, 0, 0, 0)), ((0, 0, 0), (1,) * 6)])
@pytest.mark.parametrize("order", [6, 8])
@pytest.mark.parametrize("with_metrics", [False, True])
def test_pitches_do_not_change_the_bits(ws, faces, order, with_metrics):
    """One pitch for all fields, T's its own, every field's its own: the same operations on the
    same values."""
    import torch
    from tests.test_gpu_rhs import _wavy_metrics
    n = (53, 25, 31)
    prims = random_state(*n, 19, "vortex")
    kw = dict(periodic=faces[0], d0_bound=faces[1])

    def terms(pad):
        out = []
        for q, a in enumerate(_wavy_metrics(*n)):
            t = W.ghosted_tensor(*n, pad * (q % 3))
            t[:, :, :n[0] + 8] = torch.from_numpy(np.pad(a, 4, mode="wrap"))
            out.append(t)
        return out
    got = []
    for pads in ([0, 0, 0, 0], [0, 0, 0, 3], [1, 2, 0, 7]):
        m = terms(pads[0]) if with_metrics else None
        got.append(_viscous(_fields(prims, pads), n, order, m, **kw))
    assert np.abs(got[0]).max() > 0
    assert np.array_equal(got[1], got[0]) and np.array_equal(got[2], got[0])


@pytest.mark.parametrize("order", [6, 8])
def test_planes_of_four_gigabytes(orc, ws, order):
    """T stored in planes of just over 2^32 bytes (52 GB in all, only its rows' starts written):
    64-bit addresses, within 1e-13 of the oracle as any other layout."""
    import torch
    n = (9, 4, 5)
    pitch = -(-(1 << 29) // (n[1] + 8)) + 1
    if torch.cuda.mem_get_info()[0] < 70 << 30:
        pytest.skip("needs 70 GB of device memory")
    prims = random_state(*n, 5, "rough")
    p = orc.params(*n)
    g = [ghosted(a) for a in prims]
    for a in g:
        orc.ghost_fill_periodic(p, a)
    ref = orc.viscous_rhs(p, g[1], g[2], g[3], g[4], 500.0, 0.72, 288.15, order)
    fields = _fields(prims, [0, 0, 0, 0], pitch)
    err = rel_l2(_viscous(fields, n, order), ref)
    del fields
    torch.cuda.empty_cache()
    assert err <= 1e-13
