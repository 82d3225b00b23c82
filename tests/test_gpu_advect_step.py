"""The transport step, its adjoint and the combination with the ghost fill,
each in one launch, against the oracle's separate operations, bit for bit over
the interior, the face ghosts and the three accumulated faces.  Sizes: a row
of one, two and four cells a lane, full and with lanes to spare; one cell;
marches of several planes with a short last one; rows the walk does not take
(odd beyond 64, beyond 256) and a step in place, which go through the
separate calls."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from fields import mac_grids, uniform
from opencurrent_amd import _types as T
from opencurrent_amd import device as D
from opencurrent_amd._types import BC, BCSet, HostGrid

pytestmark = pytest.mark.gpu

SIZES = [(5, 6, 64), (4, 3, 63), (3, 5, 65), (2, 9, 128), (3, 4, 126), (3, 5, 256), (2, 5, 132), (2, 2, 300),
         (1, 1, 1), (2, 1, 2), (130, 128, 6)]
H = (.5, .25, .125)


def faces(kind):
    if kind == "periodic":
        return BCSet.uniform(T.BC_PERIODIC)
    b = BCSet.uniform(T.BC_NEUMANN, 0.5)
    b.xneg, b.xpos = BC(T.BC_DIRICHELET, 1.25, 0.0), BC(T.BC_NEUMANN, -.75, 0.0)
    b.ypos, b.yneg = BC(T.BC_PERIODIC, 0.0, 0.0), BC(T.BC_PERIODIC, 0.0, 0.0)
    b.zpos = BC(T.BC_DIRICHELET, -.5, 0.0) if kind == "walls" else BC(T.BC_NONE, 0.0, 0.0)
    return b


def faces_of(g):
    """interior and face ghosts of a host grid (no edges or corners)"""
    d, a = g.desc, g.full()
    x, y, z = (slice(q, q + n) for q, n in ((d.gx, d.nx), (d.gy, d.ny), (d.gz, d.nz)))
    out = [a[x, y, z]]
    for lo, n, cut in ((d.gx, d.nx, lambda s: (s, y, z)), (d.gy, d.ny, lambda s: (x, s, z)),
                       (d.gz, d.nz, lambda s: (x, y, s))):
        out += [a[cut(slice(lo - 1, lo))], a[cut(slice(lo + n, lo + n + 1))]]
    return out


def same(got, want, what):
    for q, (a, b) in enumerate(zip(faces_of(got), faces_of(want))):
        assert np.array_equal(a, b), f"{what}, part {q}: {np.abs(a - b).max()}"


def state(n, dtype):
    gs = mac_grids(*n, dtype)
    for q, g in enumerate(gs):
        g.buf[:] = (2 * uniform(300 + q, g.buf.shape) - 1).astype(dtype)
    return gs


@pytest.mark.parametrize("kind", ["periodic", "walls", "open"])
@pytest.mark.parametrize("scheme", [T.IT_FIRST_ORDER_UPWIND, T.IT_SECOND_ORDER_CENTERED])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", SIZES)
def test_step_and_adjoint(gpu, n, dtype, scheme, kind):
    bc, dt = faces(kind), .03125
    u, v, w, phi = state(n, dtype)
    dphi, want = HostGrid.congruent(phi), phi.copy()
    O.lib().orc_passive_advect(u.ptr(), v.ptr(), w.ptr(), phi.ptr(), dphi.ptr(), *n, *H, scheme)
    want.interior()[:] = phi.interior() * dtype(1) + dphi.interior() * dtype(dt)
    O.lib().orc_bc_fill(1, want.ptr(), C.byref(bc), *H)
    du, dv, dw, dp = (D.DeviceGrid.from_host(g) for g in (u, v, w, phi))
    dd, dq, dr = D.DeviceGrid.from_host(dphi), D.DeviceGrid.from_host(phi), D.DeviceGrid.from_host(phi)
    D.passive_advect_step(du, dv, dw, dp, dq, dd, dt, *H, scheme, bc)
    same(dq.to_host(), want, "step")
    D.passive_advect_step(du, dv, dw, dr, dr, dd, dt, *H, scheme, bc)
    same(dr.to_host(), want, "step in place")

    lam, out = HostGrid.congruent(phi), HostGrid.congruent(phi)
    lam.interior()[:] = (2 * uniform(310, lam.interior().shape) - 1).astype(dtype)
    adj = mac_grids(*n, dtype)[:3]
    for q, g in enumerate(adj):
        g.buf[:] = (2 * uniform(320 + q, g.buf.shape) - 1).astype(dtype)
    dl, do = D.DeviceGrid.from_host(lam), D.DeviceGrid.from_host(out)
    da = [D.DeviceGrid.from_host(g) for g in adj]
    O.lib().orc_passive_advect_adjoint(u.ptr(), v.ptr(), w.ptr(), phi.ptr(), lam.ptr(), out.ptr(),
                                       *(g.ptr() for g in adj), dt, *n, *H, scheme)
    O.lib().orc_bc_adjoint_nocorners(out.ptr(), C.byref(bc))
    D.passive_advect_adjoint_step(du, dv, dw, dp, dl, do, *da, dt, *H, scheme, bc)
    assert np.array_equal(do.to_host().interior(), out.interior())
    for q, (a, b) in enumerate(zip(da, adj)):
        assert np.array_equal(a.to_host().buf, b.buf), "uvw"[q]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 33), (9, 8, 32), (3, 17, 70)])
def test_combination_with_fill(gpu, n, dtype):
    for kind in ("periodic", "walls", "open"):
        bc = faces(kind)
        a, b = state(n, dtype)[3], state(n, dtype)[3]
        b.buf[:] = b.buf[::-1].copy()
        want = a.copy()
        want.interior()[:] = a.interior() * dtype(1) + b.interior() * dtype(.1)
        O.lib().orc_bc_fill(1, want.ptr(), C.byref(bc), *H)
        r, g2 = D.DeviceGrid.from_host(a), D.DeviceGrid.from_host(b)
        D.grid_lincomb_fill(r, 1.0, r, .1, g2, bc, *H)
        assert np.array_equal(r.to_host().buf, want.buf), kind


def test_step_refuses(gpu):
    """what the separate calls refuse"""
    from opencurrent_amd._lib import OcuError
    u, v, w, phi = (D.DeviceGrid.from_host(g) for g in state((4, 4, 4), np.float32))
    other = D.DeviceGrid.from_host(state((4, 9, 5), np.float32)[3])
    ok, slip = faces("walls"), BCSet.uniform(T.BC_FORCED_INFLOW_VARIABLE_SLIP)
    out, d = D.DeviceGrid.congruent(phi), D.DeviceGrid.congruent(phi)
    for args in ((phi, out, d, .1, *H, T.IT_SECOND_ORDER_UPWIND, ok), (phi, out, d, .1, *H, 1, slip),
                 (phi, other, d, .1, *H, 1, ok)):
        with pytest.raises(OcuError):
            D.passive_advect_step(u, v, w, *args)
    with pytest.raises(OcuError):
        D.passive_advect_adjoint_step(u, v, w, phi, out, out, u, v, w, .1, *H, 1, ok)
    with pytest.raises(OcuError):
        D.grid_lincomb_fill(out, 1.0, phi, .1, other, ok, *H)
