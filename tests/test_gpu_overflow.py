"""FP64 relaxations whose update overflows: the diagonal (below one here, as
the solvers' factors never make it) turns a large residual into infinity, and
what follows from it is infinite or NaN where the oracle's divisions say so.
Every kernel that divides by the diagonal's reciprocal, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from fields import uniform
from opencurrent_amd import _lib
from opencurrent_amd import _types as T
from opencurrent_amd import device as D
from opencurrent_amd._types import BCSet, HostGrid, MGLevelParams

pytestmark = pytest.mark.gpu

BC_ = BCSet.uniform(T.BC_NEUMANN)
H = (1.0, 1.0, 1.0)


def params():
    p = MGLevelParams()
    p.h, p.omega = 1.0, 1.0
    p.fx = p.fy = p.fz = .05
    for f in range(6):
        p.mods[f] = -.05
    return p


def grids(n):
    u, b = HostGrid(*n), HostGrid(*n)
    u.interior()[:] = 2 * uniform(800, n) - 1
    b.interior()[:] = 2 * uniform(801, n) - 1
    at = tuple(x // 2 for x in n)
    # the update of this cell overflows, those beside it get the infinity
    b.interior()[at] = -1.5e308
    O.lib().orc_bc_fill(0, u.ptr(), C.byref(BC_), *H)
    return u, b, at


def sweep(u, b, p, times, variant):
    for _ in range(times):
        for color in (0, 1):
            O.lib().orc_mg_relax(u.ptr(), b.ptr(), color, C.byref(p), variant)
            O.lib().orc_bc_fill(0, u.ptr(), C.byref(BC_), *H)


def same(got, want, at, what):
    a, b = got.interior(), want.interior()
    assert np.isinf(b).any(), "the oracle's update does not overflow"
    assert np.array_equal(a, b, equal_nan=True), f"{what}: {a[at]} for {b[at]}"


@pytest.mark.parametrize("zero", [False, True])
@pytest.mark.parametrize("n", [(6, 6, 64), (6, 6, 128), (4, 6, 256), (5, 6, 70)])
def test_fused_sweep(gpu, n, zero):
    p, (u, b, at) = params(), grids(n)
    if zero:
        u.buf[:] = 0
    want = u.copy()
    sweep(want, b, p, 1, T.RELAX_DEVICE)
    gu, gb = D.DeviceGrid.from_host(u), D.DeviceGrid.from_host(b)
    out = D.DeviceGrid.congruent(gu)
    _lib.check(_lib.hip().ocu_mg_relax_fused_bc(gu.ptr(), out.ptr(), gb.ptr(), C.byref(p), C.byref(BC_), *H, 0,
                                                int(zero) * T.FUSED_ZERO_INPUT, None), "sweep")
    same(out.to_host(), want, at, f"rows of {n[2]}")


def test_tiles(gpu):
    p, (u, b, at) = params(), grids((16, 8, 8))
    want = u.copy()
    sweep(want, b, p, 2, T.RELAX_DEVICE)
    gu, gb = D.DeviceGrid.from_host(u), D.DeviceGrid.from_host(b)
    out = D.DeviceGrid.congruent(gu)
    _lib.check(_lib.hip().ocu_mg_smooth2(gu.ptr(), out.ptr(), gb.ptr(), None, None, C.byref(p), C.byref(BC_), 0, None,
                                         None), "tiles")
    same(out.to_host(), want, at, "tiles")


def test_bottom_blocks(gpu):
    """one iteration of the top level (nu1) and nothing after it but the
    prolongation of the zero coarse level's relaxation"""
    p, (u, b, at) = params(), grids((8, 8, 8))
    us, bs = [u, HostGrid(4, 4, 4)], [b, HostGrid(4, 4, 4)]
    dev = [[D.DeviceGrid.from_host(x) for x in v] for v in (us, bs)]
    _lib.check(_lib.hip().ocu_mg_bottom_vcycle_filled(
        *((T.Grid3DDesc * 2)(*[x.desc for x in v]) for v in dev), (MGLevelParams * 2)(p, p), (C.c_double * 6)(*[1.0] * 6),
        2, C.byref(BC_), 1, 0, 0, 0, 0, None), "bottom")
    want = u.copy()
    sweep(want, b, p, 1, T.RELAX_DEVICE)
    same(dev[0][0].to_host(), want, at, "blocks")


def test_coarsest_pairs(gpu):
    p, (u, b, at) = params(), grids((4, 6, 5))
    want = u.copy()
    sweep(want, b, p, 2, T.RELAX_HOST)
    gu, gb = D.DeviceGrid.from_host(u), D.DeviceGrid.from_host(b)
    _lib.check(_lib.hip().ocu_mg_coarse_relax_filled(gu.ptr(), gb.ptr(), 2, 0, C.byref(p), C.byref(BC_), *H, 0, None),
               "pairs")
    same(gu.to_host(), want, at, "pairs")
