"""Two relaxation iterations in one launch by tiles (ocu_mg_smooth2) against
the oracle's separate operations, bit for bit over the interior and the whole
ghost layer: with and without the zero start, the pending prolongation and
the residual + restriction.  Sizes: two blocks per axis, one tile, partial
tiles at the end of every axis, the smallest periodic side, several tiles.
The norms are sums of the same squares in another order: n terms in double,
so n * 2^-53 relative."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from fields import uniform
from opencurrent_amd import _lib
from opencurrent_amd import _types as T
from opencurrent_amd._types import BC, BCSet, HostGrid
from opencurrent_amd.device import DeviceGrid

pytestmark = pytest.mark.gpu


def faces(kind):
    b = BCSet.uniform(T.BC_NEUMANN)
    if kind == "plates":
        b.zneg, b.xpos, b.yneg, b.ypos = (BC(T.BC_DIRICHELET, 0.0, 0.0) for _ in range(4))
    if kind == "periodic":
        b = BCSet.uniform(T.BC_PERIODIC)
    if kind == "periodic_z":
        b.zneg, b.zpos = BC(T.BC_PERIODIC, 0.0, 0.0), BC(T.BC_PERIODIC, 0.0, 0.0)
        b.xneg = BC(T.BC_DIRICHELET, 0.0, 0.0)
    return b


def filled(n, dtype, seed, bc, h):
    g = HostGrid(*n, dtype=dtype)
    g.interior()[:] = 2 * uniform(seed, n) - 1
    O.lib().orc_bc_fill(0, g.ptr(), C.byref(bc), *h)
    return g


def box(g):
    d = g.desc
    return g.full()[:d.nx + 2, :d.ny + 2, :d.nz + 2]


SIZES = [(4, 4, 4), (8, 8, 8), (14, 14, 14), (10, 18, 34), (24, 20, 28), (16, 40, 16)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["closed", "plates", "periodic", "periodic_z"])
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("start", ["given", "zero", "prolonged"])
@pytest.mark.parametrize("down", [False, True])
def test_smooth2_matches_oracle(gpu, n, kind, dtype, start, down):
    bc, h, hc = faces(kind), (.25, .5, .25), (.5, 1.0, .5)
    m = tuple(x // 2 for x in n)
    u, b = filled(n, dtype, 800, bc, h), HostGrid(*n, dtype=dtype)
    b.interior()[:] = 2 * uniform(801, n) - 1
    uc, bcoarse = filled(m, dtype, 802, bc, hc), HostGrid(*m, dtype=dtype)
    p = O.level_params(bc, 0, *h)
    hip = _lib.hip()
    gu, gb, guc, gbc = (DeviceGrid.from_host(x) for x in (u, b, uc, bcoarse))
    go = DeviceGrid.congruent(gu)
    small = any(x < 14 for x, per in zip(n, (kind == "periodic",) * 2 + (kind.startswith("periodic"),)) if per)
    assert hip.ocu_mg_smooth2_ok(gu.ptr(), go.ptr(), gb.ptr(), C.byref(bc)) == int(not small)
    if small:
        pytest.skip("periodic sides below 14 cells keep the separate launches")
    import torch
    parts = hip.ocu_norm_parts()
    ws = torch.full((2 * parts + 2,), 7.0, dtype=torch.float64, device="cuda")
    print(f"smooth2 {n} {kind} {np.dtype(dtype).name} {start} {down}", flush=True)
    _lib.check(hip.ocu_mg_smooth2(gu.ptr(), go.ptr(), gb.ptr(), guc.ptr() if start == "prolonged" else None,
                                  gbc.ptr() if down else None, C.byref(p), C.byref(bc),
                                  T.FUSED_ZERO_INPUT if start == "zero" else 0,
                                  C.cast(ws.data_ptr(), _lib.DP) if down else None, None), "smooth2")
    assert np.array_equal(gu.to_host().buf, u.buf)  # the input stays
    if start == "zero":
        u.buf[:] = 0
    if start == "prolonged":
        O.lib().orc_mg_prolong(uc.ptr(), u.ptr(), 1)
        O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)
    for _ in range(2):
        for color in (0, 1):
            O.lib().orc_mg_relax(u.ptr(), b.ptr(), color, C.byref(p), T.RELAX_DEVICE)
            O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)
    assert np.array_equal(box(go.to_host()), box(u))
    if down:
        r = HostGrid.congruent(u)
        O.lib().orc_mg_residual(u.ptr(), b.ptr(), r.ptr(), p.h, p.fx, p.fy, p.fz)
        O.lib().orc_mg_restrict(r.ptr(), bcoarse.ptr())
        assert np.array_equal(gbc.to_host().interior(), bcoarse.interior())
        got = ws.cpu().numpy()[:2 * parts].reshape(parts, 2)
        x = r.interior().astype(np.float64)
        assert abs(got[:, 0].sum() - (x ** 2).sum()) <= x.size * 2.0 ** -53 * (x ** 2).sum()
        assert got[:, 1].max() == np.abs(x).max()


def test_smooth2_refuses(gpu):
    """odd sides, face values, an alias and norms without the restriction"""
    bc, h = faces("closed"), (.25, .25, .25)
    p = O.level_params(bc, 0, *h)
    hip = _lib.hip()

    def call(n, bcs, flags=0, alias=False, ws=None):
        g = [DeviceGrid(*n) for _ in range(3)]
        out = g[0] if alias else g[1]
        return hip.ocu_mg_smooth2(g[0].ptr(), out.ptr(), g[2].ptr(), None, None, C.byref(p), C.byref(bcs), flags, ws,
                                  None)

    assert call((8, 8, 8), bc) == 0
    assert call((8, 7, 8), bc) < 0
    assert call((8, 8, 2), bc) < 0
    value = faces("closed")
    value.xneg = BC(T.BC_DIRICHELET, .5, 0.0)
    assert call((8, 8, 8), value) < 0
    assert call((8, 8, 8), bc, alias=True) < 0
    assert call((8, 8, 8), bc, flags=4) < 0
    import torch
    ws = torch.zeros(2 * hip.ocu_norm_parts() + 2, dtype=torch.float64, device="cuda")
    assert call((8, 8, 8), bc, ws=C.cast(ws.data_ptr(), _lib.DP)) < 0


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["closed", "plates", "periodic", "periodic_z"])
@pytest.mark.parametrize("nu", [(2, 2), (2, 1), (1, 2), (3, 2), (2, 3), (2, 0), (4, 2)])
def test_cycles_with_tiles_match_plain_launches(gpu, kind, dtype, nu):
    """V-cycles and FMG whose levels are relaxed by tiles where the counts are
    two, against one launch per colour: the same pressure, bit for bit, in
    the buffer the caller holds, over repeated runs (an odd and an even number
    of launches that exchange a level's buffers)"""
    from opencurrent_amd.solvers import MultigridPressure3D
    n, h = (48, 32, 40), (1 / 48, 1 / 32, 1 / 40)
    bc = faces(kind)
    b = HostGrid(*n, dtype=dtype)
    r = 2 * uniform(820, n) - 1
    b.interior()[:] = r - r.mean()
    got = []
    for plain in (True, False):
        gb = DeviceGrid.from_host(b)
        mg = MultigridPressure3D(gb, *h, bc, nu1=nu[0], nu2=nu[1], convergence=T.CONVERGENCE_NONE,
                                 use_fused_relax=not plain, use_bottom=not plain, use_fused_prolong=not plain)
        base = mg.pressure_desc().base
        out = []
        for runs in (lambda: mg.run_vcycles(1), lambda: mg.run_vcycles(2), lambda: mg.run_fmg(2),
                     lambda: mg.run_fmg(1)):
            assert runs()
            assert mg.pressure_desc().base == base
            out.append(mg.pressure().buf.copy())
        got.append(out)
    for a, c in zip(*got):
        assert np.all(np.isfinite(a))
        assert np.array_equal(a, c)
