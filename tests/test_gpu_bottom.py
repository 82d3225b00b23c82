"""The bottom of a V-cycle and the coarsest level, by the general kernels and
by those that take u's ghosts from its cells (2x2x2 cells, or a pair of
cells, per thread), against the oracle's per-level operations, bit for bit:
every level's u with its ghosts and the b's below the top.  Sizes: one and several waves of blocks, more
blocks or pairs than a workgroup has threads (blocks reloaded per colour), a
coarsest level with odd sides; copy, sign-changing and periodic faces, the
anisotropic factors that FP32 keeps in float (powers of two) and others.
The operations are those of the oracle in its order, so the tolerance is
zero."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from fields import uniform
from opencurrent_amd import _lib
from opencurrent_amd import _types as T
from opencurrent_amd._types import BC, BCSet, HostGrid, MGLevelParams
from opencurrent_amd.device import DeviceGrid

pytestmark = pytest.mark.gpu


def faces(kind):
    b = BCSet.uniform(T.BC_NEUMANN)
    if kind == "plates":
        b.zneg, b.zpos, b.xpos = (BC(T.BC_DIRICHELET, 0.0, 0.0) for _ in range(3))
    if kind == "periodic":
        for f in ("xneg", "xpos", "zneg", "zpos"):
            setattr(b, f, BC(T.BC_PERIODIC, 0.0, 0.0))
        b.yneg = BC(T.BC_DIRICHELET, 0.0, 0.0)
    return b


def level(bc, h):
    """the parameters of a level >= 1 with spacings h, and its hmin"""
    return O.level_params(bc, 1, *(x / 2 for x in h))


def sweep(u, b, p, bc, h, host=False):
    """one red-black iteration with the fill that the two colours see (each
    colour's ghosts from the cells it updates: off periodic axes the second
    colour reads only ghosts of its own, which are as they were)"""
    for color in (0, 1):
        O.lib().orc_mg_relax(u.ptr(), b.ptr(), color, C.byref(p), T.RELAX_HOST if host else T.RELAX_DEVICE)
        if color or any(getattr(bc, f).type == T.BC_PERIODIC for f in BCSet.FACES):
            O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)


def coarsest(u, b, p, bc, h, iters, mode):
    if mode == 0:
        for _ in range(iters):
            sweep(u, b, p, bc, h, host=True)
        return
    ud, bd = HostGrid.congruent(u, dtype=np.float64), HostGrid.congruent(b, dtype=np.float64)
    ud.buf[:], bd.buf[:] = u.buf, b.buf
    for _ in range(iters):
        sweep(ud, bd, p, bc, h, host=True)
    u.buf[:] = ud.buf.astype(u.buf.dtype)


def oracle_vcycle(us, bs, ps, hs, bc, nu, iters, mode):
    last = len(us) - 1
    for l in range(last):
        for _ in range(nu):
            sweep(us[l], bs[l], ps[l], bc, hs[l])
        r = HostGrid.congruent(us[l])
        O.lib().orc_mg_residual(us[l].ptr(), bs[l].ptr(), r.ptr(), ps[l].h, ps[l].fx, ps[l].fy, ps[l].fz)
        O.lib().orc_mg_restrict(r.ptr(), bs[l + 1].ptr())
        us[l + 1].buf[:] = 0
    coarsest(us[last], bs[last], ps[last], bc, hs[last], iters, mode)
    for l in range(last - 1, -1, -1):
        O.lib().orc_mg_prolong(us[l + 1].ptr(), us[l].ptr(), 1)
        O.lib().orc_bc_fill(0, us[l].ptr(), C.byref(bc), *hs[l])
        for _ in range(nu):
            sweep(us[l], bs[l], ps[l], bc, hs[l])


def ghosts_equal(got, want, what):
    d = want.desc
    a, b = (g.full()[:d.nx + 2, :d.ny + 2, :d.nz + 2] for g in (got, want))
    assert np.array_equal(a, b), f"{what}: {np.abs(a - b).max()} at {np.argwhere(a != b)[:3].tolist()}"


SHAPES = {
    # (top level, levels): blocks of the top, pairs of the coarsest
    "one_wave": ((8, 8, 8), 2),         # 64 blocks, 32 pairs
    "three_levels": ((16, 16, 16), 3),  # 512 blocks
    "odd_coarsest": ((6, 10, 14), 2),   # coarsest 3 x 5 x 7
    "thin": ((4, 32, 4), 2),
    "wide": ((20, 20, 16), 2),          # 800 blocks: more than half a full workgroup
    "reloaded": ((24, 20, 28), 2),      # 1680 blocks: more than threads
    "one_wave_deep": ((8, 8, 8), 3),    # one wave for every level
    "two_waves": ((8, 8, 16), 3),       # a wave per small level, the coarsest back on the first
    "part_waves": ((12, 8, 24), 3),     # 288 blocks, 36 blocks, coarsest 3 x 2 x 6
    "four_levels": ((16, 16, 16), 4),
    "long_pairs": ((2, 2, 2052), 2),    # coarsest 1 x 1 x 1026
}


@pytest.mark.parametrize("mode", ["f64", "f32", "f32_double"])
@pytest.mark.parametrize("aniso", ["cube", "half", "ragged"])
@pytest.mark.parametrize("kind", ["closed", "plates", "periodic"])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_bottom_blocks_match_oracle(gpu, shape, kind, aniso, mode):
    n, nlev = SHAPES[shape]
    if kind == "periodic" and any(x % 2 for x in (n[0] >> (nlev - 1), n[2] >> (nlev - 1))):
        pytest.skip("periodic axes need even counts")
    dtype, cmode = (np.float64, 0) if mode == "f64" else (np.float32, int(mode == "f32_double"))
    bc = faces(kind)
    h0 = {"cube": (.125, .125, .125), "half": (.25, .25, .125), "ragged": (.1, .15, .125)}[aniso]
    us, bs, ps, hs = [], [], [], []
    for l in range(nlev):
        m = tuple(x >> l for x in n)
        h = tuple(x * 2 ** l for x in h0)
        u, b = HostGrid(*m, dtype=dtype), HostGrid(*m, dtype=dtype)
        b.interior()[:] = 2 * uniform(600 + l, m) - 1
        us.append(u), bs.append(b), hs.append(h)
        p = level(bc, h)
        p.h = min(h)
        ps.append(p)
    us[0].interior()[:] = 2 * uniform(610, n) - 1
    O.lib().orc_bc_fill(0, us[0].ptr(), C.byref(bc), *hs[0])
    print(f"bottom {shape} {kind} {aniso} {mode}", flush=True)
    match(us, bs, ps, hs, bc, cmode, ["ocu_mg_bottom_vcycle_filled", "ocu_mg_bottom_vcycle"])


def match(us, bs, ps, hs, bc, cmode, entries):
    """each entry point's bottom against the oracle's"""
    nlev, iters, hip = len(us), 5, _lib.hip()
    desc = lambda v: (T.Grid3DDesc * nlev)(*[x.desc for x in v])  # noqa: E731
    dev = [[[DeviceGrid.from_host(x) for x in v] for v in (us, bs)] for _ in entries]
    need = hip.ocu_mg_bottom_lds_bytes(desc(dev[0][0]), nlev, cmode)
    if need > hip.ocu_mg_bottom_lds_max():
        pytest.skip(f"needs {need} bytes of LDS")
    for entry, (gus, gbs) in zip(entries, dev):
        _lib.check(getattr(hip, entry)(desc(gus), desc(gbs), (MGLevelParams * nlev)(*ps),
                                       (C.c_double * (3 * nlev))(*[x for h in hs for x in h]), nlev, C.byref(bc), 2,
                                       2, iters, cmode, 0, None), "bottom")
    oracle_vcycle(us, bs, ps, hs, bc, 2, iters, cmode)
    for entry, (gus, gbs) in zip(entries, dev):
        for l in range(nlev):
            ghosts_equal(gus[l].to_host(), us[l], f"{entry}: u level {l}")
            if l:
                ghosts_equal(gbs[l].to_host(), bs[l], f"{entry}: b level {l}")


@pytest.mark.parametrize("mode", ["f64", "f32", "f32_double"])
@pytest.mark.parametrize("kind", ["closed", "plates", "values"])
@pytest.mark.parametrize("shape", ["three_levels", "odd_coarsest", "reloaded"])
def test_bottom_reads_the_ghosts_it_is_given(gpu, shape, kind, mode):
    """a ghost layer that is not the fill of u's cells is read as it stands
    (also beside faces with a value, which only the general kernel takes)"""
    n, nlev = SHAPES[shape]
    dtype, cmode = (np.float64, 0) if mode == "f64" else (np.float32, int(mode == "f32_double"))
    bc = faces("closed" if kind == "closed" else "plates")
    if kind == "values":
        bc.zneg, bc.yneg = BC(T.BC_DIRICHELET, .75, 0.0), BC(T.BC_NEUMANN, -.5, 0.0)
    us, bs, ps, hs = [], [], [], []
    for l in range(nlev):
        m, h = tuple(x >> l for x in n), (.125 * 2 ** l,) * 3
        u, b = HostGrid(*m, dtype=dtype), HostGrid(*m, dtype=dtype)
        b.interior()[:] = 2 * uniform(620 + l, m) - 1
        us.append(u), bs.append(b), hs.append(h)
        p = level(bc, h)
        p.h = min(h)
        ps.append(p)
    us[0].full()[:] = 2 * uniform(630, us[0].full().shape) - 1
    match(us, bs, ps, hs, bc, cmode, ["ocu_mg_bottom_vcycle"])


@pytest.mark.parametrize("mode", ["f64", "f32", "f32_double"])
@pytest.mark.parametrize("kind", ["closed", "plates", "periodic"])
@pytest.mark.parametrize("n", [(2, 2, 2), (4, 4, 4), (6, 4, 10), (12, 10, 14), (14, 12, 16)])
@pytest.mark.parametrize("order", [0, 1, 2])
def test_coarse_pairs_match_oracle(gpu, n, kind, mode, order):
    dtype, cmode = (np.float64, 0) if mode == "f64" else (np.float32, int(mode == "f32_double"))
    bc, h = faces(kind), (.5, .5, .5)
    u, b = HostGrid(*n, dtype=dtype), HostGrid(*n, dtype=dtype)
    u.interior()[:] = 2 * uniform(700, n) - 1
    b.interior()[:] = 2 * uniform(701, n) - 1
    O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)
    p = O.level_params(bc, 0, *h)
    print(f"pairs {n} {kind} {mode} {order}", flush=True)
    match_coarse(u, b, p, bc, h, order, cmode, ["ocu_mg_coarse_relax_filled", "ocu_mg_coarse_relax"])


def match_coarse(u, b, p, bc, h, order, cmode, entries):
    """each entry point's relaxation against the oracle's"""
    dev = [[DeviceGrid.from_host(x) for x in (u, b)] for _ in entries]
    for entry, (gu, gb) in zip(entries, dev):
        _lib.check(getattr(_lib.hip(), entry)(gu.ptr(), gb.ptr(), 6, order, C.byref(p), C.byref(bc), *h, cmode, None),
                   "coarse relax")
    dtype = u.buf.dtype
    work = [HostGrid.congruent(x, dtype=np.float64 if cmode else dtype) for x in (u, b)]
    work[0].buf[:], work[1].buf[:] = u.buf, b.buf
    for it in range(6):
        first = order == 1 or (order == 2 and it >= 3)
        for color in ((1, 0) if first else (0, 1)):
            O.lib().orc_mg_relax(work[0].ptr(), work[1].ptr(), color, C.byref(p), T.RELAX_HOST)
            O.lib().orc_bc_fill(0, work[0].ptr(), C.byref(bc), *h)
    want = u.copy()
    want.buf[:] = work[0].buf.astype(dtype)
    for entry, (gu, gb) in zip(entries, dev):
        ghosts_equal(gu.to_host(), want, f"{entry}: u")


@pytest.mark.parametrize("mode", ["f64", "f32", "f32_double"])
@pytest.mark.parametrize("kind", ["closed", "plates", "periodic"])
@pytest.mark.parametrize("n", [(2, 2, 2), (6, 4, 10), (12, 10, 14)])
@pytest.mark.parametrize("order", [0, 1, 2])
def test_coarse_relax_reads_the_ghosts_it_is_given(gpu, n, kind, mode, order):
    """a ghost layer that is not the fill of u's cells is read as it stands"""
    dtype, cmode = (np.float64, 0) if mode == "f64" else (np.float32, int(mode == "f32_double"))
    bc, h = faces(kind), (.5, .5, .5)
    u, b = HostGrid(*n, dtype=dtype), HostGrid(*n, dtype=dtype)
    u.full()[:] = 2 * uniform(720, u.full().shape) - 1
    b.interior()[:] = 2 * uniform(721, n) - 1
    match_coarse(u, b, O.level_params(bc, 0, *h), bc, h, order, cmode, ["ocu_mg_coarse_relax"])


def test_faces_the_blocks_do_not_take(gpu):
    """a face value keeps the general kernels: same bits as the oracle"""
    n, h = (8, 8, 8), (.25, .25, .25)
    bc = faces("plates")
    bc.zneg = BC(T.BC_DIRICHELET, .75, 0.0)
    u, b = HostGrid(*n), HostGrid(*n)
    u.interior()[:] = 2 * uniform(710, n) - 1
    b.interior()[:] = 2 * uniform(711, n) - 1
    O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)
    p = O.level_params(bc, 0, *h)
    gu, gb = DeviceGrid.from_host(u), DeviceGrid.from_host(b)
    _lib.check(_lib.hip().ocu_mg_coarse_relax(gu.ptr(), gb.ptr(), 4, 0, C.byref(p), C.byref(bc), *h, 0, None), "relax")
    for _ in range(4):
        for color in (0, 1):
            O.lib().orc_mg_relax(u.ptr(), b.ptr(), color, C.byref(p), T.RELAX_HOST)
            O.lib().orc_bc_fill(2, u.ptr(), C.byref(bc), *h)
    O.lib().orc_bc_fill(0, u.ptr(), C.byref(bc), *h)
    ghosts_equal(gu.to_host(), u, "u")
