"""CPU checks of the native boundary: both libraries load without a GPU and
export every entry point their headers declare; the Python layout and the
C ABI structs agree with the headers."""
import ctypes as C
import os
import re
import subprocess
import sys
from pathlib import Path

import pytest

from opencurrent_amd import _lib
from opencurrent_amd import _types as T

ROOT = Path(__file__).resolve().parent.parent


def declared(header):
    text = (ROOT / "include" / header).read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = set(re.findall(r"\b(ocu_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


@pytest.mark.parametrize("header,loader", [("ocu_hip.h", _lib.hip), ("ocu.h", _lib.host)])
def test_every_declared_symbol_is_exported(header, loader):
    lib = loader()
    names = declared(header)
    assert len(names) > 20
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_bindings_cover_the_headers():
    assert set(declared("ocu_hip.h")) == set(_lib.HIP_SIGS)
    assert set(declared("ocu.h")) == set(_lib.HOST_SIGS)


def test_struct_sizes_match_the_c_layout():
    # ocu_bc: int32 + 2 floats; ocu_bc_set: 6 of them (boundary_condition.h:38-112)
    assert C.sizeof(T.BC) == 12
    assert C.sizeof(T.BCSet) == 72
    assert C.sizeof(T.Grid3DDesc) == 8 + 10 * 4 + 8 + 8
    assert C.sizeof(T.MGLevelParams) == 11 * 8
    # ocu_ns_step_params: nine int32 (padded to 40 bytes), eight doubles
    assert C.sizeof(T.NSStepParams) == 40 + 8 * 8
    assert T.NSStepParams.hx.offset == 40


def test_host_only_entry_points_without_gpu():
    hip = _lib.hip()
    assert hip.ocu_norm_parts() == 2048
    assert hip.ocu_reduce_workspace_bytes() == 8 * 2048


def test_invalid_arguments_are_rejected_before_any_launch():
    """Argument checks run on the host: a null or inconsistent descriptor is
    an OCU_ERR_INVALID with a message, and nothing is launched."""
    hip = _lib.hip()
    assert hip.ocu_bc_fill_level1(None, None, 1.0, 1.0, 1.0, None) == -1
    assert "null" in _lib.last_error()
    g = T.layout(8, 8, 8)
    g.base = 16  # bogus, but never dereferenced: the ghost check fails first
    g0 = T.layout(8, 8, 8, 0, 0, 0)
    g0.base = 16
    bc = T.BCSet.uniform(T.BC_NEUMANN)
    assert hip.ocu_bc_fill_level1(C.byref(g0), C.byref(bc), 1.0, 1.0, 1.0, None) == -1
    assert "ghost" in _lib.last_error()
    bad = T.BCSet.uniform(T.BC_FORCED_INFLOW_VARIABLE_SLIP)
    assert hip.ocu_bc_fill_level1(C.byref(g), C.byref(bad), 1.0, 1.0, 1.0, None) == -1
    assert "invalid boundary condition" in _lib.last_error()
    c = T.layout(4, 4, 4)
    c.base = 16
    assert hip.ocu_mg_residual_restrict(C.byref(g), C.byref(g), None, C.byref(T.layout(3, 4, 4)), 1.0, 1.0, 1.0,
                                        1.0, None, None) == -1


@pytest.mark.parametrize("entry", ["ocu_mg_coarse_relax", "ocu_mg_coarse_relax_filled"])
@pytest.mark.parametrize("n", [(0, 4, 4), (4, 0, 4), (4, 4, 0)])
def test_coarse_relax_of_an_empty_grid_returns(n, entry):
    """no host division by a side: the call comes back (with an error where no
    GPU is there to launch on)"""
    code = ("import ctypes as C\n"
            "from opencurrent_amd import _lib, _types as T\n"
            "u, b = T.layout(*%r), T.layout(*%r)\n"
            "u.base, b.base = 4096, 8192\n"
            "p, bc = T.MGLevelParams(), T.BCSet.uniform(T.BC_NEUMANN)\n"
            "_lib.hip().%s(C.byref(u), C.byref(b), 2, 0, C.byref(p), C.byref(bc), 1., 1., 1., 0, None)\n"
            "print('returned')\n" % (n, n, entry))
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")  # never a launch on these addresses
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.split()[-1:] == ["returned"], (r.returncode, r.stderr[-300:])


@pytest.mark.parametrize("which", ["u_coarse", "b_coarse"])
def test_smooth2_refuses_coarse_grids_beyond_its_offsets(which):
    """the kernel's byte offsets are 32-bit: a coarse grid padded beyond them
    is refused (in a process that sees no GPU: never a launch on these
    addresses)"""
    code = ("import ctypes as C\n"
            "from opencurrent_amd import _lib, _types as T\n"
            "u, o, b = (T.layout(4, 4, 4) for _ in range(3))\n"
            "wide = T.layout(2, 2, 2, 1, 1, 1, 0, 0, 1 << 25)\n"
            "for q, g in enumerate((u, o, b, wide)): g.base = 4096 * (q + 1)\n"
            "p, bc = T.MGLevelParams(), T.BCSet.uniform(T.BC_NEUMANN)\n"
            "uc, bc_out = (C.byref(wide), None) if %r == 'u_coarse' else (None, C.byref(wide))\n"
            "_lib.hip().ocu_mg_smooth2(C.byref(u), C.byref(o), C.byref(b), uc, bc_out, C.byref(p), C.byref(bc), 0, None,\n"
            "                          None)\n"
            "print(_lib.last_error())\n" % which)
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "32-bit offsets" in r.stdout, (r.returncode, r.stdout[-300:], r.stderr[-300:])


def test_missing_library_fails_loudly(tmp_path, monkeypatch):
    monkeypatch.setattr(_lib, "LIBDIR", tmp_path)
    monkeypatch.setattr(_lib, "_hip", None)
    with pytest.raises(_lib.NativeLibraryMissing):
        _lib.hip()


def test_init_grids_of_the_wrong_layout_are_refused_before_the_library():
    """IncompressibleNS3D / ScalarAdvection3D check their host init grids
    against the init_grids layouts (eqn_incompressns3d.h:78-86) before the
    library copies whole allocations from them"""
    import numpy as np
    from opencurrent_amd import solvers
    from opencurrent_amd._lib import NSParams, ScalarParams
    from opencurrent_amd._types import HostGrid
    import fields
    u, v, w, t = fields.mac_grids(8, 8, 8)
    for P, cls in ((NSParams, solvers.IncompressibleNS3D), (ScalarParams, solvers.ScalarAdvection3D)):
        p = P()
        p.nx = p.ny = p.nz = 8
        with pytest.raises(ValueError):
            cls(p, HostGrid(8, 8, 8), v, w, t)
        with pytest.raises(ValueError):
            cls(p, u, v, w, HostGrid.congruent(t, dtype=np.float32))
        p.nz = 9
        with pytest.raises(ValueError):
            cls(p, u, v, w, t)
