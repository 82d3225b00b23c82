"""The fused NS step's march over T's interior and its shell against the
per-operator kernels, bit for bit over every element: tiles of 64 cells and 8
or 16 rows exactly full, one short and one over, several chunks of planes,
and axes of one to three cells, where second-order upwind's far samples wrap
onto the cell's own neighbours - with the flow and the temperature periodic
along different axes."""
import ctypes as C

import numpy as np
import pytest

from fields import mac_grids, uniform
from opencurrent_amd import _lib
from opencurrent_amd import _types as T
from opencurrent_amd._types import NSStepParams
from opencurrent_amd.device import DeviceGrid
from test_gpu_ns_fused import _reference_sequence, tbc_mixed, tbc_periodic_xy

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 3, 1), (3, 2, 5), (20, 8, 64), (9, 17, 65), (7, 16, 63), (5, 33, 130), (300, 9, 7)]


@pytest.mark.parametrize("scheme", [T.IT_FIRST_ORDER_UPWIND, T.IT_SECOND_ORDER_CENTERED, T.IT_SECOND_ORDER_UPWIND])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", SIZES)
def test_march_equals_operators(gpu, n, dtype, scheme):
    import torch
    bits = torch.int64 if dtype == np.float64 else torch.int32
    for flow, temp, vert, tbc in ((0, 0, T.DIR_XPOS, tbc_mixed()), (3, 3, T.DIR_YNEG, tbc_periodic_xy()),
                                  (5, 6, T.DIR_ZPOS, tbc_mixed()), (7, 0, T.DIR_XNEG, tbc_periodic_xy())):
        hosts = mac_grids(*n, dtype=dtype)
        for q, g in enumerate(hosts):
            g.buf[:] = (2 * uniform(8700 + q, g.buf.shape) - 1).astype(dtype)
        p = NSStepParams()
        p.nx, p.ny, p.nz = n
        p.advection_scheme, p.vertical_direction = scheme, vert
        p.flow_periodic, p.temp_periodic = flow, temp
        p.keep_tendencies = p.use_last = int(flow == 3)
        p.hx, p.hy, p.hz = .5, .25, .125
        p.viscosity, p.thermal_diffusion = (0.0, .02) if flow == 5 else (.01, 0.0) if flow == 7 else (.01, .02)
        p.thermal_coef, p.a_dt = -.75, float(np.float32(1e-2))
        p.a_ab = float(np.float32(-3e-3)) if p.use_last else 0.0
        ref, old = ([DeviceGrid.from_host(g) for g in hosts] for _ in range(2))
        new, d_ref, d_new, last = ([DeviceGrid.congruent(g) for g in old] for _ in range(4))
        for q, g in enumerate(last):
            g.interior().copy_(torch.as_tensor(uniform(8800 + q, tuple(g.interior().shape)).astype(dtype)))
        _reference_sequence(ref, d_ref, last, p, tbc, p.use_last, p.keep_tendencies)
        _lib.check(_lib.hip().ocu_ns_step_fused(*(g.ptr() for g in old), *(g.ptr() for g in new),
                                                *(g.ptr() for g in d_new), *(g.ptr() for g in last), C.byref(p),
                                                C.byref(tbc), None), "fused step")
        for q in range(4):
            a, b = new[q].tensor.view(bits), ref[q].tensor.view(bits)
            assert torch.equal(a, b), (flow, "uvwT"[q], int((a != b).sum()))
            if p.keep_tendencies:
                assert torch.equal(d_new[q].interior(), d_ref[q].interior()), (flow, "d uvwT"[q])
