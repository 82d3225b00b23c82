"""The MAC ghost fill in one launch against the oracle's three passes, bit for
bit over whole buffers: every combination of periodic and inflow axes with
different values and factors on all faces, from two cells per axis; and what
stays with the three launches (a face without a condition, mixed pairs, one
cell)."""
import ctypes as C
import itertools

import numpy as np
import pytest

import oracle_lib as O
from fields import mac_grids, uniform
from opencurrent_amd import _types as T
from opencurrent_amd import device as D
from opencurrent_amd._types import BC, BCSet

pytestmark = pytest.mark.gpu

PER, IN, NONE = T.BC_PERIODIC, T.BC_FORCED_INFLOW_VARIABLE_SLIP, T.BC_NONE
FACES = ("xneg", "xpos", "yneg", "ypos", "zneg", "zpos")


def bcs(types):
    b = BCSet.uniform(PER)
    for q, (f, t) in enumerate(zip(FACES, types)):
        setattr(b, f, BC(t, .25 * q - .6, .15 * q))
    return b


CASES = [tuple(t for x in axes for t in (x, x)) for axes in itertools.product((PER, IN), repeat=3)]
CASES += [(IN, PER, PER, PER, IN, IN), (PER, IN, IN, IN, NONE, IN), (NONE,) * 6]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [(2, 2, 2), (3, 2, 5), (16, 9, 64), (5, 66, 7), (1, 3, 2)])
def test_mac_fill_matches_passes(gpu, n, dtype):
    for types in CASES:
        u, v, w, _ = mac_grids(*n, dtype)
        for q, g in enumerate((u, v, w)):
            g.buf[:] = (2 * uniform(900 + q, g.buf.shape) - 1).astype(dtype)
        bc = bcs(types)
        dev = [D.DeviceGrid.from_host(g) for g in (u, v, w)]
        assert O.lib().orc_bc_fill_mac(u.ptr(), v.ptr(), w.ptr(), C.byref(bc)) == 1
        D.bc_fill_mac(*dev, bc)
        for got, want, name in zip(dev, (u, v, w), "uvw"):
            a = got.to_host().buf
            assert np.array_equal(a, want.buf), (types, name, int((a != want.buf).sum()))
