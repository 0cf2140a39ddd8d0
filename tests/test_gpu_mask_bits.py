"""The solid mask's bits on the device (MASK_SOLID, MASK_BESIDE): any non-zero
byte means solid, a mask may be set again, and scattered, edge and corner
solids follow the oracle (each node beside one looks its donors up, the others
do not)."""
import numpy as np
import pytest

import nflow
from helpers import cfg, fp32_parity

pytestmark = pytest.mark.gpu

SHAPE = (13, 15, 70)  # ny, nz, nx


def scattered(share):
    m = np.random.default_rng(7).random(SHAPE) < share
    m[0, 0, 0] = m[-1, -1, -1] = m[5, 0, 64] = m[0, 7, -1] = True
    return m


@pytest.mark.parametrize("share", [0.0, 0.02, 0.3])
def test_scattered_solids_match_the_oracle(share):
    c = cfg(nx=70, ny=13, nz=15, enable_les=1, smagorinsky=0.17, tau=0.6, ref_vel=(0.05, 0.0, 0.02),
            init_lid_velocity=1)
    fp32_parity(c, 60, mask=scattered(share))


@pytest.mark.parametrize("storage", [nflow.F32, nflow.F16])
def test_any_non_zero_byte_is_solid_and_a_mask_can_be_set_again(storage):
    m = scattered(0.1)
    odd = np.where(m, np.random.default_rng(3).choice([2, 3, 4, 128, 255], SHAPE), 0).astype(np.uint8)
    out = []
    for given in (m.astype(np.uint8), odd):
        s = nflow.Solver(nflow.defaults(**cfg(nx=70, ny=13, nz=15, tau=0.6, init_lid_velocity=1), storage=storage))
        s.set_solid_mask(~m)
        nflow._check(nflow.lib().nflow_set_solid_mask(s.h, given.ctypes.data))
        s.initialize()
        s.run(30)
        out.append((s.read_arF(), s.node_type()[0]))
        s.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][1] == nflow.NODE_STRUCT, m)
