"""k_sweep (two time steps per launch in row tiles) at the edges of its tiles:
widths on either side of the widest tile (322 nodes) and of a split, rows that
do and do not fill the 1,024 threads, single rows and planes, chunks of one
plane and taller than the box, channel ends on a tile's first and last column,
run-aligned and other widths, and batches of several lattices; each against
one step per launch, bit for bit."""
import numpy as np
import pytest

import nflow
from helpers import cfg

pytestmark = pytest.mark.gpu

LES = dict(enable_les=1, smagorinsky=0.17)


def channel(**kw):
    return cfg(casetype=nflow.CHANNEL, tau=0.56, inlet_peak=0.05, perturb=0.01, seed=3, **LES, **kw)


CASES = [
    cfg(nx=322, ny=4, nz=7, tau=0.6, init_lid_velocity=1, **LES),  # three whole rows per tile
    cfg(nx=323, ny=5, nz=6, tau=0.6, init_lid_velocity=1, **LES),  # split in x
    cfg(nx=1, ny=6, nz=40, tau=0.7, init_lid_velocity=1),  # 32 rows, the most
    cfg(nx=33, ny=3, nz=64, tau=0.6, enable_mrt=0, init_lid_velocity=1),  # 31 rows: 1,023 threads
    cfg(nx=128, ny=6, nz=17, tau=0.55, ref_vel=(0.05, 0.02, 0.03), **LES),  # run-aligned, 8 full rows
    cfg(nx=256, ny=1, nz=5, tau=0.6, init_lid_velocity=1),  # one plane
    channel(nx=322, ny=6, nz=9),
    channel(nx=324, ny=5, nz=8),  # two tiles of 162
    channel(nx=645, ny=4, nz=7),  # three tiles, the outlet's neighbour in its own
    channel(nx=128, ny=7, nz=33),
    channel(nx=3, ny=5, nz=70),
]


def run(inputs, temporal, steps_list, launches):
    b = nflow.Batch(inputs)
    b.set_tuning(256, 0, 0, 0, temporal)
    b.initialize()
    out = []
    for n in steps_list:
        b.run(n)
        out += [(b.read_arF(i), b.diagnostics(i)[0]) for i in range(len(inputs))]
    assert b.launches() == launches
    b.close()
    return out


def same(a, b):
    assert len(a) == len(b)
    for (x, m), (y, n) in zip(a, b):
        assert np.array_equal(x, y) and m == n


@pytest.mark.parametrize("k", range(len(CASES)))
def test_row_tiles_equal_one_step_per_launch(k):
    inp = [nflow.defaults(**CASES[k], storage=nflow.F32)]
    ref = run(inp, 0, [6, 5], 11)
    for h in (1, 2, 5, 200):
        same(run(inp, h, [6, 5], 8), ref)  # 3 pairs, the last re-run as 2 steps, 2 pairs and 1 step


@pytest.mark.parametrize("channels", [False, True])
def test_batches_of_several_lattices_equal_one_step_per_launch(channels):
    """Large enough that the automatic choice is two steps per launch."""
    inputs = [nflow.defaults(**cfg(nx=96, ny=100, nz=97, tau=0.55, init_lid_velocity=1, **LES)),
              nflow.defaults(**cfg(nx=150, ny=80, nz=90, tau=0.6, enable_mrt=0)),
              nflow.defaults(**cfg(nx=128, ny=96, nz=96, tau=0.53, **LES))]
    if channels:
        inputs.append(nflow.defaults(**channel(nx=300, ny=60, nz=64)))
    # 4 pairs, the last re-run as 2 steps; 1 pair and 2 steps; 3 pairs and 1 step
    same(run(inputs, -1, [8, 4, 7], 13), run(inputs, 0, [8, 4, 7], 19))
