"""k_small (a whole FP32 cavity in LDS, many steps per launch) against one step
per launch, bit for bit: at one and two nodes per thread and on either side of
the switch between them, up to its largest lattice and one node beyond, single
nodes and rows, runs of odd and even length and longer than one launch, a
batch, and restarts from an exported state."""
import numpy as np
import pytest

import nflow
from helpers import cfg

pytestmark = pytest.mark.gpu

SHAPES = [(10, 10, 10), (1, 1, 1), (3, 2, 5), (16, 8, 8), (41, 5, 5), (12, 12, 12), (1920, 1, 1), (17, 113, 1),
          (8, 15, 16)]


def inp(shape, vy=0.01, **kw):
    return nflow.defaults(**cfg(nx=shape[0], ny=shape[1], nz=shape[2], tau=0.56, ref_vel=(0.05, vy, 0.03),
                                init_lid_velocity=1, **kw), storage=nflow.F32)


def states(inputs, temporal, runs, launches=None):
    """The states after each run; launches: of all runs (default: one a step)."""
    b = nflow.Batch(inputs)
    b.set_tuning(256, 0, 0, 10, temporal)
    b.initialize()
    out = []
    for n in runs:
        b.run(n)
        out += [(b.read_arF(i), b.diagnostics(i)) for i in range(len(inputs))]
    assert b.launches() == (sum(runs) if launches is None else launches)
    b.close()
    return out


def same(a, b):
    for (x, d), (y, e) in zip(a, b):
        assert np.array_equal(x, y)
        assert d[0] == e[0] and np.array_equal(d[1], e[1]) and d[2] == e[2]


@pytest.mark.parametrize("les", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_lattices_in_lds_equal_one_step_per_launch(shape, les):
    c = [inp(shape, enable_mrt=les, enable_les=les, smagorinsky=0.17 * les)]
    runs = [1, 2, 9, 12]
    fits = shape[0] * shape[1] * shape[2] <= 1920
    same(states(c, -1, runs, launches=len(runs) if fits else None), states(c, 0, runs))


def test_runs_longer_than_one_launch():
    # no lid velocity along y: the lid's (5 - 2)(6 - 2) nodes would take mass
    # out at every step, until none is left
    c = [inp((5, 4, 6), vy=0.0)]
    same(states(c, -1, [4097, 8192], launches=4), states(c, 0, [4097, 8192]))


def test_a_batch_of_small_lattices_and_one_with_a_larger():
    small = [inp(s, enable_mrt=i % 2) for i, s in enumerate(SHAPES) if s != (17, 113, 1)]
    same(states(small, -1, [7, 10], launches=2), states(small, 0, [7, 10]))
    mixed = small + [inp((16, 16, 16))]
    same(states(mixed, -1, [7, 10]), states(mixed, 0, [7, 10]))


def test_restart_from_an_exported_state():
    a = nflow.Solver(inp((10, 11, 9)))
    a.initialize()
    a.run(20)
    mid = a.read_arF()
    a.run(15)
    b = nflow.Solver(inp((10, 11, 9)))
    b.write_arF(mid)
    b.run(15)
    assert np.array_equal(a.read_arF(), b.read_arF())
    a.close()
    b.close()


@pytest.mark.parametrize("count", [1, 16])
def test_the_autotuner_times_and_keeps_it(count):
    """10^3 runs at 1.75 us per step in LDS and 3.3 with one step per launch."""
    b = nflow.Batch([inp((10, 10, 10))] * count)
    assert b.autotune(steps_per_trial=20)["temporal"] == -1
    before = b.launches()
    b.run(100)
    assert b.launches() - before == 1
    b.close()
