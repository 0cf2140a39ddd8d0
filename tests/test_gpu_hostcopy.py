"""Copies between device memory and the caller's arrays (csrc/hostcopy.hpp):
populations written and read back unchanged at sizes on either side of the
plain, single and chunked paths (1 and 3 MiB out, 32 MiB in), of one chunk (2
MiB) and of all eight (16 MiB, where chunks are used again), into views that start off any
boundary; and from several host threads at once, more than the pool has pinned
memory for among them."""
import threading

import numpy as np
import pytest

import nflow
from helpers import cfg

pytestmark = pytest.mark.gpu


def field(shape, seed):
    a = np.zeros(shape, dtype=np.float32)
    r = np.random.default_rng(seed)
    a[1:-1, 1:-1, 1:-1] = r.random((shape[0] - 2, shape[1] - 2, shape[2] - 2, 19), dtype=np.float32) * 0.01 + 0.05
    return a


def round_trip(nx, ny, nz, seed):
    s = nflow.Solver(nflow.defaults(**cfg(nx=nx, ny=ny, nz=nz), storage=nflow.F32))
    a = field((ny + 2, nz + 2, nx + 2, 19), seed)
    s.write_arF(a)
    back = s.read_arF()
    # the same through pointers off any alignment but the element's
    raw = np.empty(a.size + 1, dtype=np.float32)[1:]
    raw[:] = a.reshape(-1)
    nflow._check(nflow.lib().nflow_write_arF(s.h, nflow._fp(raw)))
    raw[:] = -1.0
    nflow._check(nflow.lib().nflow_read_arF(s.h, nflow._fp(raw)))
    m = s.read_macro()
    s.close()
    rho = a[1:-1, 1:-1, 1:-1].astype(np.float64).sum(-1)
    return np.array_equal(back, a) and np.array_equal(raw, a.reshape(-1)) and np.allclose(m[0], rho, rtol=1e-6)


# 19 * 4 * (nx + 2)(ny + 2)(nz + 2) bytes: 0.9, 1.1, 2.9, 3.2, 16.7 and 37 MB
@pytest.mark.parametrize("n", [(21, 21, 21), (23, 22, 22), (32, 31, 32), (33, 33, 32), (60, 58, 57), (78, 77, 76)])
def test_populations_come_back_unchanged(n):
    assert round_trip(*n, seed=sum(n))


def test_two_host_threads_at_once():
    ok = {}

    def work(k):
        ok[k] = all(round_trip(50 + k, 49, 48 + j, seed=10 * k + j) for j in range(3))

    t = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert ok == {0: True, 1: True, 2: True}


@pytest.mark.parametrize("count,n", [(18, (12, 11, 10)), (6, (50, 49, 48))])
def test_more_copies_at_once_than_the_pool_holds(count, n):
    """16 blocks and 4 sets of chunks: the others take plain copies."""
    solvers = [nflow.Solver(nflow.defaults(**cfg(nx=n[0], ny=n[1], nz=n[2]), storage=nflow.F32)) for _ in range(count)]
    given = [field((n[1] + 2, n[2] + 2, n[0] + 2, 19), k) for k in range(count)]
    gate = threading.Barrier(count)
    ok = [False] * count

    def work(k):
        gate.wait()
        good = True
        for _ in range(8):
            solvers[k].write_arF(given[k])
            good = good and np.array_equal(solvers[k].read_arF(), given[k])
            mass = given[k].sum(dtype=np.float64)  # rho: 19 terms added in FP32
            good = good and abs(solvers[k].diagnostics()[0] - mass) < 19 * 2.0 ** -24 * mass
        ok[k] = good

    t = [threading.Thread(target=work, args=(k,)) for k in range(count)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    for s in solvers:
        s.close()
    assert all(ok)
