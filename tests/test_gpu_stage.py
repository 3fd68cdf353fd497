"""Positions, types and forces through the pinned staging: bit for bit what went in, at the
edges of the 256-thread blocks and past the 1024 blocks a launch takes (grid-stride), values
that a copy must not touch (infinities, not-a-number, -0, denormals), fewer and more particles
than the call before, a call that is refused leaving the state as it was, replicas of
unequal capacity each returning its own, one of more particles than are staged at a time,
and one whose capacity is large but whose particles are few.
"""
import ctypes as C

import numpy as np
import pytest

from bromoc_amd import configs
from bromoc_amd.abi import BromocError
from bromoc_amd.engine import Batch, Engine
from bromoc_amd.system import Replica, ptr

from helpers import plain

pytestmark = pytest.mark.gpu


def _sized(n):
    s = plain(seed=5, n_per_type=2).copy()
    rng = np.random.default_rng(n)
    s.ntot = s.capacity = n
    s.x, s.y, s.z = rng.uniform(-5.0, 5.0, (3, n))
    s.typei = rng.integers(1, 3, n).astype(np.int32)
    return s


def _bits(a):
    return np.ascontiguousarray(a).view(np.int64)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1024 * 256 + 7])
def test_positions_come_back_as_they_went_in(n):
    g = Engine(_sized(n))
    rng = np.random.default_rng(n + 1)
    for m in (n, max(1, n - 3), n):
        p = rng.uniform(-9.0, 9.0, (m, 3))
        p.flat[:3] = [np.inf, np.nan, -0.0]
        p.flat[-1] = 5e-324
        t = rng.integers(1, 3, m).astype(np.int32)
        g.set_positions(p, t)
        q, u = g.positions()
        assert np.array_equal(_bits(p), _bits(q)) and np.array_equal(t, u)


def test_refused_call_changes_nothing_and_forces_follow():
    s = _sized(300)
    g, h = Engine(s), Engine(s)
    p, t = g.positions()
    bad = t.copy()
    bad[-1] = 99
    with pytest.raises(BromocError):
        g.set_positions(p + 1.0, bad)
    assert np.array_equal(g.positions()[0], p) and np.array_equal(g.positions()[1], t)
    g.energy()
    h.set_positions(p)          # the same state by the other route
    h.energy()
    assert np.array_equal(g.forces(), h.forces())


def test_replicas_of_unequal_capacity():
    sh, reps = configs.replica_batch(seed=4, nrep=5, n_range=(2, 300), box=(40.0, 40.0, 60.0),
                                     dcel=1.0, half_slab=8.0, gcmc=False)
    reps = [Replica(x=r.x, y=r.y, z=r.z, typei=r.typei, capacity=len(r.x) + 5 * k, phix=r.phix)
            for k, r in enumerate(reps)]
    b = Batch(sh, reps)
    for k in (0, 4, 1, 3, 2):
        pos, typei, n = b.get(k)[:3]
        assert n == len(reps[k].x)
        assert np.array_equal(pos[:n], np.stack([reps[k].x, reps[k].y, reps[k].z], 1))
        assert np.array_equal(typei[:n], reps[k].typei)


def _one_replica(n, capacity):
    sh, _ = configs.replica_batch(seed=4, nrep=1, n_range=(2, 2), box=(40.0, 40.0, 60.0), dcel=1.0,
                                  half_slab=8.0, gcmc=False)
    rng = np.random.default_rng(n)
    p = rng.uniform(-15.0, 15.0, (n, 3))
    t = rng.integers(sh.nold + 1, sh.ntype + 1, n).astype(np.int32)
    rep = Replica(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), typei=t, capacity=capacity,
                  phix=sh.phix.data)
    return Batch(sh, [rep]), p, t


@pytest.mark.parametrize("n", [32767, 32768, 32769, 2 * 32768 + 5])
def test_replica_staged_in_parts(n):
    b, p, t = _one_replica(n, n + 7)
    for _ in range(2):
        pos, typei, m = b.get(0)[:3]
        assert m == n
        assert np.array_equal(pos[:n], p) and np.array_equal(typei[:n], t)


def test_staging_is_bounded():
    """100 particles in a replica of 4 million slots (32 bytes each): reading them back takes
    some megabytes of the process's address space, not the slots' 134."""
    def size_mb():
        with open("/proc/self/status") as f:
            return next(int(v.split()[1]) for v in f if v.startswith("VmSize")) / 1024.0

    _one_replica(100, 200)[0].get(0)      # what the first transfer of a process sets up
    b, p, _ = _one_replica(100, 1 << 22)
    x, n = np.zeros((3, 100)), C.c_int32()
    before = size_mb()
    rc = b.lib.bromoc_batch_get(b.ctx, 0, ptr(x[0]), ptr(x[1]), ptr(x[2]), None, C.byref(n), None,
                                None, None)
    grown = size_mb() - before
    assert rc == 0 and n.value == 100 and np.array_equal(x.T, p)
    print(f"address space grown by {grown:.1f} MB")
    assert grown <= 32.0
