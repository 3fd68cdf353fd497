"""Positions, types and forces through the pinned staging: bit for bit what went in, at the
edges of the 256-thread blocks and past the 1024 blocks a launch takes (grid-stride), values
that a copy must not touch (infinities, not-a-number, -0, denormals), fewer and more particles
than the call before, a call that is refused leaving the state as it was, and replicas of
unequal capacity each returning its own.
"""
import numpy as np
import pytest

from bromoc_amd import configs
from bromoc_amd.abi import BromocError
from bromoc_amd.engine import Batch, Engine
from bromoc_amd.system import Replica

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
