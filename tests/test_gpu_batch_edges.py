"""Replica batches where the step kernel's blocks of 32 partners a lane, its lane groups and
its noise rows have their edges: replicas of one ion up to a few past G * 32 partners, all
lane counts, more steps than one draw of noise covers, pairs packed within table range.

Against single systems run by the C oracle on the same Philox streams; positions 1e-8 A after
the steps, energies 1e-10 relative (the other batch tests' bar).
"""
import numpy as np
import pytest

from bromoc_amd import abi, configs
from bromoc_amd.engine import Batch
from bromoc_amd.system import Replica, replica_system
from oracle.oracle import Oracle

from helpers import energy_errs

pytestmark = pytest.mark.gpu


def _replicas(sizes, seed):
    sh, _ = configs.replica_batch(seed=seed, nrep=1, n_range=(2, 2), box=(40.0, 40.0, 60.0),
                                  dcel=1.0, half_slab=8.0, gcmc=False)
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(np.arange(-4, 5), np.arange(-4, 5), np.arange(-6, -2), indexing="ij"),
                 -1).reshape(-1, 3) * 4.0
    reps = []
    for n in sizes:
        p = g[rng.choice(len(g), n, replace=False)] + rng.uniform(-0.9, 0.9, (n, 3))
        reps.append(Replica(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(),
                            typei=rng.permutation(sh.nold + 1 + np.arange(n) % 2).astype(np.int32),
                            capacity=n + int(rng.integers(0, 9)), phix=sh.phix.data))
    return sh, reps


@pytest.mark.parametrize("lanes", [8, 16, 32, 64])
def test_partner_blocks_and_lane_groups(lanes, monkeypatch):
    monkeypatch.setenv("BROMOC_BATCH_BLOCKS", "0")
    monkeypatch.setenv("BROMOC_BATCH_LANES", str(lanes))
    sh, reps = _replicas([1, 2, lanes - 1, lanes, lanes + 1, 255, 256, 257, 300], seed=lanes)
    b = Batch(sh, reps)
    steps = 19       # two draws of noise
    eb = b.run(steps, seed=3, counter0=70, energies=True)
    for r, rep in enumerate(reps):
        o = Oracle(replica_system(sh, rep), stream=r)
        eo = o.step(steps, abi.NOISE_PHILOX, seed=3, counter0=70)
        assert float(np.max(np.abs(b.get(r)[0] - o.positions()[0]))) <= 1e-8, r
        bad = {k: v for k, v in energy_errs(eb[r], eo).items() if v > 1e-10}
        assert not bad, (r, bad)
