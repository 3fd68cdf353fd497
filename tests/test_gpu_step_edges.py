"""The step kernels' shapes (1: a block per target; 2, 4: one, two targets a wavefront) where
their splits have edges: one target, targets that leave a wavefront or a block part empty,
partners about the 64 lanes and about the 32 a lane notes at once (2048 with one wavefront, 4096
with two); table pairs, and analytic pairs with SRPMF in range.  And that picking among the
shapes costs little beside a run.

Against the C oracle: energies and norm-wise forces 1e-10 relative, as the other parity tests
(FP64 sums of up to 4100 terms in another order, ~1e-13, and pair forms to a few ulp).
"""
import time

import numpy as np
import pytest

from bromoc_amd import abi, configs
from bromoc_amd.engine import Engine
from oracle.oracle import Oracle

from helpers import energy_errs, force_err, plain

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _ions(n):
    return plain(seed=n, n_per_type=n // 2 + 1, box=max(30.0, 8.5 * n ** (1.0 / 3.0)))


def _first(s, n):
    s = s.copy()
    s.ntot = s.capacity = n
    s.x, s.y, s.z, s.typei = (np.ascontiguousarray(v[:n]) for v in (s.x, s.y, s.z, s.typei))
    return s


def _check(s, tpb, monkeypatch):
    monkeypatch.setenv("BROMOC_TPB", str(tpb))
    g, o = Engine(s), Oracle(s)
    assert g.tuning() == tpb     # before ENERGY, which takes a default shape until it is set
    eg, eo = g.energy(), o.energy()
    bad = {k: v for k, v in energy_errs(eg, eo).items() if v > TOL}
    assert not bad, bad
    if s.ntot > 1:
        assert force_err(g.forces(), o.forces()) <= TOL


@pytest.mark.parametrize("tpb", [1, 2, 4])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 63, 64, 65, 257, 2047, 2049, 4095, 4097])
def test_table_pairs(n, tpb, monkeypatch):
    _check(_first(_ions(n), n), tpb, monkeypatch)


@pytest.mark.parametrize("tpb", [1, 2, 4])
@pytest.mark.parametrize("n", [2, 9, 65, 257, 2049])
def test_analytic_pairs(n, tpb, monkeypatch):
    s = configs.with_analytic(_first(_ions(n), n), seed=n)
    _check(s, tpb, monkeypatch)


def test_tuning_drops_losers():
    """Analytic ions, where the slowest shape takes sixty times the fastest: the tuning takes
    the time of 330 to 400 steps when slow shapes are dropped after a first round, of 1600 when every
    shape is timed to the end."""
    n = 1531
    s = configs.with_analytic(_first(_ions(n), n), seed=n)
    tune, step = [], []
    for _ in range(3):
        g = Engine(s)
        t0 = time.perf_counter()
        g.tuning()
        tune.append(time.perf_counter() - t0)
        g.step(64, abi.NOISE_PHILOX, seed=1, counter0=0)
        t0 = time.perf_counter()
        g.step(128, abi.NOISE_PHILOX, seed=1, counter0=64)
        step.append((time.perf_counter() - t0) / 128)
    ratio = min(tune) / min(step)
    print(f"tuning {1e3 * min(tune):.1f} ms, {ratio:.0f} steps")
    assert ratio < 750
