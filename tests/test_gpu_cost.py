"""Options cost about what their work does: times of steps against those of the same system
without the option, in one launch shape, so that a variant that spills its registers or takes
a general path for ordinary pairs is seen.  Bounds lie between the ratio a sound variant shows
and that of one with such a fault (in the comments), 7 % or more from either.
"""
import time

import pytest

from bromoc_amd import abi, configs
from bromoc_amd.engine import Engine

from helpers import plain, with_fixed

pytestmark = pytest.mark.gpu


def _times(s, tpb, monkeypatch, steps=48):
    """Best times of a step and of ENERGY (s)."""
    monkeypatch.setenv("BROMOC_TPB", str(tpb))
    e = Engine(s)
    assert e.tuning() == tpb
    e.step(steps, abi.NOISE_PHILOX, seed=1, counter0=0)
    out = []
    for run, n in ((lambda: e.step(steps, abi.NOISE_PHILOX, seed=1, counter0=0), steps), (e.energy, 1)):
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            run()
            t.append((time.perf_counter() - t0) / n)
        out.append(min(t))
    return out


def _rf(s, **kw):
    return configs.with_rfpar(s, seed=3, shape=(101, 101, 101), dcel=2.0, **kw)


def _ions(n=12000):
    return plain(seed=5, n_per_type=n // 2, box=198.0)


def test_analytic_pair_types_beside_tables(monkeypatch):
    s = configs.pore_dna(seed=5, n_bp=8, n_ions=2500, box=(88.0, 88.0, 176.0), dcel=1.0, rpore=12.0,
                         half_slab=10.0)
    a = _times(s, 1, monkeypatch)[0]
    b = _times(configs.with_analytic(s, types=[1, 4, 9], seed=3), 1, monkeypatch)[0]
    print(f"tables {1e6 * a:.1f} us, some analytic {1e6 * b:.1f} us: {b / a:.2f}")
    assert b <= 1.6 * a            # 1.38; 1.72 with 80 spilled registers


def test_reaction_field_with_zero_cells(monkeypatch):
    a = _times(_rf(_ions()), 17, monkeypatch)[0]
    b = _times(_rf(_ions(), zero_frac=0.05, wall_radius=60.0), 17, monkeypatch)[0]
    print(f"smooth {1e6 * a:.1f} us, zero cells {1e6 * b:.1f} us: {b / a:.2f}")
    assert b <= 1.6 * a            # 1.39; 1.75 with the pair forces in the masked sweep


@pytest.mark.parametrize("nfix", [0, 4000])
def test_energy_beside_a_step(nfix, monkeypatch):
    """ENERGY adds the energies and a transfer; masked sweeps and all."""
    step, energy = _times(with_fixed(_rf(_ions(), zero_frac=0.05, wall_radius=60.0), nfix), 17, monkeypatch)
    print(f"nfix {nfix}: step {1e6 * step:.1f} us, ENERGY {1e6 * energy:.1f} us: {energy / step:.2f}")
    assert energy <= 2.0 * step    # 1.2; 6.8 with spilled sums


def test_fixed_ions(monkeypatch):
    a = _times(_ions(), 17, monkeypatch)[0]
    b = _times(with_fixed(_ions(), 4000), 17, monkeypatch)[0]
    print(f"none fixed {1e6 * a:.1f} us, a third {1e6 * b:.1f} us: {b / a:.2f}")
    assert b <= 1.13 * a           # 0.96; 1.20 with the pair forces in the masked sweep
