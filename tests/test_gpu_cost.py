"""Options cost about what their work does: times of steps against those of the same system
without the option, in one launch shape, so that a variant that spills its registers or takes
a general path for ordinary pairs is seen.  Bounds lie between the ratio a sound variant shows
and that of one with such a fault (in the comments), some 15 % from either.
"""
import time

import pytest

from bromoc_amd import abi, configs
from bromoc_amd.engine import Engine

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


def test_analytic_pair_types_beside_tables(monkeypatch):
    s = configs.pore_dna(seed=5, n_bp=8, n_ions=2500, box=(88.0, 88.0, 176.0), dcel=1.0, rpore=12.0,
                         half_slab=10.0)
    a = _times(s, 1, monkeypatch)[0]
    b = _times(configs.with_analytic(s, types=[1, 4, 9], seed=3), 1, monkeypatch)[0]
    print(f"tables {1e6 * a:.1f} us, some analytic {1e6 * b:.1f} us: {b / a:.2f}")
    assert b <= 1.55 * a           # 1.38; 1.72 with 80 spilled registers
