"""EFPOT table lookups on knot boundaries (getyd, polynom.f90:225-226) on the HIP path.

Two ions are placed exactly on knot distances r_k and one ulp either side.  The table jumps
by ~1e-9 kcal/mol at every knot (fixdy, polynom.f90:91-118), so a lookup that takes the
neighbouring segment -- as an index formed from a 1/sqrt that is one ulp off would -- misses
the oracle's pair energy by far more than the 1e-12 relative allowed here; the C oracle
itself is bit-identical to the reference on the same placements (test_oracle_vs_reference).
Checked through every launch shape of the step kernels and in the batch kernel.
"""
import numpy as np
import pytest

from bromoc_amd import abi, configs
from bromoc_amd.engine import Batch, Engine
from bromoc_amd.system import Replica, replica_system
from oracle.oracle import Oracle

from helpers import force_err

pytestmark = pytest.mark.gpu


def knot_positions(s, every=17, rmin=2.5):
    r = configs.knot_grid()
    out = []
    for k in range(1, len(r) - 1, every):
        if r[k] < rmin:
            continue
        for x in (r[k], np.nextafter(r[k], 0.0), np.nextafter(r[k], 1e9)):
            out.append(np.array([[0.0, 0.0, 0.0], [float(x), 0.0, 0.0]]))
    return out


@pytest.mark.parametrize("tpb", [1, 2, 4, 8])
def test_knot_boundaries(tpb, monkeypatch):
    monkeypatch.setenv("BROMOC_TPB", str(tpb))
    s = configs.plain_ions(seed=3, n_per_type=1, box=40.0)
    g, o = Engine(s), Oracle(s)
    assert g.tuning() == tpb
    bad = []
    for pos in knot_positions(s):
        g.set_positions(pos)
        o.set_positions(pos)
        eg, eo = g.energy(), o.energy()
        if abs(eg["eefpot"] - eo["eefpot"]) > 1e-12 * abs(eo["eefpot"]):
            bad.append((pos[1, 0], eg["eefpot"], eo["eefpot"]))
        assert force_err(g.forces(), o.forces()) <= 1e-12
    assert not bad, bad[:5]


@pytest.mark.parametrize("tpb", [1, 2, 4, 8, 17, 18, 20])
@pytest.mark.parametrize("x", [2.0, 4.0, 8.0, 16.0])
@pytest.mark.parametrize("side", ["below", "above"])
def test_root_next_to_a_tie(side, x, tpb, monkeypatch):
    """A distance whose square is a neighbour of a power of four: the exact root lies 2^-108
    (relative) below the tie between two doubles, lo and hi, with a knot between them, and only
    a correctly rounded root takes the segment below the knot."""
    monkeypatch.setenv("BROMOC_TPB", str(tpb))
    s = configs.plain_ions(seed=3, n_per_type=1, box=40.0).copy()
    if side == "below":            # hi = x, on a knot
        lo, hi, dy = float(np.nextafter(x, 0.0)), x, x * 2.0 ** -26.5
        pos = np.array([[0.0, 0.0, 0.0], [lo, dy, 0.0]])
    else:                          # lo = x; the table's start is moved by half the gap
        lo, hi, dy = x, float(np.nextafter(x, 100.0)), x * 2.0 ** -26
        pos = np.array([[0.0, 0.0, 0.0], [x, dy, 0.0]])
        s.pairs = [None if p is None else dict(p, dmi=p["dmi"] + 0.5 * (hi - lo)) for p in s.pairs]
    d2 = pos[1, 0] ** 2 + dy * dy
    seg = [int((v - s.pairs[1]["dmi"]) * (1.0 / s.res)) for v in (lo, hi)]
    assert seg[1] == seg[0] + 1 and np.sqrt(d2) == lo
    assert d2 == np.nextafter(x * x, 0.0 if side == "below" else 1e9)
    g, o = Engine(s), Oracle(s)
    assert g.tuning() == tpb
    g.set_positions(pos)
    o.set_positions(pos)
    eg, eo = g.energy(), o.energy()
    assert abs(eg["eefpot"] - eo["eefpot"]) <= 1e-12 * abs(eo["eefpot"])
    assert force_err(g.forces(), o.forces()) <= 1e-12


def _rms(e, exact):
    return float(np.sqrt(np.mean(((e - exact) / exact) ** 2)))


@pytest.mark.parametrize("tpb", [1, 2, 4, 17])
@pytest.mark.parametrize("analytic", [False, True])
def test_reciprocal_root_is_as_close_as_rounding(analytic, tpb, monkeypatch):
    """The pair energy fct / r of two ions beyond the tables has no more error over random
    distances than with the correctly rounded 1/sqrt: rms within 1.5 % (a reciprocal root
    with an rms error of 0.486 in units of 2^-53, instead of its rounding's 0.44, shows 5 %
    more)."""
    monkeypatch.setenv("BROMOC_TPB", str(tpb))
    s = configs.plain_ions(seed=3, n_per_type=1, box=200.0)
    if analytic:
        s = configs.with_analytic(s, seed=1, lj=False, srpmf=False)
    else:
        s = s.copy()
        s.pairs = [None if p is None else dict(p, sc3=0.0) for p in s.pairs]
    ta, tb = (int(s.nwtype[t]) for t in s.typei)
    fct = s.pairs[np.reshape(s.pairidx, (s.nttyp + 1, -1))[ta, tb]]["fct"]
    r = np.random.default_rng(5).uniform(21.0, 90.0, 6000)
    long = np.longdouble
    ri = (1.0 / np.sqrt((r * r).astype(long))).astype(np.float64)
    exact = long(fct) / r.astype(long)
    g, e = Engine(s), []
    assert g.tuning() == tpb
    for d in r:
        g.set_positions(np.array([[0.0, 0.0, 0.0], [d, 0.0, 0.0]]))
        e.append(g.energy()["eelec" if analytic else "eefpot"])
    ratio = _rms(np.array(e), exact) / _rms(fct * ri, exact)
    print(f"analytic {analytic} tpb {tpb}: {ratio:.4f}")
    assert ratio <= 1.015


def test_knot_boundaries_batch():
    """The batch step kernel's table lookup on the same placements, one replica per
    placement, energies after ENERGY-only evaluation."""
    s = configs.plain_ions(seed=3, n_per_type=1, box=40.0)
    sh, _ = configs.replica_batch(seed=1, nrep=1, n_range=(2, 2), box=(36.0, 36.0, 72.0),
                                  dcel=1.5, rpore=9.0, half_slab=10.0, gcmc=False)
    places = knot_positions(s, every=41)
    reps = []
    for pos in places:
        pos = pos + np.array([0.0, 0.0, 20.0])      # in the bath, clear of the pore walls
        reps.append(Replica(x=pos[:, 0].copy(), y=pos[:, 1].copy(), z=pos[:, 2].copy(),
                            typei=np.array([sh.nold + 1, sh.nold + 2], np.int32), nfix=0,
                            capacity=8, phix=np.zeros(sh.phix.data.shape, np.float32)))
    b = Batch(sh, reps)
    eb = b.energy()
    bad = []
    for r, rep in enumerate(reps):
        eo = Oracle(replica_system(sh, rep)).energy()
        if abs(eb[r]["eefpot"] - eo["eefpot"]) > 1e-12 * abs(eo["eefpot"]):
            bad.append((r, eb[r]["eefpot"], eo["eefpot"]))
    assert not bad, bad[:5]
