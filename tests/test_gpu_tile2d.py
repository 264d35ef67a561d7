"""Several 2D steps in one launch (tiles with recomputed halos) against the
FP64 oracle: grids around the tile sizes, step counts around the launch
length, every tile shape, poles and CPML across tile edges, H and E sources,
detectors with intervals, and captured graphs between plain steps."""
import json

import numpy as np
import pytest

import chiml_amd
from chiml_amd import decks
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-9, "fp32": 1e-5}


def _deck(n, prec, pml=6, steps=60, d=0.05, poles=True, filled=True):
    dk = decks.empty_deck((n[0], n[1], 1), d, steps, pml, precision=prec)
    if filled:
        r = (min(n) - 2 * pml) / 2.0 - 1.3
        dk["ObjectList"].append({"shape": "cylinder", "material": "custom", "eps": 2.5, "pols": decks.gold_like_pols() if poles else [],
                                 "radius": r * d, "length": 1.0, "loc": [0.2 * d, -0.3 * d, 0.0], "Basis_Set": [],
                                 "unit_vectors": [{"uvec": [1, 0, 0]}, {"uvec": [0, 0, 1]}, {"uvec": [0, 1, 0]}]})
    fc = 0.2
    for k, (pol, x, w) in enumerate((("Ez", n[0] // 2 + 1, 0), ("Ez", n[0] // 2, 3), ("Hx", n[0] // 2 - 1, 2), ("Hy", pml + 1, 0))):
        pulse = decks.gaussian_pulse(fc, 0.5 + 0.1 * k, 3.0, 1.0 + k)
        pulse["t_0"] = 0.2
        dk["SourceList"].append({"pol": pol, "size": [w * d, 0.0, 0.0], "PulseList": [pulse],
                                 "loc": [decks._pos(x, n[0], d) + w * d / 2.0, decks._pos(n[1] // 2 + k, n[1], d), 0.0]})
    for k, t in enumerate(("Ez", "Hx", "Hy", "Epow")):
        dk["DetectorList"].append({"type": t, "dtc_class": "cout", "fname": "d", "size": [(2 if k == 0 else 0) * d, 0.0, 0.0],
                                   "Time_Interval": decks.dt_of(d) * (1.01 + k),
                                   "loc": [decks._pos(n[0] // 2 - 3 + 3 * k, n[0], d), decks._pos(n[1] // 2 + 2 - k, n[1], d), 0.0]})
    return json.dumps(dk)


def _compare(sim, orc, prec):
    for fam in ((2,), (3, 4)):
        ref = [orc.field(c) for c in fam]
        peak = max(float(np.max(np.abs(r))) for r in ref)
        assert peak > 0
        for c, r in zip(fam, ref):
            assert float(np.max(np.abs(sim.field(c) - r))) <= TOL[prec] * peak, c
    for k, det in enumerate(sim.dtcArr()):
        v, r = det.series()[1], np.asarray(orc.detector(k)[1])
        assert v.shape == r.shape
        peak = float(np.max(np.abs(r)))
        assert float(np.max(np.abs(v - r))) <= TOL[prec] * max(peak, 1e-30), k


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [(16, 16), (17, 31), (33, 32), (48, 47), (49, 65), (64, 19), (81, 50)])
def test_small_tiles(n, prec):
    deck = _deck(n, prec, pml=3 if min(n) < 30 else 6)
    sim, orc = chiml_amd.FDTDField(deck), Oracle(deck)
    for k in (1, 8, 9, 3, 16):  # shorter, equal and longer than one launch
        sim.step(k)
        orc.step(k)
    sim.sync()
    _compare(sim, orc, prec)
    sim.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [(520, 517), (701, 650)])
def test_large_tiles(n, prec):
    deck = _deck(n, prec, pml=10)
    sim, orc = chiml_amd.FDTDField(deck), Oracle(deck)
    sim.step(21)
    sim.sync()
    orc.step(21)
    _compare(sim, orc, prec)
    sim.close()


def test_graphs_and_plain_steps_agree():
    deck = _deck((75, 66), "fp32", steps=200)
    a, b = chiml_amd.FDTDField(deck), chiml_amd.FDTDField(deck)
    b.set_graph(24)  # three launches' worth: a graph holds an even number of them
    for k in (5, 48, 7, 24, 26, 50, 24):
        a.step(k)
        b.step(k)
        a.sync()
        b.sync()
        for c in (2, 3, 4):
            assert np.array_equal(a.field(c), b.field(c)), (k, c)
    for x, y in zip(a.dtcArr(), b.dtcArr()):
        assert np.array_equal(x.series()[1], y.series()[1])
    a.close()
    b.close()
