"""Rows stored in whole 16-byte groups: grids and CPML slabs whose sizes are no
multiple of a group (4 cells in FP32, 2 in FP64), down to slabs that meet in
the middle (one thread per cell there), against the FP64 oracle."""
import json

import numpy as np
import pytest

import chiml_amd
from chiml_amd import decks
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-9, "fp32": 1e-5}


def _deck(n, pml, prec, steps=40, d=0.02):
    three = n[2] > 1
    dk = decks.empty_deck(n, d, steps, pml, precision=prec)
    loc = [0.3 * d, -0.4 * d, 0.2 * d if three else 0.0]
    ob = {"shape": "sphere" if three else "cylinder", "material": "custom", "eps": 2.0, "pols": decks.gold_like_pols(), "radius": 2.6 * d,
          "loc": loc, "Basis_Set": []}
    if not three:
        ob.update({"length": 1.0, "unit_vectors": [{"uvec": [1, 0, 0]}, {"uvec": [0, 0, 1]}, {"uvec": [0, 1, 0]}]})
    dk["ObjectList"].append(ob)
    src = [decks._pos(n[0] // 2 + 2, n[0], d), decks._pos(n[1] // 2, n[1], d), decks._pos(n[2] // 2 - 1, n[2], d) if three else 0.0]
    pulse = decks.gaussian_pulse(0.3, 1.0, 3.0, 1.0)
    pulse["t_0"] = 0.1
    dk["SourceList"].append({"pol": "Ez", "size": [0.0] * 3, "loc": src, "PulseList": [pulse]})
    # the last cells of a row, which share their group with the padding
    for t in ("Ez", "Hy"):
        dk["DetectorList"].append({"type": t, "dtc_class": "cout", "fname": "d", "size": [0.0] * 3,
                                   "loc": [decks._pos(n[0] - 2, n[0], d), src[1], src[2]]})
    if three:
        dk["FluxList"].append({"name": "flux", "size": [6 * d] * 3, "loc": [0.0] * 3, "lamL": 4.0, "lamR": 8.0, "nfreq": 4})
    return json.dumps(dk)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,pml", [((20, 18, 17), 4), ((21, 18, 17), 5), ((22, 19, 16), 3), ((23, 17, 18), 6), ((17, 16, 17), 7),
                                   ((13, 15, 16), 6), ((19, 18, 17), 0), ((33, 30, 1), 7), ((35, 21, 1), 5), ((21, 22, 1), 7), ((37, 24, 1), 0)])
def test_any_row_and_slab_size(n, pml, prec):
    deck = _deck(n, pml, prec)
    sim = chiml_amd.FDTDField(deck)
    sim.step(40)
    sim.sync()
    orc = Oracle(deck)
    orc.step(40)
    three = n[2] > 1
    for fam in (range(3), range(3, 6)):
        comps = [c for c in fam if three or c in (2, 3, 4)]
        ref = [orc.field(c) for c in comps]
        peak = max(float(np.max(np.abs(r))) for r in ref)
        assert peak > 0
        for c, r in zip(comps, ref):
            assert float(np.max(np.abs(sim.field(c) - r))) <= TOL[prec] * peak, c
    for k, det in enumerate(sim.dtcArr()):
        r = np.asarray(orc.detector(k)[1])
        fam = max(float(np.max(np.abs(orc.field(c)))) for c in ((2,) if k == 0 else (3, 4)))
        scale = max(float(np.max(np.abs(r))), fam if k == 0 else 0.0)
        assert float(np.max(np.abs(det.series()[1].ravel() - r.ravel()))) <= TOL[prec] * scale
    if three:
        f = orc.flux(0)
        f = f[1] if isinstance(f, tuple) else f
        assert float(np.max(np.abs(sim.fluxArr()[0].getFlux() - f))) <= TOL[prec] * float(np.max(np.abs(f)))
    sim.close()
