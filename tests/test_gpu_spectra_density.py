"""Flux spectra combined on the device (k_flux_faces) and the density kernel with
one lane per stored entry (k_ml_entry), against the FP64 oracle: 1e-9 in FP64
(1e-10 on populations).  An FP32 field is within 1e-5 of its peak, so the sum of
products of two of them is held to 2e-5 times five, for the parts of a face
whose flux cancels."""
import json

import numpy as np
import pytest

import chiml_amd
from chiml_amd import decks
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu

# cells a side: boxes and single planes of each normal, even and odd Simpson intervals
BOXES = [(7, 7, 7), (6, 9, 8), (1, 8, 7), (9, 1, 6), (6, 7, 1)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-4)])
@pytest.mark.parametrize("steps", [64, 77])  # whole blocks of 32 samples, and a part of one
@pytest.mark.parametrize("nfreq", [3, 70])
def test_flux_boxes_and_planes(nfreq, steps, prec, tol):
    d = 0.02
    dk = decks.empty_deck((26, 25, 27), d, steps, 5, precision=prec)
    pulse = decks.gaussian_pulse(1.0, 1.0, 3.0, 1.0)
    pulse["t_0"] = 0.1
    dk["SourceList"].append({"pol": "Ez", "size": [0.0] * 3, "loc": [2 * d, -d, d], "PulseList": [pulse]})
    for k, b in enumerate(BOXES):
        dk["FluxList"].append({"name": f"f{k}", "size": [(c - 1) * d for c in b], "loc": [0.0] * 3, "lamL": 0.2, "lamR": 1.5,
                               "nfreq": nfreq})
    deck = json.dumps(dk)
    sim = chiml_amd.FDTDField(deck)
    sim.step(steps)
    orc = Oracle(deck)
    orc.step(steps)
    for k in range(len(BOXES)):
        ref = orc.flux(k)
        peak = float(np.max(np.abs(ref)))
        assert peak > 0
        assert float(np.max(np.abs(sim.fluxArr()[k].getFlux() - ref))) <= tol * peak, k
    sim.close()


@pytest.mark.parametrize("unpacked", [False, True])
@pytest.mark.parametrize("nlev", [2, 3, 5, 7, 8])
@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 3, 7), (5, 5, 5)])
def test_density_blocks(cells, nlev, unpacked, monkeypatch):
    """One emitter, part of a block, and a last block that is not full."""
    if unpacked:
        monkeypatch.setenv("CHIML_ML_UNPACKED", "1")
    n, d, steps = 20, 0.02, 60
    dk = decks.empty_deck((n, n, n), d, steps, 4)
    dk["ObjectList"].append(decks.n_level_emitter(nlev, [(c - 0.5) * d for c in cells], (d / 2, d / 2, d / 2), seed=60 + nlev))
    fcen = decks.A_UNIT / 600e-9
    dk["SourceList"].append({"pol": "Ex", "size": [8 * d, 8 * d, 0.0], "loc": [0.0, 0.0, decks._pos(14, n, d)],
                             "PulseList": [decks.gaussian_pulse(fcen, 2.0 * fcen, 3.0, 1e8)]})
    deck = json.dumps(dk)
    sim = chiml_amd.FDTDField(deck)
    sim.step(steps)
    sim.sync()
    orc = Oracle(deck)
    orc.step(steps)
    q = sim.qeArr()[0]
    for j in range(2):
        po, pg = orc.pops(0, j), q.population(j)
        assert pg.shape == po.shape
        assert float(np.max(np.abs(pg - po))) <= 1e-10 * max(float(np.max(np.abs(po))), 1.0)
    peak = max(float(np.max(np.abs(orc.field(c)))) for c in range(3))
    for c in range(3):
        assert float(np.max(np.abs(sim.field(c) - orc.field(c)))) <= 1e-9 * peak, c
    sim.close()
