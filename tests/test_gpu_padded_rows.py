"""Padded rows and widened x CPML above the sizes that step one thread per
cell: the whole-row 3D sweeps in both precisions, with and without the
streaming hint, the 2D sweeps, and the emitter, TFSF and per-cell source
kernels on rows whose stored length is not nx.  Against the FP64 oracle, to
1e-9 (FP64) and 1e-5 (FP32) of each family's peak, as the aligned grids are."""
import numpy as np
import pytest

import chiml_amd
from oracle.pyoracle import Oracle
from tests.route_decks import CASES

pytestmark = pytest.mark.gpu

TOL = {64: 1e-9, 32: 1e-5}


def _err(a, r, scale):
    return float(np.max(np.abs(np.asarray(a) - np.asarray(r)))) / scale


@pytest.mark.parametrize("name", list(CASES))
def test_padded_rows(name):
    deck, steps, _ = CASES[name]
    sim, orc = chiml_amd.FDTDField(deck), Oracle(deck)
    sim.step(steps)
    sim.sync()
    orc.step(steps)
    tol = TOL[sim.precision]
    comps = range(6) if sim.shape[0] > 1 else (2, 3, 4)
    peaks = []
    for fam in ([c for c in comps if c < 3], [c for c in comps if c > 2]):
        ref = [orc.field(c) for c in fam]
        peaks.append(max(float(np.max(np.abs(r))) for r in ref))
        assert peaks[-1] > 0
        for c, r in zip(fam, ref):
            err = _err(sim.field(c), r, peaks[-1])
            print(f"{name} field {c}: {err:.2e}", flush=True)
            assert err <= tol, c
    for k, det in enumerate(sim.dtcArr()):
        r = np.asarray(orc.detector(k)[1])
        scale = max(float(np.max(np.abs(r))), *peaks)
        assert _err(det.series()[1].ravel(), r.ravel(), scale) <= tol, k
    for k, f in enumerate(sim.fluxArr()):
        r, got = orc.flux(k), f.getFlux()
        peak = float(np.max(np.abs(r)))
        if peak == 0:  # the waves of a large grid have not reached the box
            assert not np.any(got), k
        else:  # a sum of products of two fields, faces of both signs
            assert _err(got, r, peak) <= 10 * tol, k
    for k, q in enumerate(sim.qeArr()):
        for j in range(2):
            r = orc.pops(k, j)
            assert _err(q.population(j), r, 1.0) <= (1e-10 if sim.precision == 64 else tol), (k, j)
    sim.close()
