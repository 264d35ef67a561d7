"""Calls whose kernels depend on more than the deck -- several live contexts,
step counts, batches -- against the same deck stepped alone, bit for bit, or
against the FP64 oracle."""
import json

import numpy as np
import pytest

import chiml_amd
from chiml_amd import decks
from tests.route_decks import emitters, metal

pytestmark = pytest.mark.gpu


def _deck2(n, prec, poles=0, pml=8, steps=200, flux=False):
    d = 0.05
    dk = decks.empty_deck((n[0], n[1], 1), d, steps, pml, precision=prec)
    r = (min(n) - 2 * pml) / 4.0 + 0.3
    dk["ObjectList"].append({"shape": "cylinder", "material": "custom", "eps": 2.5, "pols": decks.gold_like_pols()[:poles], "radius": r * d,
                             "length": 1.0, "loc": [0.2 * d, -0.3 * d, 0.0], "Basis_Set": [],
                             "unit_vectors": [{"uvec": [1, 0, 0]}, {"uvec": [0, 0, 1]}, {"uvec": [0, 1, 0]}]})
    for pol, x, y in (("Ez", n[0] // 2 + 2, n[1] // 2), ("Hx", pml + 1, n[1] // 2 - 3)):
        pulse = decks.gaussian_pulse(0.3, 1.0, 3.0, 1.0)
        pulse["t_0"] = 0.1
        dk["SourceList"].append({"pol": pol, "size": [0.0] * 3, "loc": [decks._pos(x, n[0], d), decks._pos(y, n[1], d), 0.0], "PulseList": [pulse]})
    dk["DetectorList"].append({"type": "Ez", "dtc_class": "cout", "fname": "d", "size": [0.0] * 3,
                               "loc": [decks._pos(n[0] // 2 - 4, n[0], d), decks._pos(n[1] // 2 + 5, n[1], d), 0.0]})
    if flux:
        dk["FluxList"].append({"name": "flux", "size": [(n[0] // 2) * d, (n[1] // 2) * d, 0.0], "loc": [0.0] * 3, "lamL": 2.0, "lamR": 9.0,
                               "nfreq": 4})
    return json.dumps(dk)


def _results(sim):
    sim.sync()
    r = {f"f{c}": sim.field(c) for c in range(6)}
    r.update({f"d{k}": d.series()[1] for k, d in enumerate(sim.dtcArr())})
    r.update({f"x{k}": f.getFlux() for k, f in enumerate(sim.fluxArr())})
    return r


def _same(a, b, label):
    assert a.keys() == b.keys(), label
    assert np.max(np.abs(a["f2"])) > 0, label
    for k in a:
        assert np.array_equal(a[k], b[k]), (label, k, float(np.max(np.abs(a[k] - b[k]))))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_live_decks_of_different_pole_counts(prec):
    """One tile shape, three pole counts alive at once, stepped in turn."""
    sims = [chiml_amd.FDTDField(_deck2((64, 60), prec, poles=p)) for p in (3, 1, 2)]
    for _ in range(3):
        for sim in sims:
            sim.step(20)
    for p, sim in zip((3, 1, 2), sims):
        alone = chiml_amd.FDTDField(_deck2((64, 60), prec, poles=p))
        alone.step(60)
        _same(_results(alone), _results(sim), p)
        alone.close()
        sim.close()


@pytest.mark.parametrize("prec,n", [("fp32", (836, 828)), ("fp32", (831, 829)), ("fp32", (431, 429)), ("fp64", (412, 404)), ("fp64", (407, 405))])
def test_results_do_not_depend_on_the_calls(prec, n):
    """Above the sizes at which one or two steps go through the sweeps: whole
    runs, single steps between tiles, and graphs of either kind."""
    deck = _deck2(n, prec, poles=2, pml=7, steps=60)
    whole = chiml_amd.FDTDField(deck)
    whole.step(53)
    ref = _results(whole)
    whole.close()
    runs = {"pieces": [(0, (1, 1, 2, 1, 3, 1, 8, 1, 2, 9, 1, 1, 22))],
            "graphs": [(2, (1, 2, 4, 3)), (4, (4, 1, 4, 2)), (8, (8, 1, 8)), (2, (2, 1, 2)), (0, (1, 7, 2))],
            "graph4": [(4, (53,))],
            # graphs of sweeps captured and replayed on either buffer set
            "flipped": [(0, (3,)), (2, (4, 3)), (0, (7,)), (2, (6, 1)), (8, (8, 8)), (2, (2,)), (0, (3, 8))]}
    for label, plan in runs.items():
        sim = chiml_amd.FDTDField(deck)
        for graph, chunks in plan:
            sim.set_graph(graph)
            for k in chunks:
                sim.step(k)
        assert sum(sum(c) for _, c in plan) == 53
        _same(ref, _results(sim), label)
        sim.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [(45, 41), (131, 70), (257, 255)])
def test_batched_odd_flux_decks_equal_alone(n, prec):
    """2D decks that no tile takes, of sizes that are no whole groups: alone in
    one thread per cell (FP32) or in groups, batched in groups."""
    mix = [_deck2(n, prec, poles=2, pml=7, flux=True), _deck2((n[0] + 1, n[1] + 2), prec, poles=1, flux=True),
           _deck2((n[0] + 3, n[1]), prec, flux=True)]
    sims = [chiml_amd.FDTDField(d) for d in mix]
    for k in (1, 40, 7, 32):
        chiml_amd.step_batch(sims, k)
    for k, (deck, sim) in enumerate(zip(mix, sims)):
        alone = chiml_amd.FDTDField(deck)
        alone.step(80)
        _same(_results(alone), _results(sim), k)
        alone.close()
        sim.close()


def test_batched_unaligned_3d_decks_equal_alone():
    """3D metals whose rows are no whole groups: FP32 ones in groups when
    batched, alone in one thread per cell below the line and in groups above
    it; FP64 ones step alone inside the call.  One aligned deck of each
    precision and one with emitters share the launches."""
    mix = [metal((33, 30, 31), 5, "fp32", 60), metal((66, 60, 60), 7, "fp32", 60), metal((33, 30, 31), 5, "fp64", 60),
           metal((65, 62, 61), 5, "fp64", 60), metal((64, 60, 60), 8, "fp32", 60), metal((64, 60, 60), 8, "fp64", 60),
           emitters((66, 60, 60), 7, "fp32", 60, (5, 7, 3), 4), emitters((613, 615, 1), 7, "fp32", 60, (9, 5, 1), 2),
           emitters((91, 93, 1), 7, "fp64", 60, (9, 5, 1), 3)]
    sims = [chiml_amd.FDTDField(d) for d in mix]
    for k in (7, 13, 1, 20, 19):
        chiml_amd.step_batch(sims, k)
    for k, (deck, sim) in enumerate(zip(mix, sims)):
        alone = chiml_amd.FDTDField(deck)
        alone.step(60)
        a, b = _results(alone), _results(sim)
        _same(a, b, k)
        for q, p in zip(alone.qeArr(), sim.qeArr()):
            assert np.array_equal(q.population(0), p.population(0)), k
        alone.close()
        sim.close()
