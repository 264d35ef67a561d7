"""Decks whose grid takes a padded or widened layout, with the kernels that
step them: rows or x CPML that are no whole groups (4 cells in FP32, 2 in
FP64), above the sizes that step one thread per cell.  The kernels are checked
on the CPU (test_dispatch_host.py), the results against the oracle
(test_gpu_padded_rows.py).  Also 2D decks that the tiles leave to the sweeps."""
import json

from chiml_amd import decks

BITS = {"fp32": ("f", 4), "fp64": ("d", 2)}


def _h3(prec, src=1, nt=0):
    """Kernels of the whole-row 3D sweeps."""
    t, w = BITS[prec]
    return [f"k_h3_allI{t}Li{w}ELb{src}ELb0ELb1ELb{nt}E", f"k_e3_allI{t}Li{w}ELb{src}ELb1ELb{nt}E"]


def _h2(prec, src=1, det=0):
    """Kernels of the 2D sweeps (det: the E sweep takes the point detectors)."""
    t, w = BITS[prec]
    return [f"k_h2vI{t}Li{w}ELb{src}ELb0E", f"k_e2vI{t}Li{w}ELb{src}ELb{det}ELb1E"]


def _pulse(peak=1.0):
    p = decks.gaussian_pulse(0.3, 1.0, 3.0, peak)
    p["t_0"] = 0.1
    return p


def _point(n, d, cell):
    return [decks._pos(c, m, d) if m > 1 else 0.0 for c, m in zip(cell, n)]


def _add_common(dk, n, d, pml):
    """Soft sources in the CPML slabs and in the last cells of a row, point
    detectors there, and a flux box."""
    three = n[2] > 1
    mid = [m // 2 for m in n]
    last = n[0] - 2
    src = [("Ez", (mid[0] + 2, mid[1], mid[2])), ("Hx", (mid[0], 1 if pml else 3, mid[2])), ("Hy", (last, mid[1] + 1, mid[2]))]
    if three:
        src += [("Ex", (mid[0] - 1, mid[1], 1 if pml else 3)), ("Ey", (1, mid[1] - 2, mid[2])), ("Hz", (mid[0] + 3, mid[1] - 1, mid[2]))]
    for pol, cell in src:
        dk["SourceList"].append({"pol": pol, "size": [0.0] * 3, "loc": _point(n, d, cell), "PulseList": [_pulse()]})
    for t in ("Ez", "Hy"):
        dk["DetectorList"].append({"type": t, "dtc_class": "cout", "fname": "d", "size": [0.0] * 3, "loc": _point(n, d, (last, mid[1] + 1, mid[2]))})
    fs = [(m // 3) * d if m > 1 else 0.0 for m in n]
    dk["FluxList"].append({"name": "flux", "size": fs, "loc": [0.0] * 3, "lamL": 2.0, "lamR": 9.0, "nfreq": 4})


def _metal(n, d, pml):
    """A metal from right of the middle out through the last cells of a row
    (in 2D, where a CPML may hold none, to the CPML)."""
    three = n[2] > 1
    lo, hi = n[0] // 2 + 5, n[0] + 3 if three or pml == 0 else n[0] - pml - 2
    size = [(hi - lo) * d, (n[1] // 3) * d, (n[2] // 3) * d if three else 0.0]
    loc = [decks._pos(lo, n[0], d) + size[0] / 2.0 + 0.01 * d, 0.3 * d, 0.2 * d if three else 0.0]
    return {"shape": "block", "material": "custom", "eps": 1.5, "pols": decks.gold_like_pols(), "size": size, "loc": loc, "Basis_Set": []}


def metal(n, pml, prec, steps):
    d = 0.02 if n[2] > 1 else 0.05
    dk = decks.empty_deck(n, d, steps, pml, precision=prec)
    if n[2] > 1:  # metal inside a CPML needs a dielectric there
        dk["ObjectList"].append({"shape": "block", "material": "custom", "eps": 2.25, "eps_diag": [2.0, 2.25, 2.5], "pols": [],
                                 "size": [(m + 3) * d for m in n], "loc": [0.0] * 3, "Basis_Set": []})
    dk["ObjectList"].append(_metal(n, d, pml))
    _add_common(dk, n, d, pml)
    return json.dumps(dk)


def emitters(n, pml, prec, steps, cells, levels):
    d = 0.02 if n[2] > 1 else 0.05
    dk = decks.empty_deck(n, d, steps, pml, precision=prec)
    size = [(c - 0.5) * d if m > 1 else 0.0 for c, m in zip(cells, n)]
    dk["ObjectList"].append(decks.n_level_emitter(levels, size, tuple(d / 2 if m % 2 == 0 else 0.0 for m in n), seed=70 + levels))
    _add_common(dk, n, d, pml)
    for s in dk["SourceList"]:
        s["PulseList"] = [_pulse(1e8)]
    return json.dumps(dk)


def tfsf(n, pml, prec, steps, box, m):
    d = 0.02 if n[2] > 1 else 0.05
    # scatters out of the box to the ends of the rows
    ob = {"shape": "sphere" if n[2] > 1 else "cylinder", "material": "custom", "eps": 3.0, "pols": decks.gold_like_pols(), "radius": 6.2 * d,
          "length": 1.0, "loc": [0.3 * d, -0.2 * d, 0.0], "Basis_Set": [],
          "unit_vectors": [{"uvec": [1, 0, 0]}, {"uvec": [0, 0, 1]}, {"uvec": [0, 1, 0]}]}
    return decks.tfsf_deck(n, steps, box, m=m, psi=50.0, pml=pml, d=d, precision=prec, ndet=4, objects=[ob])


def oblique(n, pml, prec, steps):
    d = 0.05
    dk = decks.empty_deck(n, d, steps, pml, precision=prec)
    for pol, x, phi in (("Hx", -6, 30.0), ("Hy", 5, 200.0)):
        dk["SourceList"].append({"pol": pol, "size": [8 * d, 4 * d, 0.0], "loc": [x * d, 3 * d, 0.0], "phi": phi, "PulseList": [_pulse()]})
    return json.dumps(dk)


def no_tiles(n, pml, prec, steps, points, sets):
    """A 2D deck without a flux box that the tiles leave to the sweeps: points x
    points detector cells in one tile, or so many metals of different poles."""
    d = 0.05
    dk = decks.empty_deck(n, d, steps, pml, precision=prec)
    for k in range(sets):
        pols = [dict(p, gamma=p["gamma"] * (1.0 + 0.1 * k)) for p in decks.gold_like_pols()[:1]]
        dk["ObjectList"].append({"shape": "block", "material": "custom", "eps": 2.0, "pols": pols, "size": [1.6 * d, 9.6 * d, 0.0],
                                 "loc": [(2 * k - sets) * d, 0.0, 0.0], "Basis_Set": []})
    dk["SourceList"].append({"pol": "Ez", "size": [0.0] * 3, "loc": _point(n, d, (n[0] // 2 + 1, n[1] // 2 + 6, 0)), "PulseList": [_pulse()]})
    dk["DetectorList"].append({"type": "Ez", "dtc_class": "cout", "fname": "d", "size": [(points - 1) * d, (points - 1) * d, 0.0],
                               "loc": [decks._pos(17, n[0], d) + (points - 1) * d / 2.0, decks._pos(17, n[1], d) + (points - 1) * d / 2.0, 0.0]})
    return json.dumps(dk)


# name -> (deck, steps, kernels)
CASES = {
    "metal_fp32": (metal((66, 60, 60), 7, "fp32", 40), 40, _h3("fp32")),
    "metal_fp64": (metal((65, 62, 61), 5, "fp64", 40), 40, _h3("fp64")),
    "metal_67_fp32": (metal((67, 61, 60), 8, "fp32", 40), 40, _h3("fp32")),
    "wide_cpml_fp32": (metal((68, 60, 61), 6, "fp32", 40), 40, _h3("fp32")),  # whole rows, x CPML of no whole groups
    "wide_cpml_fp64": (metal((66, 60, 61), 7, "fp64", 40), 40, _h3("fp64")),
    "no_cpml_fp32": (metal((69, 60, 60), 0, "fp32", 40), 40, _h3("fp32")),
    "no_cpml_fp64": (metal((65, 60, 60), 0, "fp64", 40), 40, _h3("fp64")),
    "streamed_fp32": (metal((201, 197, 198), 9, "fp32", 12), 12, _h3("fp32", nt=1)),
    "streamed_fp64": (metal((159, 157, 157), 6, "fp64", 12), 12, _h3("fp64", nt=1)),
    "emitters_fp32": (emitters((66, 60, 60), 7, "fp32", 40, (5, 7, 3), 4), 40, _h3("fp32") + ["k_ml_entryIfLi4E"]),
    "emitters_fp64": (emitters((65, 62, 61), 5, "fp64", 40, (5, 3, 7), 3), 40, _h3("fp64") + ["k_ml_entryIdLi3E"]),
    "tfsf_fp32": (tfsf((66, 60, 62), 7, "fp32", 60, (31, 29, 31), (0, 0, 1)), 60, _h3("fp32", src=0) + ["k_tfsf_stepIf"]),
    "tfsf_fp64": (tfsf((65, 62, 61), 5, "fp64", 60, (31, 33, 29), (1, 1, 1)), 60, _h3("fp64", src=0) + ["k_tfsf_stepId"]),
    "metal_2d_fp32": (metal((621, 613, 1), 9, "fp32", 60), 60, _h2("fp32")),
    "metal_2d_fp64": (metal((101, 93, 1), 9, "fp64", 60), 60, _h2("fp64")),
    "no_cpml_2d_fp64": (metal((103, 93, 1), 0, "fp64", 60), 60, _h2("fp64")),
    "no_cpml_2d_fp32": (metal((615, 613, 1), 0, "fp32", 60), 60, _h2("fp32")),
    "metal_2d_small_fp32": (metal((101, 93, 1), 9, "fp32", 60), 60, ["k_update_hIfLi2E", "k_update_eIfLi2E"]),
    "emitters_2d_fp32": (emitters((613, 615, 1), 7, "fp32", 60, (9, 5, 1), 2), 60, _h2("fp32") + ["k_ml_entryIfLi2E"]),
    "emitters_2d_fp64": (emitters((91, 93, 1), 7, "fp64", 60, (9, 5, 1), 3), 60, _h2("fp64") + ["k_ml_entryIdLi3E"]),
    "tfsf_2d_fp32": (tfsf((101, 94, 1), 7, "fp32", 90, (41, 39, 1), (0, 1, 0)), 90, _h2("fp32", src=0, det=1) + ["k_tfsf_stepIf"]),
    "tfsf_2d_fp64": (tfsf((101, 94, 1), 7, "fp64", 90, (41, 39, 1), (1, 2, 0)), 90, _h2("fp64", src=0, det=1) + ["k_tfsf_stepId"]),
    "oblique_2d_fp32": (oblique((101, 94, 1), 7, "fp32", 60), 60, _h2("fp32", src=0) + ["k_cell_srcIf"]),
    "many_points_2d_fp64": (no_tiles((48, 44, 1), 4, "fp64", 60, 9, 1), 60, ["k_h2vIdLi2ELb1ELb0E", "k_e2vIdLi2ELb1ELb0ELb0E"]),
    "many_points_2d_fp32": (no_tiles((48, 44, 1), 4, "fp32", 60, 9, 1), 60, ["k_h2vIfLi4ELb1ELb0E", "k_e2vIfLi4ELb1ELb0ELb0E"]),
    "many_poles_2d_fp64": (no_tiles((48, 44, 1), 4, "fp64", 60, 1, 9), 60, ["k_h2vIdLi2ELb1ELb0E", "k_e2vIdLi2ELb1ELb1ELb0E"]),
    "many_poles_2d_fp32": (no_tiles((48, 44, 1), 4, "fp32", 60, 1, 9), 60, ["k_h2vIfLi4ELb1ELb0E", "k_e2vIfLi4ELb1ELb1ELb0E"]),
    "oblique_2d_fp64": (oblique((101, 94, 1), 7, "fp64", 60), 60, _h2("fp64", src=0) + ["k_cell_srcId"]),
}
