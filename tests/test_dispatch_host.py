"""Host-side choices of the device layer (which kernels a call launches, with
what shared memory, and what happens when memory runs out), seen on the CPU:
a stand-in for the HIP runtime (tests/c/fake_hip.cpp) records the calls that
libchiml_amd.so makes.  Each test runs in a process of its own, since the
stand-in has to be loaded before the library."""
import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, json, re, sys
fake = ctypes.CDLL({fake!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_hip_log.restype = ctypes.c_char_p
fake.fake_hip_fail_size.argtypes = [ctypes.c_size_t]
fake.fake_hip_held.restype = ctypes.c_size_t
import chiml_amd
from chiml_amd import decks

def deck2(n, prec, poles=0, steps=400, pml=8, flux=False):
    d = 0.05
    dk = decks.empty_deck((n[0], n[1], 1), d, steps, pml, precision=prec)
    dk["ObjectList"].append({{"shape": "cylinder", "material": "custom", "eps": 2.5, "pols": decks.gold_like_pols()[:poles],
                             "radius": 5.3 * d, "length": 1.0, "loc": [0.0] * 3, "Basis_Set": [],
                             "unit_vectors": [{{"uvec": [1, 0, 0]}}, {{"uvec": [0, 0, 1]}}, {{"uvec": [0, 1, 0]}}]}})
    dk["SourceList"].append({{"pol": "Ez", "size": [0.0] * 3, "loc": [0.0] * 3, "PulseList": [decks.gaussian_pulse(0.2, 0.2, 3.0, 1.0)]}})
    if flux:
        dk["FluxList"].append({{"name": "f", "size": [20 * d, 20 * d, 0.0], "loc": [0.0] * 3, "lamL": 2.0, "lamR": 9.0, "nfreq": 3}})
    return json.dumps(dk)

def log():
    out = fake.fake_hip_log().decode().split("\\n")[:-1]
    fake.fake_hip_clear()
    return [line.split() for line in out]

def kernels(lines):
    # the launched kernels by their short names, the step counter's left out
    names = [re.search("k_[a-z0-9_]+", line[1]).group() for line in lines if line[0] in ("launch", "capture")]
    return [k for k in names if not k.startswith("k_set_step")]
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    gxx = shutil.which("g++")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if not gxx or not os.path.exists(os.path.join(rocm, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("needs g++ and the HIP headers")
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.check_call([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                           "-o", so, os.path.join(ROOT, "tests", "c", "fake_hip.cpp")])
    return so


def run(fake, body):
    """Runs body after PRELUDE; what it prints last is JSON."""
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(fake=fake) + body], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.strip().split("\n")[-1])


def test_tile_lds_limit_outlives_a_smaller_deck(fake):
    """A kernel's limit of dynamic LDS belongs to the process: a deck with
    fewer poles must not lower it below what a live one launches with."""
    lines = run(fake, """
a = chiml_amd.FDTDField(deck2((64, 64), "fp32", poles=3))
b = chiml_amd.FDTDField(deck2((64, 64), "fp32", poles=1))
for sim in (a, b, a):
    sim.step(8)
print(json.dumps(log()))
""")
    limit, tiles = {}, 0
    for line in lines:
        if line[0] == "attribute":
            limit[line[1]] = int(line[2])
        elif line[0] == "launch" and "k_tile2" in line[1]:
            tiles += 1
            assert int(line[4]) <= limit[line[1]]
    assert tiles == 3


def test_detector_cell_past_the_grid(fake, tmp_path):
    """A detector cell outside a 2D grid is never sampled; the tables of the
    tiles must not be written for it."""
    exe, lib = str(tmp_path / "far_detector"), os.path.join(ROOT, "chiml_amd", "libchiml_amd.so")
    subprocess.check_call(["gcc", "-std=c99", "-I", os.path.join(ROOT, "include"), "-o", exe, os.path.join(ROOT, "tests", "c", "far_detector.c"),
                           "-Wl,--no-as-needed", fake, lib, "-Wl,-rpath," + os.path.dirname(lib), "-Wl,--unresolved-symbols=ignore-in-shared-libs"])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", (r.returncode, r.stdout, r.stderr)


@pytest.mark.parametrize("prec,word", [("fp32", 4), ("fp64", 8)])
def test_no_memory_for_a_second_set_of_fields(fake, prec, word):
    """A 2D deck whose second set of fields does not fit runs on the sweeps,
    which need one set, and holds no part of the second."""
    out = run(fake, f"""
fake.fake_hip_fail_size(68 * 61 * {word})  # the second set's fields: the first set's three are one allocation
a = chiml_amd.FDTDField(deck2((68, 61), "{prec}", poles=1))
refused = [line for line in log() if line[0] == "refused"]
a.step(3)
k = kernels(log())
fake.fake_hip_fail_size(0)
b = chiml_amd.FDTDField(deck2((68, 61), "{prec}", poles=1))
log()
b.step(3)
print(json.dumps([len(refused), k, kernels(log()), a.footprint(), b.footprint(), float(abs(a.field(2)).max())]))
""")
    refused, sweeps, tiles, one, two, _ = out
    assert refused == 1
    assert sweeps == ["k_h2v", "k_e2v"] * 3
    assert tiles == ["k_tile2"]
    assert one < two


def test_field_step_timing_counts_the_steps(fake):
    """profile_only("field_step") times the field update of every step, in
    whatever number of launches the steps are taken."""
    got = run(fake, """
out = []
for flux in (False, True):
    sim = chiml_amd.FDTDField(deck2((68, 61), "fp32", flux=flux))
    sim.profile_only("field_step")
    sim.step(20)
    sim.step(1)
    ms, n = sim.profile_read("field_step")
    out.append([ms > 0, n])
print(json.dumps(out))
""")
    assert got == [[True, 21], [True, 21]]


# n, steps of one call, tiles? -- both sides of each line of tile_pays
SHORT = {"fp32": [(388, 1, True), (412, 1, False), (412, 2, True), (1988, 2, True), (2012, 2, False), (2012, 3, True)],
         "fp64": [(388, 1, True), (412, 1, False), (412, 2, True), (788, 2, True), (812, 2, False), (812, 3, True)]}
GRAPH = {"fp32": [(388, 2, True), (412, 2, False), (988, 4, True), (1012, 4, False), (1012, 6, True)],
         "fp64": [(388, 2, True), (412, 2, False), (608, 4, True), (632, 4, False), (632, 6, True)]}


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_short_calls_on_large_2d_grids_take_the_sweeps(fake, prec):
    """One or two steps (or a graph of 2 or 4) of a large 2D grid go through
    the sweeps, in place; from three steps a launch on, tiles."""
    got = run(fake, f"""
out = []
for n, k, _ in {SHORT[prec]}:
    sim = chiml_amd.FDTDField(deck2((n, n), "{prec}"))
    log()
    sim.step(k)
    out.append(kernels(log()))
for n, k, _ in {GRAPH[prec]}:
    sim = chiml_amd.FDTDField(deck2((n, n), "{prec}"))
    sim.set_graph(k)
    log()
    sim.step(k)
    sim.step(k)
    lines = log()
    assert [line[0] for line in lines].count("graph") == 2
    out.append(kernels([line for line in lines if line[0] == "capture"]))
print(json.dumps(out))
""")
    for (n, k, tiles), names in zip(SHORT[prec], got):
        assert names == (["k_tile2"] if tiles else ["k_h2v", "k_e2v"] * k), (n, k)
    for (n, k, tiles), names in zip(GRAPH[prec], got[len(SHORT[prec]):]):
        assert names == (["k_tile2"] * 2 if tiles else ["k_h2v", "k_e2v"] * k), (n, k)


def test_changing_graphs_of_a_tiled_deck(fake):
    """Graphs of tiles and of sweeps in one run: each replay starts on the
    buffers it was captured on, and a graph of sweeps on its counter slot."""
    lines = run(fake, """
sim = chiml_amd.FDTDField(deck2((432, 432), "fp32"))
log()
sim.set_graph(2)    # sweeps
sim.step(5)         # two replays and a step
sim.step(4)         # a step (the replays start on the other counter slot), a replay and a step
sim.set_graph(16)   # tiles
sim.step(19)        # a replay, then three steps to the other buffers
sim.step(16)
print(json.dumps([line[:2] for line in log() if "k_set_step" not in line[1]]))
""")
    seen = [(a, b.split("k_", 1)[1].split("I", 1)[0] if "k_" in b else b) for a, b in lines]
    sweep, captured = [("launch", "h2v"), ("launch", "e2v")], [("capture", "h2v"), ("capture", "e2v")]
    tile = [("capture", "tile2")] * 2
    assert seen == (captured * 2 + [("graph", "1")] * 2 + sweep + sweep + [("graph", "1")] + sweep
                    + tile + [("graph", "2"), ("launch", "tile2")] + tile + [("graph", "3")])


@pytest.mark.parametrize("prec,w", [("fp32", 4), ("fp64", 2)])
def test_2d_sweeps_fuse_products_on_unaligned_grids_only(fake, prec, w):
    """The E sweep's fused form (rows or x CPML of no whole groups) is an
    instantiation of its own: on the others it cost registers and a wave."""
    names = run(fake, f"""
out = []
for n, pml in (((1024, 900), 8), ((1025, 900), 8), ((1024, 900), 9)):
    sim = chiml_amd.FDTDField(deck2(n, "{prec}", pml=pml, flux=True))
    log()
    sim.step(1)
    out.append([line[1] for line in log() if "k_e2v" in line[1]])
print(json.dumps(out))
""")
    kind = "d" if prec == "fp64" else "f"
    want = [f"k_e2vI{kind}Li{w}ELb1ELb0ELb{fma}E" for fma in (0, 1, 1)]
    assert all(len(n) == 1 and k in n[0] for n, k in zip(names, want)), names


def test_small_unaligned_2d_grids_step_per_cell(fake):
    """FP32, below the line of GridLayout::cellwise and with a source; a batch
    takes the groups all the same."""
    got = run(fake, """
out = []
for n, prec in (((257, 255), "fp32"), ((701, 699), "fp32"), ((260, 255), "fp32"), ((257, 255), "fp64")):
    a, b = (chiml_amd.FDTDField(deck2(n, prec, flux=True)) for _ in range(2))
    log()
    a.step(1)
    alone = kernels(log())
    chiml_amd.step_batch([a, b], 1)
    out.append([alone, kernels(log())])
print(json.dumps(out))
""")
    cells, groups = ["k_update_h", "k_update_e", "k_sample"], ["k_h2v", "k_e2v", "k_sample"]
    assert [g[0] for g in got] == [cells, groups, groups, groups]
    assert all(g[1][:3] == ["k_bh2v", "k_be2v", "k_bsample"] for g in got)


def test_padded_row_decks_take_the_kernels_they_are_for(fake):
    """The decks that test_gpu_padded_rows.py compares with the oracle."""
    sys.path.insert(0, ROOT)
    from tests.route_decks import CASES
    got = run(fake, """
from tests.route_decks import CASES
out = {}
for name, (deck, _, _) in CASES.items():
    sim = chiml_amd.FDTDField(deck)
    log()
    sim.step(1)
    out[name] = [line[1] for line in log()]
    sim.close()
print(json.dumps(out))
""")
    for name, (_, _, kernels) in CASES.items():
        for k in kernels:
            assert any(k in line for line in got[name]), (name, k, got[name])


def test_no_memory_for_the_flux_tables(fake):
    """A flux spectrum is read on the host where the card has no room for the
    faces' tables; what was taken of them is given back."""
    got = run(fake, """
import numpy as np
sim = chiml_amd.FDTDField(deck2((68, 61), "fp64", flux=True))
sim.step(4)
held, out = fake.fake_hip_held(), []
for n in (1, 2, 3):
    fake.fake_hip_refuse(n)
    f = sim.fluxArr()[0].getFlux()
    fake.fake_hip_refuse(0)
    out.append([f.size, fake.fake_hip_held() == held, [k for k in kernels(log()) if "flux" in k]])
f = sim.fluxArr()[0].getFlux()
out.append([f.size, fake.fake_hip_held() > held, [k for k in kernels(log()) if "flux" in k]])
print(json.dumps(out))
""")
    assert got == [[3, True, []]] * 3 + [[3, True, ["k_flux_faces"]]]
