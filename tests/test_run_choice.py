"""Invariants of the rule that picks a SOAP run's kernel and decomposition
(csrc/soap_choice.h), over random plans and batches, on the host."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest

import run_choice

SLICE = 256 << 20
FASTEST, LONG_RUNS, SHORT_ROWS, LEAST = range(4)


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    return run_choice.compiled(tmp_path_factory.mktemp("run_choice"))


def _molecules(count, atoms):
    return SimpleNamespace(offsets=np.arange(count + 1) * atoms, pbc=np.zeros((count, 3)), cells=np.zeros((count, 3, 3)))


def _random(rng):
    options = {}
    if rng.random() < 0.4:
        options["weighting"] = {"w0": 0.5}
    if rng.random() < 0.5:
        options["compression"] = str(rng.choice(["mu2", "mu1nu1", "crossover"]))
    if rng.random() < 0.4:
        options["polynomial"] = True
    plan = run_choice.plan_values(int(rng.integers(1, 9)), int(rng.integers(1, 13)), int(rng.integers(0, 12)),
                                  str(rng.choice(["off", "inner", "outer"])), str(rng.choice(["float32", "float64"])), options)
    structures = int(np.exp(rng.uniform(0, np.log(5000))))
    largest = int(np.exp(rng.uniform(0, np.log(30000))))
    atoms = largest + int((structures - 1) * rng.uniform(0.1, 1.0) * min(largest, 200))
    images = largest * int(rng.choice([1, 27, 125]))
    rows = int(min(images, rng.choice([512, 278, 670, 5000])))
    return {**plan, "structures": structures, "atoms": atoms, "largest_structure": largest, "most_images": images,
            "row_bound": max(1, rows), "units": 256, "budget": int(rng.choice([0, 1 << 20, 50 << 20, 1 << 30]))}


def test_one_mode_within_its_limits(rule):
    rng = np.random.default_rng(0)
    seen = set()
    for _ in range(20000):
        v = _random(rng)
        for saving in range(4):
            c = run_choice.evaluate(rule, v, saving)
            modes = [c["block_inner"], c["block_runs"], c["block_outer"], c["block_outer_lds"], c["quad"]]
            assert sum(modes) <= 1 and c["block"] >= max(modes[:4])
            assert not (c["block"] and c["quad"])
            if c["block"]:
                assert sum(modes[:4]) == (v["average"] != 0) and v["block_waves"] > 0
            if c["block_small"]:
                assert c["block_inner"] and v["largest_structure"] <= 64 and not v["radial_basis"]
            if c["block_outer_lds"]:
                assert v["features"] * 8 <= 48 * 1024 and not v["radial_basis"]
            if c["block_outer"]:
                assert v["atoms"] * v["features"] * 8 <= 1 << 32
            if c["f32_exps"]:
                assert c["block"] and v["block_every_form"] and v["block_float32"]
                assert not (v["weighted"] and v["average"] == 1 and c["block_inner"])
            assert 1 <= c["run"] <= 32
            # radial functions: an item's centres fit a slice, and where nothing
            # may be kept beside the partial rows there are none (nor weights)
            if c["poly_centre"]:
                assert v["radial_basis"] and not c["poly_inside"]
                item = (v["largest_structure"] if c["block_inner"] else
                        c["run"] if v["average"] and not c["block_outer"] else 1)
                assert item == 1 or item * c["poly_centre"] * 8 <= SLICE
            if saving == LEAST and (v["weighted"] or v["radial_basis"]):
                assert not c["block"] and c["poly_least"] == 0
            if saving >= SHORT_ROWS:
                assert not c["block_runs"] and not c["block_outer"]
            if saving >= LONG_RUNS and v["average"] and not c["block_inner"] and not c["block_outer"] and not c["poly_centre"]:
                assert c["run"] == 32
            seen.add(tuple(modes))
    assert len(seen) == 6


@pytest.mark.parametrize("shape,average,structures,atoms,expected", [
    ((3, 8, 7), "inner", 4, 20, "species-major structures"), ((3, 8, 7), "inner", 4, 70, "runs"),
    ((3, 8, 7), "inner", 1100, 70, "whole structures"), ((3, 8, 7), "outer", 4, 20, "centre rows"),
    ((3, 8, 7), "outer", 600, 20, "rows in LDS"), ((5, 2, 6), "off", 600, 20, "tile kernel"),
    ((5, 2, 6), "off", 600, 70, "rows"), ((4, 9, 4), "outer", 600, 20, "tile kernel"),
    ((2, 13, 4), "off", 600, 20, "tile kernel"), ((9, 4, 4), "off", 600, 20, "tile kernel"),
    # rows in LDS of too few structures, whose centre rows do not fit either
    ((2, 12, 7), "outer", 150, 50, "tile kernel"), ((2, 12, 7), "outer", 600, 50, "rows in LDS"),
])
def test_modes(rule, shape, average, structures, atoms, expected):
    plan = run_choice.plan_values(*shape, average)
    assert run_choice.mode(rule, plan, run_choice.batch_values(_molecules(structures, atoms), 4.0)) == expected


def test_small_structures_are_not_split(rule):
    """Molecules of at most a run: one row each, nothing for the finalize to add."""

    plan = run_choice.plan_values(1, 3, 0, "inner", options={"compression": "mu2"})
    molecules = dict(structures=3000, atoms=15000, largest_structure=8, most_images=8, row_bound=16, units=256,
                     budget=50 << 20)
    assert run_choice.evaluate(rule, {**plan, **molecules})["run"] >= 8


@pytest.mark.parametrize("atoms,waves,longest,shortest", [
    (1000, 8, 8, 4), (3000, 8, 16, 16), (6000, 8, 32, 32), (6000, 4, 16, 16), (12000, 4, 32, 32), (40000, 16, 32, 32),
])
def test_runs_of_a_structure_on_the_tile_kernels(rule, atoms, waves, longest, shortest):
    """One structure's centres in runs: short ones fill the device, but the
    finalize walks their rows one after another."""

    plan = run_choice.plan_values(3, 8, 10, "inner")
    plan["quad_waves"] = waves
    cell = dict(structures=1, atoms=atoms, largest_structure=atoms, most_images=27 * atoms, row_bound=512, units=256,
                budget=1 << 30)
    c = run_choice.evaluate(rule, {**plan, **cell})
    assert c["quad"] and shortest <= c["run"] <= longest


def test_runs_that_already_fill_the_device_stay_long(rule):
    plan = run_choice.plan_values(4, 8, 6, "inner")
    for structures, atoms, run in ((500, 85, 32), (200, 130, 32), (60, 130, 3)):
        batch = dict(structures=structures, atoms=structures * atoms, largest_structure=atoms + 30,
                     most_images=atoms + 30, row_bound=160, units=256, budget=1 << 30)
        c = run_choice.evaluate(rule, {**plan, **batch})
        assert c["block_runs"] and c["run"] == run


def test_slices_of_radial_rows_hold_runs_for_the_device(rule):
    """By row: runs short enough that a slice has 2,048 wavefronts of them."""

    plan = run_choice.plan_values(3, 8, 1, "inner", options={"polynomial": True})
    batch = dict(structures=500, atoms=42500, largest_structure=100, most_images=100, row_bound=112, units=256,
                 budget=1 << 30)
    c = run_choice.evaluate(rule, {**plan, **batch})
    assert c["poly_centre"] and not c["block"]
    slice_centres = SLICE // (8 * c["poly_centre"])
    assert slice_centres // c["run"] >= 2048
