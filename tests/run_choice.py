"""The kernel and decomposition a SOAP run takes: csrc/soap_choice.h compiled
for the host, on the sizes a plan and a batch give it."""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import numpy as np

from conftest import ROOT, SOAP_PAD

FIELDS = ("average", "radial_basis", "compression", "weighted", "S", "Sc", "n", "L", "l_max", "features", "use_mfma",
          "tiles", "quad_waves", "block_waves", "block_kg", "block_ncr", "block_forced", "block_float32",
          "block_every_form", "block_width", "quad_width", "tile_width", "structures", "atoms", "largest_structure",
          "most_images", "row_bound", "units", "budget")
RESULTS = ("block", "block_inner", "block_small", "block_runs", "block_outer", "block_outer_lds", "f32_exps", "quad",
           "poly_inside", "run", "partial_width", "poly_centre", "poly_least")

SOURCE = """
#include "soap_choice.h"
extern "C" void choose_run(const int64_t* v, int saving, int64_t* out) {
    mdx::ChoiceInput in;
    int i = 0;
%s
    const mdx::Choice c = mdx::choose(in, saving);
    int o = 0;
%s
}
""" % ("\n".join(f"    in.{f} = static_cast<decltype(in.{f})>(v[i++]);" for f in FIELDS),
       "\n".join(f"    out[o++] = static_cast<int64_t>(c.{f});" for f in RESULTS[:-2])
       + "\n    out[o++] = mdx::poly_layout_of(in, c).centre;\n    out[o++] = static_cast<int64_t>(mdx::poly_least_bytes(in, c));")

EVERY_FORM = {(3, 1, 1), (6, 2, 2), (4, 2, 3), (8, 2, 3), (9, 3, 1)}  # (l_max, radial groups, coefficient registers)
AVERAGES = {"off": 0, "inner": 1, "outer": 2}
COMPRESSIONS = {"off": 0, "mu2": 1, "mu1nu1": 2, "crossover": 3}


def compiled(folder: Path):
    (folder / "choice.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT / 'mdescriptor_amd' / 'csrc'}",
                    str(folder / "choice.cpp"), "-o", str(folder / "choice.so")], check=True)
    return ctypes.CDLL(str(folder / "choice.so"))


def evaluate(lib, values: dict, saving: int = 0) -> dict:
    out = (ctypes.c_int64 * len(RESULTS))()
    lib.choose_run((ctypes.c_int64 * len(FIELDS))(*(int(values[f]) for f in FIELDS)), saving, out)
    return dict(zip(RESULTS, out))


def plan_values(species: int, n: int, l_max: int, average: str, dtype: str = "float64", options: dict | None = None) -> dict:
    """The rule's input of a plan (as mdx_hip_soap_plan_create fills it)."""

    options = options or {}
    compression = COMPRESSIONS[options.get("compression", "off")]
    polynomial = "polynomial" in options
    weighted = bool(options.get("weighting") or options.get("species_weights"))
    coefficient_species = 1 if compression == 1 else species
    groups, degrees, channels = (n + 3) // 4, l_max + 1, coefficient_species * n
    need = coefficient_species if groups == 3 else -(-coefficient_species * groups // 4)
    held = [c for c in {1: (1, 2), 2: (1, 2, 3), 3: (1, 2, 3, 5)}.get(groups, ()) if c >= need]
    block = bool(held) and 2 <= l_max <= 9 and not (polynomial and groups > 2)
    registers = held[0] if block else 0
    every = (l_max, groups, registers) in EVERY_FORM
    float32 = every and dtype == "float32" and not polynomial and (
        (average == "off" and (compression != 2 or not weighted)) or (average == "inner" and compression == 0))
    columns = sum((2 * l + 4) // 4 for l in range(degrees))
    padded = 4 * columns + (4 - 4 * columns) % 32
    features = {0: channels * (channels + 1) // 2, 1: n * (n + 1) // 2, 2: channels * n,
                3: species * n * (n + 1) // 2}[compression] * degrees
    return dict(average=AVERAGES[average], radial_basis=polynomial, compression=compression, weighted=weighted, S=species,
                Sc=coefficient_species, n=n, L=degrees, l_max=l_max, features=features, use_mfma=1,
                tiles=max(1, degrees * n // 16),
                quad_waves=int(n <= 8 and l_max <= 10 and not (polynomial or weighted or compression)),
                block_waves=min(4, degrees) if block else 0, block_kg=groups, block_ncr=registers, block_forced=0,
                block_float32=float32, block_every_form=every, block_width=columns * registers * 64,
                quad_width=(4 * -(-channels // 4) + 1) * padded, tile_width=(channels + n * (compression == 2) + 1) * padded)


def batch_values(batch, r_cut: float, units: int = 256) -> dict:
    """The rule's input of a batch whose search has not been counted yet
    (orthorhombic cells)."""

    sizes = np.diff(batch.offsets)
    images = []
    for s, atoms in enumerate(sizes):
        count = 1
        if np.asarray(batch.pbc[s])[0]:
            for edge in np.diag(batch.cells[s]):
                count *= 2 * int((r_cut + SOAP_PAD) / edge + 1.0) + 1
        images.append(int(atoms) * count)
    most = max(images)
    rows = min(512, max(16, -(-most // 16) * 16))
    atoms = int(sizes.sum())
    return dict(structures=len(sizes), atoms=atoms, largest_structure=int(sizes.max()), most_images=most, row_bound=rows,
                units=units, budget=max(0, int(0.85 * (64 << 20)) - 4 * atoms * rows - 44 * sum(images)))


def mode(lib, plan: dict, batch: dict) -> str:
    """Name of the mode a run takes."""

    c = evaluate(lib, {**plan, **batch})
    if not c["block"]:
        return "tile kernel"
    names = {"block_small": "species-major structures", "block_inner": "whole structures", "block_runs": "runs",
             "block_outer": "centre rows", "block_outer_lds": "rows in LDS"}
    return next((name for key, name in names.items() if c[key]), "rows")
