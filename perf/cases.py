"""Performance cases of the SOAP and NeighborList descriptors on one GPU.

A case is a plain dict: what the structures are (``system``, how many, how
many atoms each), the descriptor's parameters, and the entry point a program
calls (``call``):

  compute   ``SOAP.compute``: host arrays in, a host matrix out
  into      ``SOAP.compute_into``: host arrays in, rows into a torch tensor on the GPU
  run       a resident batch takes new positions and runs (``DeviceBatch.set_positions`` + ``run``)
  frames    a trajectory on a resident batch, pipelined (``DeviceBatch.run_frame`` ..., ``wait``)
  pairs     ``NeighborList.compute``: host arrays in, pair values and samples out

``exact`` is the same descriptor written with torch operations in float64.
"""

from __future__ import annotations

import math
import random
from typing import Any

import numpy as np
import torch

import mdescriptor_amd as mdx
from mdescriptor_amd import _hip
from mdescriptor_amd.descriptors.basis import basis_gto, basis_polynomial

ELEMENTS = (1, 6, 7, 8, 9)
FRACTIONS = (0.5, 0.3, 0.1, 0.06, 0.04)
# atoms per cubic angstrom: organic or aqueous condensed phases, a close-packed alloy, liquid silicon
DENSITY = {"organic": 0.10, "alloy": 4 / 3.6 ** 3, "silicon": 0.055}
MOLECULE_SPACING = 1.5  # angstrom between bonded sites of an isolated molecule
FCC_CONSTANT, FCC_DISPLACEMENT = 3.6, 0.07  # the alloy's lattice and its largest displacement per coordinate
# midway between the lattice's neighbour shells: no displacement moves a pair across such a cutoff, so the number
# of pairs is the same for all seeds
SHELL_CUTOFFS = (4.0, 4.75, 5.39, 5.96)
WHOLE_MOLECULE = 12.0  # wider than any of the molecules
FRAMES = 4
POW_W0 = {"function": "pow", "r0": 2.0, "c": 1.0, "d": 1.0, "m": 4.0, "w0": 1.0}
POLY_W = {"function": "poly", "r0": 9.0, "c": 1.0, "m": 1.0}
EXP_W = {"function": "exp", "r0": 2.0, "c": 1.0, "d": 1.0}
WEIGHTINGS = {"": None, "pow": POW_W0, "poly": POLY_W, "exp": EXP_W}

_DEFAULTS = dict(system="organic", structures=1, fewest=64, most=64, triclinic=False, species=3, n=8, l=6, r_cut=5.0,
                 average="off", dtype="float64", rbf="gto", weighting="", compression="off", call="into",
                 half=False)


def _case(**values: Any) -> dict:
    return {**_DEFAULTS, **values}


def listed() -> list[dict]:
    return [
        # interactive use: one molecule, the descriptor's own defaults (n_max 8, l_max 6, inner average, float64)
        _case(name="molecule-default", system="molecule", fewest=21, most=21, species=3, average="inner",
              call="compute"),
        # one step of a small molecular dynamics run: a 192-atom water-like box, rows stay on the GPU
        _case(name="box-step", fewest=192, most=192, species=2, n=4, l=3, r_cut=4.5, call="run"),
        # several replicas of that box stepped together, frames pipelined
        _case(name="box-frames", structures=64, fewest=192, most=192, species=2, n=4, l=3, r_cut=4.5, call="frames"),
        # featurising a data set of small ragged periodic cells into host memory, a wider radial basis
        _case(name="dataset-rows", structures=40, fewest=23, most=230, triclinic=True, species=3, n=9, l=5,
              call="compute"),
        # large condensed-phase cells of four elements, float32 rows for a model on the same GPU
        _case(name="hcno-rows", structures=16, fewest=4096, most=4096, species=4, dtype="float32", call="run"),
        # a library of isolated molecules, one averaged row each
        _case(name="molecules-inner", system="molecule", structures=20000, fewest=9, most=29, species=5, n=6, l=4,
              average="inner"),
        # the same with averaged power spectra
        _case(name="molecules-outer", system="molecule", structures=3000, fewest=9, most=29, species=5, n=6, l=4,
              average="outer"),
        # a five-component alloy at a high angular resolution
        _case(name="alloy-rows", system="alloy", fewest=10976, most=10976, species=5, n=8, l=8, r_cut=6.0,
              dtype="float32"),
        # one large elemental cell, the widest basis
        _case(name="silicon-large", system="silicon", fewest=216000, most=216000, species=1, n=12, l=9, r_cut=5.5,
              dtype="float32", call="run"),
        # distance weighting with a compressed spectrum, odd basis sizes
        _case(name="weighted-crossover", structures=9, fewest=700, most=1100, triclinic=True, species=3, n=7, l=6,
              weighting="pow", compression="crossover"),
        # the polynomial radial basis
        _case(name="polynomial-rows", structures=3, fewest=900, most=1100, species=3, n=6, l=5, rbf="polynomial"),
        # neighbour pairs of large supercells into host memory
        _case(name="pairs", system="alloy", structures=3, fewest=5324, most=5324, species=5, r_cut=5.96, call="pairs"),
    ]


def _log_uniform(rng: random.Random, low: float, high: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng: random.Random) -> dict:
    while True:
        case = _draw(rng)
        pairs = _pairs(case)
        size = 4 if case["dtype"] == "float32" else 8
        rows = _atoms(case) if case["average"] == "off" else case["structures"]
        rows *= FRAMES if case["call"] == "frames" else 1
        fits = case["species"] * case["n"] * (case["l"] + 1) ** 2 <= 6000
        cost = work(case)["flops"]
        small = rows * _features(case) * size < 3e8 and pairs < 3e7 and cost < 2e11
        if fits and small and (case["rbf"] == "gto" or pairs < 1.5e6):
            return case


def _draw(rng: random.Random) -> dict:
    call = rng.choice(["compute", "into", "into", "run", "run", "frames", "pairs"])
    system = rng.choice(["organic", "organic", "molecule", "alloy", "silicon"] if call != "pairs" else
                        ["molecule", "alloy"])
    case = _case(call=call, system=system, species=rng.randint(1, 5), n=rng.randint(2, 10), l=rng.randint(1, 9),
                 r_cut=round(rng.uniform(4.0, 6.0), 2), dtype=rng.choice(["float32", "float64"]),
                 average=rng.choice(["off", "off", "inner", "outer"]))
    if system == "silicon":
        case["species"] = 1
    if case["n"] > 8:
        case["r_cut"] = max(case["r_cut"], 5.0)
    if system == "molecule":
        case["structures"] = _log_uniform(rng, 1, 6000)
        case["fewest"] = rng.randint(3, 15)
        case["most"] = case["fewest"] + rng.randint(0, 20)
        if case["average"] == "off" and rng.random() < 0.7:
            case["average"] = "inner"
    elif system == "alloy":
        case["structures"] = _log_uniform(rng, 1, 20)
        repeat = _log_uniform(rng, 2, (10000 // case["structures"]) ** (1.0 / 3.0))
        case["fewest"] = case["most"] = 4 * repeat ** 3
    else:
        case["structures"] = _log_uniform(rng, 1, 64)
        case["fewest"] = _log_uniform(rng, 16, max(17, 40000 // case["structures"]))
        case["most"] = case["fewest"] + rng.choice([0, case["fewest"] // 3])
        case["triclinic"] = rng.random() < 0.5
    if call == "pairs":
        case.update(average="off", dtype="float64", half=rng.random() < 0.5,
                    r_cut=WHOLE_MOLECULE if system == "molecule" else rng.choice(SHELL_CUTOFFS))
        return case
    option = rng.random()
    if option < 0.15:
        case.update(weighting=rng.choice(["pow", "poly", "exp"]), n=min(case["n"], 8), l=min(case["l"], 7))
    elif option < 0.3:
        case.update(compression=rng.choice(["mu2", "mu1nu1", "crossover"]), n=min(case["n"], 8),
                    l=min(case["l"], 7))
    elif option < 0.4:
        case.update(rbf="polynomial", n=min(case["n"], 7), l=min(case["l"], 7))
    return case


# ------------------------------------------------------------------ inputs

def _sizes(case: dict) -> np.ndarray:
    """Atoms of each structure: the case's own, whatever the seed."""

    rng = np.random.Generator(np.random.PCG64([case["structures"], case["fewest"], case["most"]]))
    return rng.integers(case["fewest"], case["most"] + 1, size=case["structures"])


def _species(case: dict) -> list[int]:
    if case["system"] == "alloy":
        return [24, 26, 27, 28, 29][:case["species"]]
    if case["system"] == "silicon":
        return [14]
    return list(ELEMENTS[:case["species"]])


def _numbers(case: dict, rng: np.random.Generator, total: int) -> np.ndarray:
    species = np.asarray(_species(case))
    if case["system"] == "alloy":
        return rng.choice(species, size=total)
    weights = np.asarray(FRACTIONS[:len(species)])
    return rng.choice(species, size=total, p=weights / weights.sum())


def _lattice_sites(rng: np.random.Generator, count: int) -> tuple[np.ndarray, float]:
    """`count` distinct sites of a cubic lattice over the unit cell, displaced at
    random inside their lattice cells, and the lattice constant."""

    grid = int(math.ceil(count ** (1.0 / 3.0) - 1e-9))
    chosen = np.sort(rng.permutation(grid ** 3)[:count])
    sites = np.stack(np.unravel_index(chosen, (grid, grid, grid)), axis=1)
    return (sites + 0.5 + rng.uniform(-0.25, 0.25, size=(count, 3))) / grid, 1.0 / grid


def _molecules(rng: np.random.Generator, sizes: np.ndarray) -> np.ndarray:
    """Compact random clusters: of a 4 x 4 x 4 lattice of bonded sites, each
    molecule takes those nearest a random point, displaced a little and placed
    at a random offset."""

    structures, grid = len(sizes), 4
    sites = np.stack(np.unravel_index(np.arange(grid ** 3), (grid, grid, grid)), axis=1).astype(np.float64)
    centre = rng.uniform(1.0, 2.0, size=(structures, 1, 3))
    distance = np.sum((sites[None] - centre) ** 2, axis=2)
    order = np.argsort(distance, axis=1)
    positions = sites[order] + rng.uniform(-0.15, 0.15, size=(structures, grid ** 3, 3))
    positions = positions * MOLECULE_SPACING + rng.uniform(-20.0, 20.0, size=(structures, 1, 3))
    return positions[np.arange(grid ** 3)[None, :] < sizes[:, None]]


def _batch(case: dict, seed: int) -> mdx.StructureBatch:
    rng = np.random.Generator(np.random.PCG64(seed))
    sizes = _sizes(case)
    structures = len(sizes)
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    numbers = _numbers(case, rng, int(offsets[-1]))
    ids = tuple(str(i) for i in range(structures))
    if case["system"] == "molecule":
        return mdx.StructureBatch(numbers, _molecules(rng, sizes), np.zeros((structures, 3, 3)),
                                  np.zeros((structures, 3), dtype=np.int32), offsets, ids)
    positions, cells = [], []
    if case["system"] == "alloy":
        repeat = round((case["fewest"] / 4) ** (1.0 / 3.0))
        sites = np.stack(np.unravel_index(np.arange(repeat ** 3), (repeat,) * 3), axis=1)[:, None]
        sites = (sites + 0.5 * np.array([[0, 0, 0], [1, 1, 0], [1, 0, 1], [0, 1, 1]])).reshape(-1, 3) + 0.25
        moves = rng.uniform(-FCC_DISPLACEMENT, FCC_DISPLACEMENT, size=(structures, len(sites), 3))
        positions = list(sites * FCC_CONSTANT + moves)
        cells = [np.eye(3) * FCC_CONSTANT * repeat] * structures
        sizes = []
    for count in sizes:
        length = (count / DENSITY[case["system"]]) ** (1.0 / 3.0)
        cell = np.eye(3) * length
        if case["triclinic"]:
            cell[1, 0], cell[2, 0], cell[2, 1] = rng.uniform(-0.2, 0.2, size=3) * length
        fractional, _ = _lattice_sites(rng, int(count))
        positions.append(fractional @ cell)
        cells.append(cell)
    return mdx.StructureBatch(numbers, np.concatenate(positions), np.asarray(cells),
                              np.ones((structures, 3), dtype=np.int32), offsets, ids)


def _frames(positions: np.ndarray, seed: int, count: int) -> np.ndarray:
    """Positions of `count` frames: the structure with thermal displacements."""

    rng = np.random.Generator(np.random.PCG64([seed, 1]))
    return positions[None] + rng.normal(scale=0.02, size=(count, *positions.shape))


def _soap(case: dict) -> mdx.SOAP:
    return mdx.SOAP(species=_species(case), rbf=case["rbf"], n_max=case["n"], l_max=case["l"], r_cut=case["r_cut"],
                    average=case["average"], weighting=WEIGHTINGS[case["weighting"]],
                    compression={"mode": case["compression"], "species_weighting": None},
                    output=mdx.OutputOptions(dtype=case["dtype"]))


def prepare(case: dict, seed: int) -> dict:
    batch = _batch(case, seed)
    state: dict[str, Any] = {"case": case, "batch": batch}
    if case["call"] == "pairs":
        state["pairs"] = mdx.NeighborList(cutoff=case["r_cut"], full_neighbor_list=not case["half"])
        return state
    soap = state["soap"] = _soap(case)
    if case["call"] == "compute":
        return state
    rows = batch.atoms if case["average"] == "off" else batch.structures
    shape = (rows, soap.feature_count)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.float64
    count = FRAMES if case["call"] == "frames" else 1
    state["out"] = [torch.empty(shape, dtype=dtype, device="cuda") for _ in range(count)]
    if case["call"] == "into":
        return state
    settings = soap.settings
    payload = settings.hip_payload()["radial_basis"]
    options = {"compression": settings.compression, "weighting": settings.weighting}
    plan = state["plan"] = _hip.SoapPlan(
        _hip.shared_context(0), species=settings.species, n_max=settings.n_max, l_max=settings.l_max,
        r_cut=settings.r_cut, sigma=settings.sigma, alphas=payload.get("alphas"), betas=payload.get("betas"),
        average=settings.average, dtype=case["dtype"],
        options=_hip.plan_options(options, list(settings.species), payload))
    state["device_batch"] = _hip.DeviceBatch(plan, batch)
    state["positions"] = torch.from_numpy(_frames(batch.positions, seed, count)).cuda()
    return state


def run(state: dict) -> Any:
    case = state["case"]
    if case["call"] == "pairs":
        result = state["pairs"].compute(state["batch"])
        return result.values, result.samples
    if case["call"] == "compute":
        return state["soap"].compute(state["batch"]).values
    out = state["out"]
    pitch = out[0].stride(0) * out[0].element_size()
    if case["call"] == "into":
        return state["soap"].compute_into(state["batch"], out[0])
    resident, positions = state["device_batch"], state["positions"]
    if case["call"] == "run":
        resident.set_positions(positions[0].data_ptr())
        resident.run(out[0].data_ptr(), pitch)
        return out[0]
    for frame, rows in zip(positions, out):
        resident.run_frame(frame.data_ptr(), rows.data_ptr(), pitch)
    resident.wait()
    return out


# -------------------------------------------------------------------- work

def _atoms(case: dict) -> float:
    return case["structures"] * (case["fewest"] + case["most"]) / 2.0


def _cutoff(case: dict) -> float:
    """Neighbour radius: SOAP looks past r_cut to where a unit Gaussian has fallen to 1e-3."""

    return case["r_cut"] + (0.0 if case["call"] == "pairs" else math.sqrt(-2.0 * math.log(1e-3)))


def _pairs(case: dict) -> float:
    size = (case["fewest"] + case["most"]) / 2.0
    if case["system"] == "molecule":
        return case["structures"] * size * size  # every atom sees the whole molecule
    return _atoms(case) * (1.0 + 4.0 / 3.0 * math.pi * _cutoff(case) ** 3 * DENSITY[case["system"]])


def _features(case: dict) -> int:
    s, n, degrees = case["species"], case["n"], case["l"] + 1
    if case["compression"] == "mu2":
        return n * (n + 1) // 2 * degrees
    if case["compression"] == "mu1nu1":
        return s * n * n * degrees
    if case["compression"] == "crossover":
        return s * n * (n + 1) // 2 * degrees
    return s * n * (s * n + 1) // 2 * degrees


def work(case: dict) -> dict:
    """Of one pass: the atoms read once and the rows written once; the
    multiply-adds of the expansion (per pair, n radial functions times
    (l + 1)^2 harmonics, one exponential per radial function and degree), of
    the basis change and of the power spectrum."""

    atoms, pairs = _atoms(case), _pairs(case)
    if case["call"] == "pairs":
        kept = (pairs - atoms) * (0.5 if case["half"] else 1.0)
        return {"bytes": atoms * 28 + kept * 80, "flops": pairs * 8}
    s, n, degrees = case["species"], case["n"], case["l"] + 1
    harmonics = degrees * degrees
    size = 4 if case["dtype"] == "float32" else 8
    rows = atoms if case["average"] == "off" else case["structures"]
    spectra = case["structures"] if case["average"] == "inner" else atoms
    radial = n * degrees if case["rbf"] == "gto" else 100 * (2 + 2 * degrees + 2 * n * degrees)
    flops = pairs * (radial + 2 * n * harmonics)
    flops += spectra * (2 * s * n * n * harmonics + 2 * _features(case) / degrees * harmonics)
    frames = FRAMES if case["call"] == "frames" else 1
    return {"bytes": frames * (atoms * 28 + rows * _features(case) * size), "flops": frames * flops}


def tolerance(case: dict) -> Any:
    if case["call"] == "pairs":
        return "exact"
    # float32 rows: the rounding of a float64 value (2.5e-8 measured)
    if case["dtype"] == "float32":
        return {"rel": 1e-7, "max": 1e-6}
    # float64 rows: the basis change cancels more the more radial functions there are (measured against exact():
    # 2e-13 at 8, 1e-12 at 9 and 10, more at the shortest cutoffs), the polynomial kernels' recurrence amplifies
    # rounding near the origin (2e-12, single values 5e-11)
    if case["rbf"] == "polynomial":
        return {"rel": 1e-11, "max": 4e-10}
    return {"rel": 5e-12, "max": 5e-11} if case["n"] <= 8 else {"rel": 2e-11, "max": 2e-10}


# ------------------------------------------------------------------- exact

def _harmonics(x: torch.Tensor, y: torch.Tensor, z: torch.Tensor, l_max: int) -> list[torch.Tensor]:
    """Real regular solid harmonics, one (..., 2l+1) tensor per degree."""

    r2 = x * x + y * y + z * z
    cos, sin = {(0, 0): torch.ones_like(x)}, {(0, 0): torch.zeros_like(x)}
    for m in range(l_max + 1):
        if m > 0:
            f = -(2.0 * m - 1.0)
            cos[m, m] = f * (x * cos[m - 1, m - 1] - y * sin[m - 1, m - 1])
            sin[m, m] = f * (x * sin[m - 1, m - 1] + y * cos[m - 1, m - 1])
        for part in (cos, sin):
            if m < l_max:
                part[m + 1, m] = (2.0 * m + 1.0) * z * part[m, m]
            for l in range(m + 2, l_max + 1):
                part[l, m] = ((2.0 * l - 1.0) * z * part[l - 1, m] - (l + m - 1.0) * r2 * part[l - 2, m]) / (l - m)
    result = []
    for l in range(l_max + 1):
        norm = [math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - m) / math.factorial(l + m))
                * (math.sqrt(2.0) if m else 1.0) for m in range(l + 1)]
        columns = [norm[m] * cos[l, m] for m in range(l, 0, -1)] + [norm[0] * cos[l, 0]]
        columns += [norm[m] * sin[l, m] for m in range(1, l + 1)]
        result.append(torch.stack(columns, dim=-1))
    return result


def _weight(case: dict, distance: torch.Tensor, own: torch.Tensor) -> torch.Tensor:
    options = WEIGHTINGS[case["weighting"]]
    if options is None:
        return torch.ones_like(distance)
    ratio = distance / options["r0"]
    if options["function"] == "poly":
        value = options["c"] * (1.0 + 2.0 * ratio ** 3 - 3.0 * ratio ** 2) ** options["m"]
        value = torch.where(distance > options["r0"], torch.zeros_like(value), value)
    elif options["function"] == "pow":
        value = options["c"] / (options["d"] + ratio ** options["m"])
    else:
        value = options["c"] / (options["d"] + torch.exp(-ratio))
    return torch.where(own, torch.full_like(value, options["w0"]), value) if "w0" in options else value


def _polynomial_radial(case: dict, distance: torch.Tensor) -> list[torch.Tensor]:
    """Projections on the radial basis of a unit Gaussian at `distance`, per degree."""

    eta, l_max = 0.5, case["l"]
    grid, weights, values = (torch.from_numpy(a).cuda() for a in basis_polynomial(case["r_cut"], case["n"]))
    quadrature = (weights * grid ** 2)[:, None] * values.T
    centre = (distance <= 1e-14)[..., None]
    r = torch.where(centre, torch.ones_like(distance[..., None]), distance[..., None])
    prefactor = 0.25 / (eta * r * grid)
    minus, plus = torch.exp(-eta * (grid - r) ** 2), torch.exp(-eta * (grid + r) ** 2)
    kernels = [prefactor * (minus - plus)]
    if l_max >= 1:
        kernels.append(prefactor * (minus + plus - 2.0 * kernels[0]))
    for l in range(2, l_max + 1):
        kernels.append((kernels[l - 2] - prefactor * (4.0 * l - 2.0) * kernels[l - 1]).clamp_min(0.0))
    result = []
    for l, kernel in enumerate(kernels):
        own = torch.exp(-eta * grid ** 2) if l == 0 else torch.zeros_like(grid)
        kernel = torch.where(centre, own, kernel)
        scale = 4.0 * math.pi * torch.where(centre, torch.ones_like(r), r) ** -l
        result.append((kernel @ quadrature) * scale)
    return result


def _coefficients(case: dict, centres: torch.Tensor, images: torch.Tensor, kind: torch.Tensor,
                  own: torch.Tensor) -> list[torch.Tensor]:
    """Per degree the (blocks, centres, species, n, 2l+1) coefficients of blocks
    of centres (b, c, 3) among candidate images (b, i, 3); kind is the species
    of an image, -1 for none, own its atom where it is the atom itself, else -1."""

    n, l_max, s = case["n"], case["l"], 1 if case["compression"] == "mu2" else case["species"]
    offset = images[:, None] - centres[..., :3][:, :, None]
    x, y, z = offset.unbind(-1)
    d2 = x * x + y * y + z * z
    near = (d2 <= _cutoff(case) ** 2) & (kind >= 0)[:, None]
    is_own = own[:, None] == centres[..., 3][:, :, None].to(own.dtype)
    weight = _weight(case, torch.sqrt(d2), is_own) * near
    hot = torch.stack([(kind == t) if s > 1 else (kind >= 0) for t in range(s)], dim=-1)[:, None].to(d2.dtype)
    result = []
    if case["rbf"] == "gto":
        alphas, betas = (torch.from_numpy(a).cuda() for a in basis_gto(case["r_cut"], n, l_max))
    else:
        projected = _polynomial_radial(case, torch.sqrt(d2))
    for l, y_l in enumerate(_harmonics(x, y, z, l_max)):
        angular = (weight[..., None, None] * hot[..., None] * y_l[..., None, :]).flatten(-2)
        if case["rbf"] == "gto":
            eta = 0.5
            denominator = alphas[l] + eta
            radial = torch.exp(-(alphas[l] * eta / denominator) * d2[..., None])
            fold = math.pi ** 1.5 * betas[l] * (eta ** l * denominator ** (-l - 1.5))
            c = torch.matmul(fold, torch.matmul(radial.transpose(-1, -2).contiguous(), angular))
        else:
            c = torch.matmul(projected[l].transpose(-1, -2).contiguous(), angular)
        result.append(c.unflatten(-1, (s, 2 * l + 1)).transpose(-3, -2))
    return result


def _power_spectrum(case: dict, c: list[torch.Tensor]) -> torch.Tensor:
    """Rows of features from per-degree (rows, species, n, 2l+1) coefficients."""

    n, mode = case["n"], case["compression"]
    s = c[0].shape[1]
    upper = torch.triu_indices(n, n)

    def block(a: torch.Tensor, b: torch.Tensor, l: int, triangle: bool) -> torch.Tensor:
        gram = math.pi * math.sqrt(8.0 / (2 * l + 1)) * torch.matmul(a, b.transpose(-1, -2).contiguous())
        return gram[:, upper[0], upper[1]] if triangle else gram.flatten(1)

    parts = []
    if mode == "mu1nu1":
        summed = [v.sum(1) for v in c]
        parts = [block(v[:, t], summed[l], l, False) for t in range(s) for l, v in enumerate(c)]
    else:
        for t1 in range(s):
            for t2 in range(t1, s if mode == "off" else t1 + 1):
                parts += [block(v[:, t1], v[:, t2], l, t1 == t2) for l, v in enumerate(c)]
    return torch.cat(parts, dim=1)


def _neighbourhoods(case: dict, batch: mdx.StructureBatch, positions: np.ndarray) -> list[tuple]:
    """Blocks (centres, images, species, own): of each structure, the centres of
    one box of a grid as wide as the cutoff and every image in reach of it."""

    cutoff = _cutoff(case)
    kinds = np.searchsorted(_species(case), batch.numbers)
    blocks = []
    for i in range(batch.structures):
        first, last = int(batch.offsets[i]), int(batch.offsets[i + 1])
        home, cell = positions[first:last], batch.cells[i]
        atoms = np.arange(first, last)
        low, high = home.min(0) - cutoff, home.max(0) + cutoff
        images, atom_of, is_home = [home], [atoms], [np.ones(len(home), dtype=bool)]
        if batch.pbc[i].all():
            reach = np.floor(cutoff * np.linalg.norm(np.linalg.inv(cell), axis=0) + 1.01).astype(int)
            ranges = [np.arange(-k, k + 1) for k in reach]
            for shift in np.stack(np.meshgrid(*ranges, indexing="ij"), -1).reshape(-1, 3):
                if not shift.any():
                    continue
                moved = home + ((shift[0] * cell[0] + shift[1] * cell[1]) + shift[2] * cell[2])
                inside = np.all((moved >= low) & (moved <= high), axis=1)
                images.append(moved[inside])
                atom_of.append(atoms[inside])
                is_home.append(np.zeros(int(inside.sum()), dtype=bool))
        xyz, atom, here = np.concatenate(images), np.concatenate(atom_of), np.concatenate(is_home)
        boxes = np.floor((xyz - low) / cutoff).astype(np.int64)
        dims = boxes.max(0) + 3
        key = ((boxes[:, 0] + 1) * dims[1] + boxes[:, 1] + 1) * dims[2] + boxes[:, 2] + 1
        order = np.argsort(key, kind="stable")
        xyz, atom, here, key = xyz[order], atom[order], here[order], key[order]
        for box in np.unique(key[here]):
            near = []
            for dx in (-1, 0, 1):
                for dy in (-1, 0, 1):
                    row = box + (dx * dims[1] + dy) * dims[2]
                    a, b = np.searchsorted(key, [row - 1, row + 2])
                    near.append(np.arange(a, b))
            near = np.concatenate(near)
            a, b = np.searchsorted(key, [box, box + 1])
            centres = np.arange(a, b)[here[a:b]]
            blocks.append((atom[centres], xyz[centres], xyz[near], kinds[atom[near]],
                           np.where(here[near], atom[near], -1)))
    return blocks


def _exact_rows(case: dict, batch: mdx.StructureBatch, positions: np.ndarray) -> torch.Tensor:
    n, l_max, s = case["n"], case["l"], 1 if case["compression"] == "mu2" else case["species"]
    total = batch.atoms
    structure = torch.from_numpy(np.repeat(np.arange(batch.structures), np.diff(batch.offsets))).cuda()
    count = torch.from_numpy(np.diff(batch.offsets)).cuda().to(torch.float64)[:, None]
    features = _features(case)
    rows = torch.zeros((total if case["average"] == "off" else batch.structures, features), dtype=torch.float64,
                       device="cuda")
    sums = [torch.zeros((batch.structures, s, n, 2 * l + 1), dtype=torch.float64, device="cuda")
            for l in range(l_max + 1)]
    blocks = sorted(_neighbourhoods(case, batch, positions), key=lambda b: (len(b[2]), len(b[0])))
    # values per (centre, image) pair held at once
    width = n + s * (2 * l_max + 1) + 8 + (600 if case["rbf"] != "gto" else 0)
    start = 0
    while start < len(blocks):
        stop, c_most, i_most = start, 0, 0
        while stop < len(blocks):
            c_new, i_new = max(c_most, len(blocks[stop][0])), max(i_most, len(blocks[stop][2]))
            if stop > start and (stop + 1 - start) * c_new * i_new * width > 6e8:
                break
            c_most, i_most, stop = c_new, i_new, stop + 1
        group = blocks[start:stop]
        start = stop
        b = len(group)
        atoms = np.full((b, c_most), -1)
        centres, images = np.zeros((b, c_most, 4)), np.zeros((b, i_most, 3))
        kind, own = np.full((b, i_most), -1), np.full((b, i_most), -1)
        for j, (atom, xyz, near, k, o) in enumerate(group):
            atoms[j, :len(atom)] = atom
            centres[j, :len(atom), :3], centres[j, :len(atom), 3] = xyz, atom
            images[j, :len(near)], kind[j, :len(near)], own[j, :len(near)] = near, k, o
        used = torch.from_numpy(atoms >= 0).cuda()
        index = torch.from_numpy(atoms).cuda()[used]
        c = _coefficients(case, *(torch.from_numpy(v).cuda() for v in (centres, images, kind, own)))
        c = [v[used] for v in c]
        if case["average"] == "inner":
            for l, v in enumerate(c):
                sums[l].index_add_(0, structure[index], v)
        elif case["average"] == "outer":
            rows.index_add_(0, structure[index], _power_spectrum(case, c))
        else:
            rows[index] = _power_spectrum(case, c)
    if case["average"] == "inner":
        return _power_spectrum(case, [v / count[:, :, None, None] for v in sums])
    return rows / count if case["average"] == "outer" else rows


def exact(case: dict, seed: int) -> Any:
    if case["call"] == "pairs":
        return None  # compared bit for bit; the order of a centre's pairs is the search's own
    batch = _batch(case, seed)
    if case["call"] in ("compute", "into"):
        rows = _exact_rows(case, batch, batch.positions)
        return rows.cpu().numpy() if case["call"] == "compute" else rows
    count = FRAMES if case["call"] == "frames" else 1
    frames = [_exact_rows(case, batch, p) for p in _frames(batch.positions, seed, count)]
    return frames if case["call"] == "frames" else frames[0]
