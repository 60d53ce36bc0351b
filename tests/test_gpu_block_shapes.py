"""The register-coefficient kernel over its compiled shapes, against the oracle.

Every number of radial groups (n_max 1-4, 5-8, 9-12) with every number of
coefficient registers, exactly filled and rounded up to the next compiled
one, at the smallest and largest l_max and in between, with each average;
every mode of an average (which the run's own rule, evaluated on the host,
says a batch takes), neighbour weights and every compression.  Gates as in
test_gpu_parity.py: float64 |delta| <= 1e-10 (|ref| + max|row|), float32 the
same form at 2e-5.
"""

from __future__ import annotations

import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

import run_choice
from conftest import scaled_error
from mdescriptor_amd import _hip
from mdescriptor_amd.descriptors.basis import basis_gto, basis_polynomial

pytestmark = pytest.mark.gpu

GATES = {"float64": 1e-10, "float32": 2e-5}
SPECIES = [1, 6, 7, 8, 9, 14, 15, 16]
POW_W0 = {"weighting": {"function": "pow", "r0": 2.0, "c": 1.0, "d": 1.0, "m": 4.0, "w0": 0.5}}

# (species, n_max, l_max)
SHAPES = [
    (4, 4, 2), (1, 1, 3), (5, 3, 4), (8, 4, 5), (6, 2, 9),            # one radial group
    (2, 8, 2), (1, 5, 5), (4, 7, 3), (3, 8, 7), (6, 6, 6), (5, 8, 9),  # two
    (1, 9, 2), (2, 12, 4), (3, 9, 5), (4, 10, 6), (5, 9, 8), (2, 11, 9),  # three (four species: five registers)
]


def _structures(seed, sizes, species):
    """Alternating periodic boxes and isolated clusters with every species,
    atoms at least 0.9 A apart."""

    rng = np.random.default_rng(seed)
    numbers, positions, cells, pbc = [], [], [], []
    for i, atoms in enumerate(sizes):
        periodic = i % 2 == 0
        grid = int(np.ceil(atoms ** (1.0 / 3.0)))
        sites = np.stack(np.unravel_index(rng.permutation(grid ** 3)[:atoms], (grid,) * 3), axis=1)
        spacing = 2.2 if periodic else 1.6
        positions.append((sites + 0.5) * spacing + rng.uniform(-0.3, 0.3, (atoms, 3)))
        numbers.append(np.resize(species, atoms)[rng.permutation(atoms)])
        cells.append(np.eye(3) * grid * spacing * (1.0 if periodic else 0.0))
        pbc.append([1, 1, 1] if periodic else [0, 0, 0])
    return SimpleNamespace(numbers=np.concatenate(numbers).astype(np.int32), positions=np.concatenate(positions),
                           cells=np.asarray(cells), pbc=np.asarray(pbc, np.int32),
                           offsets=np.concatenate([[0], np.cumsum(sizes)]))


def _check(ctx, oracle, batch, shape, average, dtype, options=None):
    count, n_max, l_max = shape
    species = SPECIES[:count]
    r_cut = 6.0 if n_max > 8 else 4.0
    alphas, betas = basis_gto(r_cut, n_max, l_max)
    arguments = dict(species=species, n_max=n_max, l_max=l_max, r_cut=r_cut, sigma=1.0, alphas=alphas, betas=betas,
                     average=average, options=options)
    plan = _hip.SoapPlan(ctx, dtype=dtype, **arguments)
    try:
        values, timing = plan.compute(batch)
    finally:
        plan.close()
    assert timing["expansion_tiles"] <= -1000
    expected = oracle.soap(batch, **arguments)
    assert values.shape == expected.shape
    assert np.all(np.isfinite(values))
    error = scaled_error(values, expected)
    assert error <= GATES[dtype], f"{shape} {average} {dtype} {options}: scaled error {error:.3e}"


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("average", ["off", "inner", "outer"])
def test_shape(hip_context, oracle, shape, average):
    # 21 atoms a structure (periodic ones among them) and a lone atom; then
    # structures past a wavefront: averages as runs or centre rows, all of them
    for sizes, dtype in (((21, 13, 1, 20), "float64"), ((70, 66), "float32")):
        _check(hip_context, oracle, _structures(sum(shape), sizes, SPECIES[:shape[0]]), shape, average, dtype)


@pytest.mark.parametrize("shape", [(4, 4, 2), (3, 8, 7), (4, 7, 3), (2, 9, 5), (4, 9, 4)])
@pytest.mark.parametrize("average", ["off", "inner", "outer"])
@pytest.mark.parametrize("name", ["pow_w0", "species_weights", "mu2", "mu1nu1", "crossover", "pow_w0_mu1nu1"])
def test_shape_options(hip_context, oracle, shape, average, name):
    options = {}
    if "pow_w0" in name:
        options.update(POW_W0)
    if name == "species_weights":
        options["species_weights"] = [0.5 + 0.25 * i for i in range(shape[0])]
    if name.split("_")[-1] in ("mu2", "mu1nu1", "crossover"):
        options["compression"] = name.split("_")[-1]
    for sizes, dtype in (((21, 13, 1, 20), "float64"), ((70, 66), "float32")):
        _check(hip_context, oracle, _structures(sum(shape), sizes, SPECIES[:shape[0]]), shape, average, dtype, options)


def _clusters(seed, sizes, species):
    """Isolated clusters only: few neighbours a structure."""

    batch = _structures(seed, sizes, species)
    batch.cells[:], batch.pbc[:] = 0.0, 0
    return batch


@pytest.fixture(scope="module")
def run_rule(tmp_path_factory):
    return run_choice.compiled(tmp_path_factory.mktemp("run_choice"))


# structures of each mode of an average; forced: MDX_HIP_SOAP_KERNEL=block,
# under which structures past a wavefront are formed whole however few
MODES = {
    "species-major structures": ("inner", (21, 13, 1, 20), False),
    "whole structures": ("inner", (70, 66), True),
    "runs": ("inner", (70, 66), False),
    "centre rows": ("outer", (21, 13, 1, 20), False),
    "rows in LDS": ("outer", (5, 1, 7, 4, 6) * 104, False),
}


@pytest.mark.parametrize("shape", [(4, 4, 2), (8, 4, 5), (3, 8, 7), (4, 7, 3), (2, 9, 5), (5, 6, 4), (4, 8, 6)])
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("name", ["default", "pow_w0", "mu2", "mu1nu1", "crossover", "pow_w0_mu1nu1"])
def test_modes_of_an_average(hip_context, oracle, run_rule, monkeypatch, shape, mode, name):
    average, sizes, forced = MODES[mode]
    options = dict(POW_W0) if "pow_w0" in name else {}
    if name.split("_")[-1] in ("mu2", "mu1nu1", "crossover"):
        options["compression"] = name.split("_")[-1]
    if forced:
        monkeypatch.setenv("MDX_HIP_SOAP_KERNEL", "block")
    count, n_max, l_max = shape
    batch = _clusters(sum(shape), sizes, SPECIES[:count])
    for dtype in ("float64", "float32"):
        plan = run_choice.plan_values(count, n_max, l_max, average, dtype, options)
        plan["block_forced"] = forced
        r_cut = 6.0 if n_max > 8 else 4.0
        assert run_choice.mode(run_rule, plan, run_choice.batch_values(batch, r_cut)) == mode
        _check(hip_context, oracle, batch, shape, average, dtype, options)


def test_outer_average_past_the_lds_row(hip_context, oracle):
    """Small structures whose row is too wide for the LDS accumulation (more
    than 48 KB): a float64 partial row per centre."""

    _check(hip_context, oracle, _structures(5, (21, 13, 1, 20), SPECIES[:5]), (5, 9, 8), "outer", "float64")


@pytest.mark.parametrize("shape", [
    (1, 1, 2), (4, 4, 3), (5, 3, 7), (2, 5, 2), (4, 5, 5), (5, 5, 6), (3, 4, 9),  # radial functions in step groups
    (2, 4, 1), (3, 3, 10), (8, 2, 11),                                 # by row, for the 16x16 kernel
    (3, 4, 1), (6, 8, 0), (7, 5, 3), (8, 6, 4),                        # in that kernel (clusters, or many species)
])
@pytest.mark.parametrize("average", ["off", "inner", "outer"])
@pytest.mark.parametrize("name", ["default", "pow_w0", "mu1nu1"])
def test_polynomial_basis(hip_context, oracle, run_rule, shape, average, name):
    """Radial functions computed before the expansion, for the kernel that
    reads them in step groups and for the one that reads them by row; a lone
    atom (only the pair at distance zero), weights and a compression."""

    count, n_max, l_max = shape
    species = SPECIES[:count]
    options = {"default": {}, "pow_w0": dict(POW_W0), "mu1nu1": {"compression": "mu1nu1"}}[name]
    options["polynomial"] = basis_polynomial(4.0, n_max)
    for build, sizes, dtype in ((_structures, (21, 13, 1, 20), "float64"), (_structures, (70, 66), "float32"),
                                (_clusters, (21, 13, 1, 20), "float64")):
        batch = build(sum(shape), sizes, species)
        arguments = dict(species=species, n_max=n_max, l_max=l_max, r_cut=4.0, sigma=1.0, alphas=None, betas=None,
                         average=average, options=options)
        plan = _hip.SoapPlan(hip_context, dtype=dtype, **arguments)
        try:
            values, timing = plan.compute(batch)
        finally:
            plan.close()
        assert (timing["expansion_tiles"] <= -1000) == (2 <= l_max <= 9 and (n_max <= 4 or count <= 6))
        # radial functions in step groups, by row, or in the 16x16 kernel
        values_in = {**run_choice.plan_values(*shape, average, dtype, options), **run_choice.batch_values(batch, 4.0)}
        choice = run_choice.evaluate(run_rule, values_in)
        assert choice["poly_inside"] == (shape in ((3, 4, 1), (6, 8, 0), (7, 5, 3), (8, 6, 4)) and
                                         (count > 6 or values_in["row_bound"] < 32 * count))
        expected = oracle.soap(batch, **arguments)
        assert values.shape == expected.shape
        assert np.all(np.isfinite(values))
        error = scaled_error(values, expected)
        assert error <= GATES[dtype], f"{shape} {average} {dtype} {name}: scaled error {error:.3e}"


@pytest.mark.parametrize("l_max", [1, 10, 4])
@pytest.mark.parametrize("average", ["off", "inner", "outer"])
def test_polynomial_rows_past_a_slot(hip_context, oracle, l_max, average):
    """Centres of more rows than the first slots hold (512; about 600 here):
    the search is run again and its rows counted, so the slots' stride passes
    the row bound that sizes the radial functions.  A host call, a resident
    run, two pipelined frames and a no-allocation run, each against the
    oracle; l_max 1 and 10 by row, 4 in step groups."""

    rng = np.random.default_rng(l_max)
    sizes, species, r_cut = (30, 24), SPECIES[:2], 7.6
    positions, cells = [], []
    for atoms in sizes:
        edge = (atoms / 0.1) ** (1.0 / 3.0)
        sites = np.stack(np.unravel_index(rng.permutation(64)[:atoms], (4, 4, 4)), axis=1)
        positions.append((sites + 0.5) * edge / 4 + rng.uniform(-0.2, 0.2, (atoms, 3)))
        cells.append(np.eye(3) * edge)
    batch = SimpleNamespace(numbers=np.resize(species, sum(sizes)).astype(np.int32), positions=np.concatenate(positions),
                            cells=np.asarray(cells), pbc=np.ones((2, 3), np.int32),
                            offsets=np.concatenate([[0], np.cumsum(sizes)]))
    arguments = dict(species=species, n_max=3, l_max=l_max, r_cut=r_cut, sigma=1.0, alphas=None, betas=None,
                     average=average, options={"polynomial": basis_polynomial(r_cut, 3)})
    expected = oracle.soap(batch, **arguments)
    context = _hip.Context(0)  # whose slots no earlier batch has widened
    plan = _hip.SoapPlan(context, dtype="float64", **arguments)
    pitch = plan.features * 8
    resident = _hip.DeviceBatch(plan, batch)
    out = _hip.DeviceMemory(expected.nbytes)

    def check(values, what):
        error = scaled_error(values, expected)
        assert error <= GATES["float64"], f"l_max {l_max} {average} {what}: scaled error {error:.3e}"

    def rows():
        return out.to_host(np.empty_like(expected))

    try:
        values, timing = plan.compute(batch)
        assert timing["pairs"] > 512 * sum(sizes)
        check(values, "compute")
        resident.run(out.address, pitch)
        check(rows(), "run")
        resident.close()
        resident = _hip.DeviceBatch(plan, batch)
        for _ in range(2):
            resident.run_frame(batch.positions, out.address, pitch)
        resident.wait()
        check(rows(), "frames")
        context.check(context.lib.mdx_hip_soap_run_noalloc(context.handle, plan.handle, resident.handle,
                                                           ctypes.c_void_p(out.address), pitch, None, None))
        check(rows(), "noalloc")
    finally:
        out.free()
        resident.close()
        plan.close()
        context.close()


def _free_device_bytes() -> int:
    runtime = _hip.DeviceMemory.runtime()
    runtime.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t), ctypes.POINTER(ctypes.c_size_t)]
    runtime.hipMemGetInfo.restype = ctypes.c_int
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert runtime.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return int(free.value)


def test_polynomial_large_structure_among_many(hip_context):
    """Inner averages of enough structures for a workgroup each, one of them
    too large for a slice of radial functions (256 MiB): its centres are
    summed in runs, and the run takes little more memory than such a slice.
    Rows against those of the two kinds of structure by themselves."""

    rng = np.random.default_rng(4)
    atoms, lone = 12000, 1100
    edge = (atoms / 0.1) ** (1.0 / 3.0)
    sites = np.stack(np.unravel_index(rng.permutation(23 ** 3)[:atoms], (23,) * 3), axis=1)
    large = SimpleNamespace(numbers=np.resize([1, 8], atoms).astype(np.int32),
                            positions=(sites + 0.5) * edge / 23 + rng.uniform(-0.3, 0.3, (atoms, 3)),
                            cells=np.eye(3)[None] * edge, pbc=np.ones((1, 3), np.int32), offsets=np.array([0, atoms]))
    pairs = SimpleNamespace(numbers=np.resize([1, 8], 2 * lone).astype(np.int32),
                            positions=rng.uniform(0.5, 1.5, (2 * lone, 3)) + np.resize([[0.0] * 3, [1.0] * 3], (2 * lone, 3)),
                            cells=np.zeros((lone, 3, 3)), pbc=np.zeros((lone, 3), np.int32),
                            offsets=np.arange(lone + 1) * 2)
    both = SimpleNamespace(numbers=np.concatenate([pairs.numbers, large.numbers]),
                           positions=np.concatenate([pairs.positions, large.positions]),
                           cells=np.concatenate([pairs.cells, large.cells]), pbc=np.concatenate([pairs.pbc, large.pbc]),
                           offsets=np.concatenate([pairs.offsets, pairs.offsets[-1] + large.offsets[1:]]))
    plan = _hip.SoapPlan(hip_context, species=[1, 8], n_max=3, l_max=2, r_cut=4.5, sigma=1.0, alphas=None, betas=None,
                         average="inner", dtype="float64", options={"polynomial": basis_polynomial(4.5, 3)})
    expected = np.concatenate([plan.compute(pairs)[0], plan.compute(large)[0]])
    batch = _hip.DeviceBatch(plan, both)
    out = _hip.DeviceMemory(expected.nbytes)
    try:
        free = _free_device_bytes()
        timing = batch.run(out.address, plan.features * 8)
        assert free - _free_device_bytes() < 500 << 20
        assert timing["expansion_tiles"] <= -1000
        assert scaled_error(out.to_host(np.empty_like(expected)), expected) <= GATES["float64"]
    finally:
        out.free()
        batch.close()
        plan.close()


@pytest.mark.parametrize("shape,average,name", [
    ((4, 4, 2), "off", "default"), ((3, 8, 7), "off", "default"), ((2, 5, 5), "off", "mu1nu1"),
    ((2, 9, 5), "off", "default"), ((2, 9, 5), "off", "pow_w0"), ((3, 8, 7), "inner", "default"),
    ((4, 7, 3), "outer", "default"),
    # shapes whose float32 rows take float32 exps: not with these
    ((4, 8, 6), "inner", "mu2"), ((4, 8, 6), "inner", "mu1nu1"), ((4, 8, 6), "inner", "pow_w0"),
    ((4, 8, 6), "off", "pow_w0_mu1nu1"), ((5, 6, 4), "outer", "crossover"),
])
def test_float32_rows_of_float64_exps(hip_context, shape, average, name):
    """Float32 rows that take the exps of float64 rows are those rows rounded,
    bit for bit (exps of another error differ in some of them: a packed basis,
    whose fold amplifies it).  Structures of at most a wavefront of atoms and
    one past it."""

    options = dict(POW_W0) if "pow_w0" in name else {}
    if name.split("_")[-1] in ("mu2", "mu1nu1", "crossover"):
        options["compression"] = name.split("_")[-1]
    count, n_max, l_max = shape
    r_cut = 4.0 if n_max > 8 else 3.0
    alphas, betas = basis_gto(r_cut, n_max, l_max)
    rows = {}
    for sizes in ((21, 13, 1, 20), (70, 66)):
        for dtype in ("float64", "float32"):
            plan = _hip.SoapPlan(hip_context, species=SPECIES[:count], n_max=n_max, l_max=l_max, r_cut=r_cut, sigma=1.0,
                                 alphas=alphas, betas=betas, average=average, dtype=dtype, options=options)
            try:
                rows[dtype], timing = plan.compute(_structures(sum(shape), sizes, SPECIES[:count]))
            finally:
                plan.close()
            assert timing["expansion_tiles"] <= -1000
        if average == "inner" and name == "pow_w0" and sizes[0] > 64:
            continue  # a few large structures: float32 exps
        np.testing.assert_array_equal(rows["float32"], rows["float64"].astype(np.float32))


@pytest.mark.parametrize("shape,average,compression", [
    ((5, 2, 6), "off", "off"), ((8, 1, 9), "off", "off"), ((6, 3, 8), "off", "off"), ((5, 3, 2), "outer", "off"),
    ((5, 5, 6), "outer", "off"), ((5, 8, 9), "outer", "mu1nu1"),
])
def test_molecules_of_padded_shapes(hip_context, oracle, shape, average, compression):
    """Structures of few neighbours whose power spectrum this kernel would pad
    take the tile kernels; larger ones of the same shape stay."""

    count, n_max, l_max = shape
    alphas, betas = basis_gto(4.0, n_max, l_max)
    arguments = dict(species=SPECIES[:count], n_max=n_max, l_max=l_max, r_cut=4.0, sigma=1.0, alphas=alphas,
                     betas=betas, average=average, options={"compression": compression} if compression != "off" else {})
    plan = _hip.SoapPlan(hip_context, dtype="float64", **arguments)
    try:
        for sizes, block in (((21, 13, 1, 20), False), ((66, 70), True)):
            batch = _structures(9, sizes, SPECIES[:count])
            if not block:
                batch.cells[:], batch.pbc[:] = 0.0, 0
            values, timing = plan.compute(batch)
            assert (timing["expansion_tiles"] <= -1000) == block
            assert scaled_error(values, oracle.soap(batch, **arguments)) <= GATES["float64"]
    finally:
        plan.close()


def test_runs_keep_the_rows_sums(hip_context, oracle):
    """Inner averages from many short runs: their rows are summed before the
    beta fold, which amplifies the sums' rounding, so the error stays near that
    of the oracle's own order of sums (1e-13 of the row; the gate is 1e-10)."""

    rng = np.random.default_rng(8)
    sizes = (400, 380)
    batch = _structures(8, sizes, SPECIES[:2])
    batch.positions = batch.positions + rng.uniform(-0.1, 0.1, batch.positions.shape)
    alphas, betas = basis_gto(4.0, 8, 3)
    arguments = dict(species=SPECIES[:2], n_max=8, l_max=3, r_cut=4.0, sigma=1.0, alphas=alphas, betas=betas,
                     average="inner")
    plan = _hip.SoapPlan(hip_context, dtype="float64", **arguments)
    try:
        values, timing = plan.compute(batch)
    finally:
        plan.close()
    assert timing["expansion_tiles"] <= -1000
    assert scaled_error(values, oracle.soap(batch, **arguments)) <= 1e-11
