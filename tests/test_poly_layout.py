"""Extents of the polynomial basis' radial functions in a run's scratch
(csrc/poly_layout.h, compiled here for the host): every value that
k_poly_radial writes and the expansion kernels read lies inside the slice that
the run reserves, and no two share a place, whatever the graph's layout."""

from __future__ import annotations

import ctypes
import subprocess

import numpy as np
import pytest

from conftest import ROOT

SOURCE = """
#include "poly_layout.h"
extern "C" void layout(int64_t bound, int species, int degrees, int channels, int groups, int64_t* out) {
    const mdx::PolyLayout l = mdx::poly_layout(bound, species, degrees, channels, groups != 0);
    out[0] = l.groups;
    out[1] = l.centre;
}
extern "C" int64_t row(int64_t size, int64_t centre, int64_t first, int64_t row, int values) {
    return mdx::poly_row(size, centre, first, row, values);
}
extern "C" int64_t group(int64_t groups, int64_t centre, int64_t first, int64_t group, int values) {
    return mdx::poly_group(groups, centre, first, group, values);
}
extern "C" int slots(int radial_groups) { return mdx::poly_group_slots(radial_groups); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("poly_layout")
    (folder / "host.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT / 'mdescriptor_amd' / 'csrc'}",
                    str(folder / "host.cpp"), "-o", str(folder / "host.so")], check=True)
    lib = ctypes.CDLL(str(folder / "host.so"))
    for name in ("row", "group"):
        getattr(lib, name).restype = ctypes.c_int64
        getattr(lib, name).argtypes = [ctypes.c_int64] * 4 + [ctypes.c_int]
    lib.layout.argtypes = [ctypes.c_int64] + [ctypes.c_int] * 4 + [ctypes.POINTER(ctypes.c_int64)]
    return lib


def _graph(kind: str, species: int, rng):
    """Rows per centre and species, the slot stride (0: compact) and row bound
    of a graph, as build_graph and complete_graph leave them."""

    most = {"pending": 512, "counted": 230, "rebuilt": 670, "compact": 670, "lone": 1}[kind]
    totals = rng.integers(1, most + 1, 40)
    totals[rng.integers(0, 40, 4)] = most
    counts = np.stack([rng.multinomial(t, np.ones(species) / species) for t in totals])
    slots = {"pending": 512, "counted": 512, "rebuilt": 1024, "compact": 0, "lone": 512}[kind]
    return counts, slots, most


@pytest.mark.parametrize("kind", ["pending", "counted", "rebuilt", "compact", "lone"])
@pytest.mark.parametrize("species,degrees,channels", [(1, 1, 1), (2, 2, 4), (3, 11, 3), (5, 4, 8), (12, 3, 5), (2, 2, 16)])
def test_by_row(host, kind, species, degrees, channels):
    rng = np.random.default_rng(1)
    counts, _, bound = _graph(kind, species, rng)
    size = (ctypes.c_int64 * 2)()
    host.layout(bound, species, degrees, channels, 0, size)
    assert size[0] == 0
    values = degrees * channels
    first, count = 7, 29
    used = np.zeros(count * size[1], np.int32)
    for centre in range(first, first + count):
        for row in range(int(counts[centre].sum())):
            at = host.row(size[1], centre, first, row, values)
            assert 0 <= at and at + values <= used.size
            used[at:at + values] += 1
    assert used.max() == 1


@pytest.mark.parametrize("kind", ["pending", "counted", "rebuilt", "compact", "lone"])
@pytest.mark.parametrize("species,degrees,channels", [(1, 3, 1), (4, 4, 4), (5, 8, 3), (2, 3, 5), (6, 7, 8)])
def test_step_groups(host, kind, species, degrees, channels):
    rng = np.random.default_rng(2)
    counts, _, bound = _graph(kind, species, rng)
    size = (ctypes.c_int64 * 2)()
    host.layout(bound, species, degrees, channels, 1, size)
    slots = host.slots((channels + 3) // 4)
    values = degrees * 64
    first, count = 3, 31
    used = np.zeros(count * size[1], np.int32)
    for centre in range(first, first + count):
        groups = int(((counts[centre] + slots - 1) // slots).sum())
        assert groups <= size[0]
        for group in range(groups):
            at = host.group(size[0], centre, first, group, values)
            assert 0 <= at and at + values <= used.size
            used[at:at + values] += 1
    assert used.max() == 1


@pytest.mark.parametrize("kind", ["counted", "rebuilt"])
def test_slot_stride_is_wider_than_the_bound(kind):
    """Why a slice is not addressed by the graph's row slots: once the rows
    have been counted, the slots' stride passes the bound that sizes it."""

    _, slots, bound = _graph(kind, 2, np.random.default_rng(3))
    assert (29 - 1) * slots + bound > 29 * bound
