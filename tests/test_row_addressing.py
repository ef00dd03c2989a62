"""The element pass reads rows of doubles with 32-bit byte offsets in the
tet-per-lane and tet-per-wave layouts.  For every mesh that a context accepts
(up to 2e9 nodes) the layout launched must keep its largest offset below 4 GB;
element per lane has 64-bit addresses.  The rules of snac_amd/csrc/snh_layout.h
are compiled here and asked for columns, slabs and cubes around the limits."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LANE, ELEMENT, LOWREG, WAVE = 0, 1, 2, 3
MESHES = [(2, 2, 2), (17, 9, 17), (2, 2, 1 << 24), (2, 2, (1 << 27) - 1), (2, 2, 1 << 27), (2, 2, (1 << 27) + 1),
          (2, 2, 170000000), (2, 3, 89478485), (2, 3, 89478486), (3, 3, 60000000), (814, 814, 809), (814, 814, 814),
          (377, 377, 379), (378, 378, 379), (2, 16400, 16400), (2, 2, 499999999)]


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("layout")
    (d / "l.c").write_text('#include "snh_layout.h"\n'
                           "int layout(int v, long long N, long long E) { return elem_layout(v, N, E); }\n"
                           "int untuned(int p, int v, long long EI, long long E)"
                           " { return default_elem_variant(p, v, EI, E); }\n"
                           "int batch(long long N, long long E) { return batch_addressable(N, E); }\n")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-I", os.path.join(ROOT, "snac_amd", "csrc"), "-o",
                           str(d / "l.so"), str(d / "l.c")])
    lib = C.CDLL(str(d / "l.so"))
    lib.layout.argtypes = [C.c_int, C.c_longlong, C.c_longlong]
    lib.untuned.argtypes = [C.c_int, C.c_int, C.c_longlong, C.c_longlong]
    lib.batch.argtypes = [C.c_longlong, C.c_longlong]
    return lib


def _largest_offset(layout, N, E):
    """of the rows a layout reads, in bytes"""
    if layout == LANE:
        return 8 * max(10 * E - 1, N - 1)
    return 8 * max(E - 1, N - 1) if layout == WAVE else 0


@pytest.mark.parametrize("nodes", MESHES, ids=str)
def test_offsets_fit_32_bits(rules, nodes):
    I, J, K = nodes
    N, E = I * J * K, (I - 1) * (J - 1) * (K - 1)
    assert N <= 2e9
    for v in (LANE, ELEMENT, LOWREG, WAVE):
        got = rules.layout(v, N, E)
        assert _largest_offset(got, N, E) < 1 << 32, (v, got)
        if _largest_offset(v, N, E) < 1 << 32:
            assert got == v   # a layout that can address the mesh stays
    if rules.batch(N, E):
        assert _largest_offset(LANE, N, E) < 1 << 32 and _largest_offset(WAVE, N, E) < 1 << 32


# (plastic, visco-plastic, elements along x, elements): the faster layout of
# an untuned context, as measured
UNTUNED = [((0, 0, 16, 8112), LANE), ((0, 0, 32, 16384), WAVE), ((0, 0, 8, 819200), WAVE),
           ((1, 0, 100, 441000), LANE), ((1, 0, 192, 884736), WAVE), ((1, 0, 64, 800000), WAVE),
           ((1, 0, 8, 819200), LANE), ((1, 0, 16, 819200), LANE), ((1, 0, 48, 825600), LANE),
           ((1, 0, 16, 2048000), WAVE), ((0, 1, 8, 819200), WAVE), ((0, 1, 100, 441000), LANE)]


@pytest.mark.parametrize("case,layout", UNTUNED, ids=str)
def test_untuned_layout(rules, case, layout):
    assert rules.untuned(*case) == layout
