"""The eight-wave node gather at the sizes where it can go wrong: node rows
around 64 and 128 nodes (a block of 64 nodes then ends on, before or after a
row), rows shorter than a block, one element thick, and the three kinds of
shares (plain, tet densities, other dt types), bit for bit against the
oracle."""
import numpy as np
import pytest

from snac_amd import _abi, problem as P
from tests.parity import run_both

pytestmark = pytest.mark.gpu

SIZES = [(62, 2, 3), (63, 3, 2), (64, 2, 9), (65, 3, 3), (126, 1, 2), (128, 2, 1), (1, 1, 70), (2, 9, 5), (31, 2, 17)]


def _same(p, steps):
    ref, got, rsc, gsc = run_both(p, steps)
    for f in ("coord", "velocity", "stress"):
        assert np.array_equal(ref[f], got[f]), f
    assert rsc["dt"] == gsc["dt"] and rsc["vmax"] == gsc["vmax"]


@pytest.mark.parametrize("elements", SIZES, ids=str)
def test_plain(elements):
    _same(P.elastic_box_compression(elements=elements, extent_km=tuple(2.0 * e for e in elements)), 8)


@pytest.mark.parametrize("elements", [(63, 3, 2), (65, 3, 3), (7, 9, 5)], ids=str)
def test_tet_densities(elements):
    _same(P.maxwell_thermal(elements=elements, extent_km=tuple(2.0 * e for e in elements)), 6)


@pytest.mark.parametrize("dt_type", [_abi.DT_CONSTANT, _abi.DT_WAVE])
def test_other_dt_types(dt_type):
    p = P.elastic_box_compression(elements=(64, 3, 5), extent_km=(128.0, 6.0, 10.0))
    p.dtType, p.timeStep = dt_type, 1.0e-3
    _same(p, 6)


# above 400000 nodes the per-node gather, whose rows are turned within bands
# of 16 planes: fewer rows than the turn, a last band of one, three and sixteen
# planes, rows shorter than a block
@pytest.mark.parametrize("elements", [(750, 1, 272), (1200, 2, 114), (30, 25, 511)], ids=str)
def test_turned_rows(elements):
    _same(P.elastic_box_compression(elements=elements, extent_km=tuple(2.0 * e for e in elements)), 2)


# the heat gather in both forms: up to 200000 nodes and above; the stress holds
# the temperature (density, viscosity) of the steps before
@pytest.mark.parametrize("elements", [(5, 3, 9), (64, 3, 5), (62, 30, 99), (63, 31, 97)], ids=str)
def test_heat(elements):
    p = P.maxwell_thermal(elements=elements, extent_km=tuple(2.0 * e for e in elements))
    ref, got, _, _ = run_both(p, 3)
    for f in ("velocity", "stress"):
        assert np.array_equal(ref[f], got[f]), f
