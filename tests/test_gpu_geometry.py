"""The geometry pass on both sides of its rule (tets over five waves up to
20000 elements, in one lane beyond) and around 64 elements a block: the least
length scale and the time step that follows from it, bit for bit."""
import pytest

from snac_amd import problem as P
from tests.parity import run_both

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (63, 1, 1), (8, 2, 4), (65, 1, 1), (13, 5, 7), (25, 20, 40), (29, 15, 46)]


@pytest.mark.parametrize("elements", SIZES, ids=str)
def test_least_length(elements):
    p = P.elastic_box_compression(elements=elements, extent_km=(2.0 * elements[0], 1.5 * elements[1], 1.0 * elements[2]))
    _, _, ref, got = run_both(p, 6)
    assert ref["minLengthScale"] == got["minLengthScale"] and ref["dt"] == got["dt"]
