"""Material maps that mix laws without a plastic one among them (elastic with
Maxwell), and a context without any law, in every element layout: the kernel
for a mix serves all laws, and the launch has to bring the waves that kernel
is compiled for.  Sizes with a partial last block of 64 elements; the untuned
layout on both sides of its rule; bit for bit against the oracle."""
import numpy as np
import pytest

from snac_amd import Context, _abi, problem as P
from tests.parity import run_both

pytestmark = pytest.mark.gpu

FIELDS = ("coord", "velocity", "stress")


def _elastic_maxwell(elements):
    p = P.maxwell_viscoelastic(elements=elements, extent_km=tuple(1.5 * e for e in elements))
    upper = P.MaterialSpec(rheology=_abi.RHEOLOGY_ELASTIC, alpha=0.0, beta=0.0, lam=2.0e10, mu=2.5e10,
                           density=2500.0)
    p.materials = [p.materials[0], upper]
    ni, nj, nk = elements
    mat = np.zeros((nk, nj, ni), dtype=np.uint8)
    mat[:, nj // 2:, :] = 1
    p.element_material = mat.reshape(-1)
    return p


def _same(p, steps, variant):
    ref, got, rsc, gsc = run_both(p, steps, variant=variant, fields=FIELDS)
    for f in FIELDS:
        assert np.array_equal(ref[f], got[f]), f
    assert rsc["dt"] == gsc["dt"] and rsc["vmax"] == gsc["vmax"]


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
@pytest.mark.parametrize("elements", [(4, 2, 3), (9, 5, 7)], ids=str)
def test_elastic_with_maxwell(elements, variant):
    _same(_elastic_maxwell(elements), 12, variant)


@pytest.mark.parametrize("elements", [(21, 10, 25), (31, 16, 27)], ids=str)
def test_elastic_with_maxwell_untuned(elements):
    _same(_elastic_maxwell(elements), 6, None)


@pytest.mark.parametrize("variant", [0, 3])
def test_no_law(variant):
    """Stress is rotated and its trace averaged, and nothing is added."""
    def run(v):
        p = P.elastic_box_compression(elements=(7, 5, 6))
        p.materials[0].rheology = 0
        c = Context(p).Construct().Build().Initialise()
        c.set_elem_variant(v)
        c.Execute(8)
        s = c.state(fields=FIELDS)
        c.Destroy()
        return s
    ref, got = run(1), run(variant)
    for f in FIELDS:
        assert np.array_equal(ref[f], got[f]), f
