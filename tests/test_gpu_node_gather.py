"""The per-node gather, which takes the meshes above the eight-wave gather's
range, in its two row orders and for everything that its instantiations tell
apart: turned rows (88 to 288 nodes, 24 and more of them along y) with last
bands of 16, one and fifteen planes, and rows in bands just outside that rule;
element materials, tet densities and the other dt types; the heat gather with
element materials.  Bit for bit against the oracle.  The mixed-precision
gather, which takes every size, in both orders: the same bits."""
import numpy as np
import pytest

from snac_amd import Context, _abi, problem as P
from tests.parity import run_both

pytestmark = pytest.mark.gpu


def _box(elements):
    return P.elastic_box_compression(elements=elements, extent_km=tuple(2.0 * e for e in elements))


def _two(p):
    upper = P.MaterialSpec(rheology=p.materials[0].rheology, alpha=0.0, beta=0.0, lam=2.0e10, mu=2.5e10,
                           density=2500.0, activationE=0.0, srexponent=1.0, refvisc=1.0e21)
    p.materials = [p.materials[0], upper]
    mat = np.zeros(p.elements[::-1], dtype=np.uint8)
    mat[:, p.elements[1] // 2:, :] = 1
    p.element_material = mat.reshape(-1)
    return p


def _dt(p, kind):
    p.dtType, p.timeStep = kind, 1.0e-3
    return p


def _thermal(elements):
    return P.maxwell_thermal(elements=elements, extent_km=tuple(2.0 * e for e in elements))


def _same(p, steps, fields=("coord", "velocity", "stress")):
    assert p.n_nodes > 400000
    ref, got, rsc, gsc = run_both(p, steps, fields=fields)
    for f in fields:
        assert np.array_equal(ref[f], got[f]), f
    assert rsc["dt"] == gsc["dt"] and rsc["vmax"] == gsc["vmax"]


@pytest.mark.parametrize("elements", [(128, 24, 127), (127, 24, 128), (87, 23, 190), (287, 23, 62), (86, 24, 190),
                                      (288, 23, 62), (128, 22, 144), (99, 25, 159)], ids=str)
def test_row_orders(elements):
    _same(_box(elements), 2)


@pytest.mark.parametrize("case", ["materials", "densities", "densities_materials", "constant", "wave",
                                  "wave_materials"])
@pytest.mark.parametrize("elements", [(128, 24, 128), (60, 40, 161)], ids=["turned", "bands"])
def test_kinds(elements, case):
    p = _thermal(elements) if "densities" in case else _box(elements)
    if "materials" in case:
        p = _two(p)
    if "constant" in case or "wave" in case:
        p = _dt(p, _abi.DT_CONSTANT if "constant" in case else _abi.DT_WAVE)
    _same(p, 3 if "densities" in case else 2,
          ("coord", "velocity", "stress") + (("temperature",) if "densities" in case else ()))


@pytest.mark.parametrize("elements", [(128, 23, 15), (99, 30, 16), (287, 24, 31), (128, 25, 2)], ids=str)
def test_mixed_gather_orders_agree(elements, monkeypatch):
    """Bands of another height than the default are not turned."""
    def run():
        p = P.mohr_coulomb_extension(elements=elements, extent_km=tuple(2.0 * e for e in elements))
        p.precision = _abi.PRECISION_MIXED
        c = Context(p).Construct().Build().Initialise()
        c.Execute(6)
        s, sc = c.state(fields=("coord", "velocity", "stress")), c.scalars()
        c.Destroy()
        return s, sc
    got, gsc = run()
    monkeypatch.setenv("SNH_NODE_BAND", "0")
    ref, rsc = run()
    for f in ref:
        assert np.array_equal(ref[f], got[f]), f
    assert rsc == gsc
