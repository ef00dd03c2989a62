"""Tets whose volume lies a few last places below a power of two, where the
reciprocal of the volume comes closest to a rounding midpoint: the spin takes
the correctly rounded one, so a stress turned through a large angle in one
step has the oracle's bits, in every element layout."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from snac_amd import Context, _abi, problem as P

pytestmark = pytest.mark.gpu

FIELDS = ("stress", "coord", "velocity")


def _problem(last_places):
    """Elements of 3 x 2 x 1 with lx a few last places shorter: corner tets of
    volume 1, middle ones of 2, less those last places and rounding."""
    p = P.elastic_box_compression(elements=(3, 3, 4))
    p.extent = ((0.0, 9.0 * (1.0 - last_places * 2.0 ** -53)), (-6.0, 0.0), (0.0, 4.0))
    p.hydrostatic = False
    p.dtType, p.timeStep = _abi.DT_CONSTANT, 0.25
    return p


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_spin_bits(variant):
    below = 0
    for places in range(0, 24):
        p = _problem(places)
        rng = np.random.default_rng(places)
        v = rng.standard_normal((p.n_nodes, 3))
        s = 1.0e6 * rng.standard_normal((p.n_elements, 10, 6))
        o = Oracle(p)
        o.set_state(velocity=v, stress=s)
        o.timestep_zero()
        o.step(1)
        c = Context(p).Construct()
        c.set_state(velocity=v, stress=s)
        c.timestep_zero()
        vol = c.state(fields=("volume",))["volume"]
        m, _ = np.frexp(vol)
        below += int(np.sum((m < 1.0) & (m > 1.0 - 16 * 2.0 ** -53)))
        c.set_elem_variant(variant)
        c.Execute(1)
        ref, got = o.state(), c.state(fields=FIELDS)
        for f in FIELDS:
            assert np.array_equal(ref[f], got[f]), (places, f)
        o.close()
        c.Destroy()
    assert below > 1000   # the volumes are where the test wants them
