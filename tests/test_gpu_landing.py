"""Downloads of a state: what was uploaded comes back bit for bit, below and
above the size from which pinned chunks and threads carry it, with a remainder
in the last chunk, and from more threads at once than there are chunks for."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from snac_amd import Context, problem as P

pytestmark = pytest.mark.gpu


def _loaded(elements, seed):
    rng = np.random.default_rng(seed)
    c = Context(P.mohr_coulomb_extension(elements=elements)).Construct()
    s = {"coord": rng.standard_normal((c.N, 3)), "velocity": rng.standard_normal((c.N, 3)),
         "stress": rng.standard_normal((c.E, 10, 6)), "plastic_strain": rng.random((c.E, 10))}
    c.set_state(**s)
    return c, s


@pytest.mark.parametrize("elements", [(3, 2, 5), (23, 21, 31), (24, 21, 31), (64, 33, 41)], ids=str)
def test_round_trip(elements):
    c, s = _loaded(elements, 1)
    for _ in range(2):
        got = c.state(fields=tuple(s))
        for f in s:
            assert np.array_equal(got[f], s[f]), f
    assert np.array_equal(c.state(fields=("stress",))["stress"], s["stress"])


def test_concurrent_downloads():
    made = [_loaded((40, 20, 20 + k), k) for k in range(5)]
    with ThreadPoolExecutor(5) as ex:
        for _ in range(3):
            for (c, s), got in zip(made, ex.map(lambda m: m[0].state(fields=tuple(m[1])), made)):
                for f in s:
                    assert np.array_equal(got[f], s[f]), f
