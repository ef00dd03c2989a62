"""State downloads that are too small to allocate the pinned chunks at once:
repeated ones of 13 MB, through the plain copy first and the chunks once they
have come to 80 MB, with the context remade in between (the chunks go with the
last one), beside a small and a large download of other contexts, all bit for
bit."""
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


def _same(c, s):
    got = c.state(fields=tuple(s))
    for f in s:
        assert np.array_equal(got[f], s[f]), f


def test_repeats_of_one_context():
    for again in range(3):
        c, s = _loaded((29, 30, 26), again)
        for _ in range(9):
            _same(c, s)
        c.Destroy()


def test_once_per_context():
    for k in range(6):
        c, s = _loaded((29, 30, 26 + k), k)
        _same(c, s)
        c.Destroy()


def test_beside_other_sizes():
    made = [_loaded(e, k) for k, e in enumerate([(29, 30, 26), (4, 3, 5), (64, 33, 41), (31, 30, 25)])]
    for order in ((0, 1, 2, 3), (2, 0, 3, 1), (3, 3, 3, 0)):
        for k in order:
            _same(*made[k])
    for c, _ in made:
        c.Destroy()
