"""Sync (snh_sync) reduces the block partials that the last geometry and node
passes left, and repeated on an unchanged state it gives the same scalars:
after the batched and the branch launches of an ensemble, after a capture that
has recorded passes without running them, and after the autotuner's launches,
all of which write or count other partials than a step of the context does."""
import numpy as np
import pytest

from snac_amd import Context, _abi, problem as P
from snac_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu

KEYS = ("dt", "speedOfSound", "minLengthScale", "vmax")


def _stretched(elements, seed=0):
    """An elastic box whose x-faces move apart and whose last z-plane moves
    fastest: the least length grows from step to step and the largest
    prescribed velocity lies among the last nodes."""
    p = P.elastic_box_compression(elements=elements, extent_km=tuple(2.0 * e for e in elements))
    v = P.CM_PER_YEAR * (1.0 + 0.1 * seed)
    p.bcs = [("left", _abi.VX, (-v, 0.0, 0.0)), ("right", _abi.VX, (v, 0.0, 0.0)),
             ("front", _abi.VZ, (-v, 0.0, 0.0)), ("bottom", _abi.VY, (0.0, 0.0, 0.0)),
             ("back", _abi.VZ, (0.0, 0.0, 7.0 * v))]
    return p


def _made(p):
    return Context(p).Construct().Build().Initialise()


def _synced_twice(c):
    before = c.scalars()
    c.sync()
    c.synchronize()
    after = c.scalars()
    return [before[k] for k in KEYS], [after[k] for k in KEYS]


@pytest.mark.parametrize("batch", ["1", "0"])
@pytest.mark.parametrize("sizes", [[(16, 8, 16), (9, 5, 13)], [(30, 10, 70), (24, 33, 30)]], ids=["small", "large"])
def test_sync_after_ensemble_steps(sizes, batch, monkeypatch):
    monkeypatch.setenv("SNH_ENSEMBLE_BATCH", batch)
    members = [_made(_stretched(e, k)) for k, e in enumerate(sizes)]
    ens = Ensemble(members, graph_steps=4, autotune=False)
    assert ens.batched == (batch == "1")
    for n in (8, 3, 4):
        ens.step(n).synchronize()
        for c in members:
            before, after = _synced_twice(c)
            assert before == after
    ens.destroy()


@pytest.mark.parametrize("batch", ["1", "0"])
def test_sync_between_create_and_step(batch, monkeypatch):
    """The members have stepped (every partial written), then start again at
    rest: the partials of the old velocities must not be counted because a
    capture has recorded, not run, the passes that would rewrite them."""
    monkeypatch.setenv("SNH_ENSEMBLE_BATCH", batch)
    members = [_made(_stretched(e, k)) for k, e in enumerate([(16, 8, 16), (9, 5, 13)])]
    for c in members:
        c.Execute(3)
        c.set_state(velocity=np.zeros((c.N, 3)))
        c.timestep_zero()
    ens = Ensemble(members, graph_steps=4, autotune=False)
    for c in members:
        before, after = _synced_twice(c)
        assert before == after
    ens.destroy()


@pytest.mark.parametrize("elements", [(16, 8, 16), (40, 20, 41)], ids=str)
def test_sync_after_autotune(elements):
    c = _made(_stretched(elements))
    c.Execute(5)
    c.autotune()
    before, after = _synced_twice(c)
    assert before == after


def _forms(kind, dt_type):
    out = []
    for k, e in enumerate([(6, 3, 6), (10, 4, 8), (7, 5, 14)]):
        p = _stretched(e, k)
        p.dtType = dt_type
        if dt_type == _abi.DT_CONSTANT:
            p.timeStep = 1.0e-3
        if kind == "two_materials":
            soft = P.MaterialSpec(rheology=_abi.RHEOLOGY_ELASTIC, alpha=0.0, beta=0.0, lam=1.0e10, mu=1.5e10,
                                  density=2700.0)
            p.materials = [p.materials[0], soft]
            mat = np.zeros(e[::-1], dtype=np.uint8)
            mat[:, :, e[0] // 2:] = 1
            p.element_material = mat.reshape(-1)
        out.append(p)
    return out


@pytest.mark.parametrize("dt_type", [_abi.DT_CONSTANT, _abi.DT_WAVE])
@pytest.mark.parametrize("kind", ["one_material", "two_materials"])
def test_batched_members_of_other_dt_types(kind, dt_type, monkeypatch):
    """The batched node pass in the form for every dt type."""
    monkeypatch.setenv("SNH_ENSEMBLE_BATCH", "1")
    fields = ("coord", "velocity", "stress")
    members = [_made(p) for p in _forms(kind, dt_type)]
    ens = Ensemble(members, graph_steps=4, autotune=False)
    assert ens.batched
    ens.step(8).synchronize()
    got = [c.state(fields=fields) for c in members]
    ens.destroy()
    for p, s in zip(_forms(kind, dt_type), got):
        c = _made(p)
        c.Execute(8)
        ref = c.state(fields=fields)
        for f in fields:
            assert np.array_equal(ref[f], s[f]), f
