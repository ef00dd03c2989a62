"""snh_autotune keeps the fastest element layout and node pass of those that
it has timed, also where two layouts lie within a few percent of each other."""
import pytest

from snac_amd import Context, problem as P

pytestmark = pytest.mark.gpu

NAMES = ["elem_ms_tet_per_lane", "elem_ms_element_per_lane", "elem_ms_element_per_lane_lowreg", "elem_ms_tet_per_wave"]


@pytest.mark.parametrize("elements", [(128, 54, 128), (96, 48, 96), (20, 10, 20)], ids=str)
def test_the_fastest_is_kept(elements, monkeypatch):
    monkeypatch.delenv("SNH_ELEM_VARIANT", raising=False)
    c = Context(P.mohr_coulomb_extension(elements=elements)).Construct().Build().Initialise()
    c.Execute(5)
    rep = c.autotune()
    print(f"  {rep}", flush=True)
    ms = [rep[n] for n in NAMES]
    assert ms[rep["elem_variant"]] == min(ms)
    c.Destroy()
