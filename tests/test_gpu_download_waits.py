"""Every entry point that returns host-visible values has synchronised the
context's stream when it returns: a state download also when none of the
fields asked for is held on the device."""
import ctypes as C

import pytest
import torch

from snac_amd import Context, problem as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fields", [("plastic_strain",), ("viscosity",), (), ("coord",)], ids=str)
def test_download_waits_for_the_stream(fields):
    """An elastic context holds neither plastic strain nor viscosity: both
    come back as zeros filled in on the host."""
    s = torch.cuda.Stream()
    c = Context(P.elastic_box_compression(elements=(64, 32, 64))).Construct().Build().Initialise()
    c._check(c.lib.snh_set_stream(c.h, C.c_void_p(s.cuda_stream)))
    c.Execute(2)
    c.step(400)
    got = c.state(fields=fields)
    assert s.query(), "work of the steps was still in flight"
    for f in fields:
        if f != "coord":
            assert not got[f].any()
    c.Destroy()
