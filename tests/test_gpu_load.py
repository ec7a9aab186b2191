"""Slab packing and the final reductions at the edges of their tiles: K chunks of 16 that end in
VVVO, in T2 or past both, virtual blocks of one to sixteen real indices, the packed layout below, on
and above the diagonal, and tuple counts around the reduction's table of 256."""

import numpy as np
import pytest

from libcc_amd import synth
from libcc_amd.triples import TriplesContext
from oracle import port

pytestmark = pytest.mark.gpu


def _solve(inp, packed):
    ctx = TriplesContext(inp["no"], inp["nu"])
    try:
        ctx.load(dict(inp, vvvo=synth.pack_vvvo(inp["vvvo"])) if packed else inp, packed_vvvo=packed)
        return ctx.energy()
    finally:
        ctx.close()


# no (no-1) (no+4) / 6 tuples: 2 .. 270, 256 lying between no=11 and no=12's 275
@pytest.mark.parametrize("no,nu", [(2, 15), (3, 16), (2, 17), (4, 30), (5, 31), (3, 33), (2, 47), (11, 5), (12, 18)],
                         ids=lambda v: str(v))
def test_layouts_agree_and_match_oracle(no, nu):
    inp = synth.make_inputs(no, nu, 70 + no)
    full, packed = _solve(inp, False), _solve(inp, True)
    want = port.triples(inp)
    # the same slabs from either layout, so the same bits; the oracle sums in another order
    assert full["etd"] == packed["etd"] and full["ets"] == packed["ets"]
    assert np.array_equal(full["v1"], packed["v1"])
    assert abs(full["etd"] - want["etd"]) <= 1e-12 * abs(want["etd"])
    np.testing.assert_allclose(full["v1"], want["v1"], rtol=1e-10, atol=1e-12 * np.abs(want["v1"]).max())
