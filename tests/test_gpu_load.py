"""Slab packing and the final reductions at the edges of their tiles: K chunks of 16 that end in
VVVO, in T2 or past both, virtual blocks of one to sixteen real indices, the packed layout below, on
and above the diagonal, and tuple counts around the reduction's table of 256."""

import ctypes

import numpy as np
import pytest

from libcc_amd import CcxError, lib, synth
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


# no (no-1) (no+4) / 6 tuples, 2 (no=2) to 352 (no=12); the reduction takes its table 256 at a time, which
# lies between no=10 (210 tuples, one pass) and no=11 (275, two)
@pytest.mark.parametrize("no,nu", [(2, 15), (3, 16), (2, 17), (4, 30), (5, 31), (3, 33), (2, 47), (10, 5), (11, 5),
                                   (12, 18)], ids=lambda v: str(v))
def test_layouts_agree_and_match_oracle(no, nu):
    inp = synth.make_inputs(no, nu, 70 + no)
    full, packed = _solve(inp, False), _solve(inp, True)
    want = port.triples(inp)
    # the same slabs from either layout, so the same bits; the oracle sums in another order
    assert full["etd"] == packed["etd"] and full["ets"] == packed["ets"]
    assert np.array_equal(full["v1"], packed["v1"])
    assert abs(full["etd"] - want["etd"]) <= 1e-12 * abs(want["etd"])
    np.testing.assert_allclose(full["v1"], want["v1"], rtol=1e-10, atol=1e-12 * np.abs(want["v1"]).max())


def _same(got, want):
    return got["etd"] == want["etd"] and got["ets"] == want["ets"] and np.array_equal(got["v1"], want["v1"])


@pytest.mark.parametrize("on_device", [True, False], ids=["device", "host"])
def test_good_load_after_a_refused_one(on_device):
    """A refused input leaves the loaded problem as it was, and nothing that a load on another stream
    could meet."""
    import torch

    inp = synth.make_inputs(4, 36, 1001)
    bad = dict(inp, t2=np.array(inp["t2"], order="F"))
    bad["t2"][3, 5, 1, 2] = np.inf
    if on_device:
        # a device buffer of each array in Fortran order, kept until the end
        put = lambda d: {k: torch.from_numpy(np.asfortranarray(v).ravel(order="F").copy()).cuda()
                         for k, v in d.items() if isinstance(v, np.ndarray)}
        inp_l, bad_l = put(inp), put(bad)
    else:
        inp_l, bad_l = inp, bad
    want = _solve(inp, False)
    ctx = TriplesContext(4, 36)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for s in streams * 2:
        print(f"load refused, then good, stream {s.cuda_stream:#x}", flush=True)
        ctx.load(inp_l)
        with pytest.raises(CcxError) as err:
            ctx.load(bad_l)
        assert err.value.status == 5
        assert lib().ccx_set_stream(ctx._ctx, ctypes.c_void_p(s.cuda_stream)) == 0
        assert _same(ctx.energy(), want)
        ctx.load(inp_l)
        assert _same(ctx.energy(), want)
    ctx.close()


def test_upload_above_the_kept_bound():
    """no=2, nu=260 uploads 272 MiB, more than the 256 MiB buffer a context keeps: taken and given back by
    each load, with the same slabs as from device arrays."""
    import torch

    inp = synth.make_inputs(2, 260, 9)
    ctx = TriplesContext(2, 260)
    ctx.load({k: torch.from_numpy(np.asfortranarray(v).ravel(order="F").copy()).cuda()
              for k, v in inp.items() if isinstance(v, np.ndarray)})
    want = ctx.energy()
    for _ in range(2):
        print("host load no=2 nu=260", flush=True)
        ctx.load(inp)
        assert _same(ctx.energy(), want)
    ctx.close()
