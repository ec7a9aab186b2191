"""State that a context of the C host layer keeps between calls, on a stand-in for the device layer
(fake_dev.c: host memory with a budget, no kernels), so that failing calls, full devices and queued
work can be had without a GPU."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

from libcc_amd import synth

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "libcc_amd", "csrc")
OK, ERR_DEVICE, ERR_ALLOC, ERR_INPUT = 0, 2, 3, 5
KEYS = ("eh", "ep", "t1", "t2", "vm", "voe", "vvvo")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host_layer.so")
    subprocess.run(["gcc", "-O1", "-g", "-shared", "-fPIC", "-w", "-pthread", f"-I{CSRC}", os.path.join(CSRC, "ccx_host.c"),
                    os.path.join(HERE, "fake_dev.c"), "-o", so, "-lm"], check=True)
    return ctypes.CDLL(so)


class Ctx:
    """A context of the stand-in build and its inputs."""

    def __init__(self, host, no, nu, arrays=None):
        self.host, self.no, self.nu = host, no, nu
        if arrays is None:
            inp = synth.make_inputs(no, nu, 1)
            arrays = {k: np.asfortranarray(inp[k]).ravel(order="F").copy() for k in KEYS}
        self.arrays = arrays
        self.p = ctypes.c_void_p()
        assert host.ccx_create(ctypes.c_int64(no), ctypes.c_int64(nu), ctypes.byref(self.p)) == OK

    def load(self, on_device=True):
        fn = self.host.ccx_load_device if on_device else self.host.ccx_load_host
        return fn(self.p, *[ctypes.c_void_p(self.arrays[k].ctypes.data) for k in KEYS], 0)

    def stream(self, n):
        assert self.host.ccx_set_stream(self.p, ctypes.c_void_p(n)) == OK

    def energy(self, form=0):
        return self.host.ccx_energy(self.p, form, None, None, None, 0)

    def close(self):
        assert self.host.ccx_destroy(self.p) == OK


@pytest.fixture
def ctx(host):
    c = Ctx(host, 3, 20)
    yield c
    c.close()


def _fail(host, name, n=1):
    ctypes.c_int.in_dll(host, name).value = n


def test_good_load_after_a_bad_one_on_another_stream(ctx):
    """The clearing of the flag must not be left queued on the stream of the refused load."""
    ctx.stream(0x10)
    ctx.arrays["t2"][7] = np.nan
    assert ctx.load() == ERR_INPUT
    ctx.arrays["t2"][7] = 0.25
    ctx.stream(0x20)
    assert ctx.load() == OK
    assert ctx.energy() == OK


def test_good_load_after_a_scan_that_failed(host, ctx):
    """A scan that fails after it set the flag (its result could not be fetched) leaves no trace."""
    assert ctx.load() == OK
    _fail(host, "fake_fail_scan")
    assert ctx.load() == ERR_DEVICE
    assert ctx.load() == OK


def test_good_load_after_the_first_clearing_failed(host, ctx):
    _fail(host, "fake_fail_zero_flag")
    assert ctx.load() == ERR_DEVICE
    assert ctx.load() == OK


@pytest.mark.parametrize("on_device", [True, False])
def test_bad_load_keeps_the_problem_that_was_loaded(ctx, on_device):
    assert ctx.load(on_device) == OK
    ctx.arrays["vvvo"][-1] = np.inf
    assert ctx.load(on_device) == ERR_INPUT
    assert ctx.energy() == OK


def _room(host, value=None):
    room = ctypes.c_longlong.in_dll(host, "fake_room")
    if value is not None:
        room.value = value
    return room.value


@pytest.fixture
def small_batch(monkeypatch):
    monkeypatch.setenv("CCX_ADJ_BATCH_MB", "8")


def _gradient(c, outputs=False):
    outs = [None] * 5
    if outputs:
        outs = [np.zeros(c.arrays[k].size) for k in ("t1", "t2", "vm", "voe", "vvvo")]
    return c.host.ccx_gradient(c.p, None, None, *[None if a is None else ctypes.c_void_p(a.ctypes.data) for a in outs], 0)


def _gradient_workspace(c):
    """bytes the context keeps after a gradient"""
    before = _room(c.host)
    assert _gradient(c) == OK
    return before - _room(c.host)


@pytest.fixture
def full_device(host, small_batch):
    """full_device(n) leaves n bytes of the device free: the rest is someone else's."""
    yield lambda n: _room(host, n)
    _room(host, ctypes.c_longlong.in_dll(host, "fake_total").value)


@pytest.mark.parametrize("what", ["fp32", "bf16x3", "virtual", "tuple_w", "gradient_outputs"])
def test_kept_memory_is_given_back_to_the_same_context(host, full_device, what):
    """Whatever fits a device on which no gradient has run fits it after one: the kept workspace and
    upload buffer go back when an allocation fails."""
    c = Ctx(host, 3, 40)
    assert c.load(on_device=False) == OK      # leaves an upload buffer
    assert _gradient_workspace(c) > 0
    full_device(1000)
    etd, w = ctypes.c_double(), np.zeros(c.nu ** 3)
    if what == "gradient_outputs":            # its own workspace is in use: the upload buffer must do
        rc = _gradient(c, outputs=True)
    elif what == "virtual":
        rc = host.ccx_energy_abc(c.p, ctypes.byref(etd))
    elif what == "tuple_w":
        rc = host.ccx_tuple_w(c.p, ctypes.c_int64(3), ctypes.c_int64(2), ctypes.c_int64(1), ctypes.c_void_p(w.ctypes.data))
    else:
        rc = c.energy({"fp32": 1, "bf16x3": 2}[what])
    assert rc == OK
    c.close()


def test_kept_memory_is_given_back_to_another_context(host, full_device):
    a, b = Ctx(host, 3, 40), Ctx(host, 2, 20)
    assert a.load() == OK
    kept = _gradient_workspace(a)
    full_device(1000)
    assert b.load() == OK
    assert _room(host) > kept // 2
    full_device(1 << 40)
    assert _gradient(a) == OK                 # takes its workspace anew
    a.close()
    b.close()


def test_workspace_in_use_is_not_given_back(host, full_device):
    """Another thread's allocation fails while a gradient runs: that gradient keeps its memory."""
    a, b = Ctx(host, 3, 40), Ctx(host, 2, 20)
    assert a.load() == OK
    assert _gradient(a) == OK
    got = []

    @ctypes.CFUNCTYPE(None)
    def during():
        room = _room(host)
        _room(host, 1000)
        got.append((b.load(), _room(host)))
        _room(host, room)

    hook = ctypes.c_void_p.in_dll(host, "fake_during_adjoint")
    hook.value = ctypes.cast(during, ctypes.c_void_p).value
    try:
        assert _gradient(a) == OK
    finally:
        hook.value = None
    assert got and all(rc == ERR_ALLOC and room <= 1000 for rc, room in got)
    a.close()
    b.close()


def test_workspace_is_kept_only_while_half_the_device_is_free(host, full_device):
    c = Ctx(host, 3, 40)
    assert c.load() == OK
    total = ctypes.c_longlong.in_dll(host, "fake_total").value
    kept = _gradient_workspace(c)
    assert kept > 0
    room = full_device(total // 2 - 1)
    assert _gradient(c) == OK
    assert _room(host) == room + kept
    full_device(total // 2 + kept)
    assert _gradient_workspace(c) == kept
    c.close()


def test_workspace_grows_with_the_batch(host, monkeypatch, full_device):
    c = Ctx(host, 4, 36)
    assert c.load() == OK
    kept = []
    before = _room(host)
    for mb in ("1", "4", "2", "64"):
        monkeypatch.setenv("CCX_ADJ_BATCH_MB", mb)
        assert _gradient(c) == OK
        kept.append(before - _room(host))
    assert kept[0] < kept[1] == kept[2] < kept[3]
    c.close()
    assert _room(host) >= before


@pytest.mark.parametrize("nu,keeps", [(20, True), (260, False)], ids=["small", "272MiB"])
def test_upload_buffer_is_kept_up_to_its_bound(host, nu, keeps):
    """The buffer of no=2, nu=260 is above the bound of 256 MiB: given back by every load."""
    sizes = {"eh": 2, "ep": nu, "t1": 2 * nu, "t2": 4 * nu ** 2, "vm": 8 * nu, "voe": 4 * nu ** 2, "vvvo": 2 * nu ** 3}
    c = Ctx(host, 2, nu, {k: np.zeros(n) for k, n in sizes.items()})
    assert c.load() == OK                     # every buffer but the upload's is there now
    before = _room(host)
    for _ in range(2):
        assert c.load(on_device=False) == OK
        assert (_room(host) < before) == keeps
    c.close()


@pytest.mark.parametrize("no,packed", [(1, 0), (2, 0), (3, 1)])
def test_virtual_triple_route(host, no, packed):
    """The matrix cores take 16 occupied indices at a time: not for one (whose cubes are their one
    zeroed element) or two."""
    c = Ctx(host, no, 20)
    assert c.load() == OK
    routes, etd = ctypes.c_int.in_dll(host, "fake_packed_routes"), ctypes.c_double()
    before = routes.value
    assert host.ccx_energy_abc(c.p, ctypes.byref(etd)) == OK
    assert routes.value - before == packed
    c.close()
