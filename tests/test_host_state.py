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

    def __init__(self, host, no, nu):
        self.host, self.no, self.nu = host, no, nu
        inp = synth.make_inputs(no, nu, 1)
        self.arrays = {k: np.asfortranarray(inp[k]).ravel(order="F").copy() for k in KEYS}
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
