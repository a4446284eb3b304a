"""What the library's host code does where a one-GPU machine cannot show it:
other current devices, failures half way, several threads.  Runs the host code
itself on the CPU (hostlib.py); no kernel is executed."""
import ctypes
import os
import threading

import numpy as np
import pytest

import hostlib

P = ctypes.c_void_p


def ptr(a):
    return a.ctypes.data_as(P)


@pytest.fixture(scope="module")
def H(tmp_path_factory):
    h = hostlib.load(hostlib.build(str(tmp_path_factory.mktemp("hostlib"))))
    assert h.phf_init() == 0, h.phf_last_error()
    return h


@pytest.fixture(autouse=True)
def _clean(H):
    yield
    H.hr_on_launch(None)
    H.hr_fail(b"", -1)
    H.hr_pin_delay_us(0)
    H.hr_set_device(0)


def system(H, n, seed=0):
    """A system of n blobs and its arrays."""
    xyw = np.random.default_rng(seed).random((3, n))
    s = P()
    rc = H.phf_system_create(ptr(xyw[0]), ptr(xyw[1]), ptr(xyw[2]), ctypes.c_int64(n),
                             ctypes.byref(s))
    assert rc == 0, H.phf_last_error()
    return s, xyw


def get(H, s, n):
    out = np.zeros((3, n))
    rc = H.phf_system_get(s, ptr(out[0]), ptr(out[1]), ptr(out[2]))
    return rc, out


@pytest.mark.parametrize("n", [100, 300000])
def test_results_on_a_thread_of_another_device(H, n):
    """Results are fetched, in one packed transfer or through the pinned slots,
    whichever device the calling thread uses, and it stays that thread's."""
    s, xyw = system(H, n)
    for dev in (1, 0, 1):
        H.hr_set_device(dev)
        rc, out = get(H, s, n)
        assert rc == 0, (dev, H.phf_last_error())
        assert H.hr_device() == dev
        assert np.array_equal(out, xyw)
    assert H.phf_system_destroy(s) == 0
