"""Saving and restoring the state work on the system's device also while another one is current, as
the other state transfers do."""

import ctypes as C

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_save_and_restore_with_another_device_current():
    kyn = ota.KynLib()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime the library has loaded
    count, current = C.c_int(), C.c_int()
    assert hip.hipGetDeviceCount(C.byref(count)) == 0
    if count.value < 2:
        pytest.skip("needs two GPUs")
    spec = W.rotor_config_spec(num_nodes=6, num_qps=10, num_steps=2)
    s = ota.KynSystem(kyn, spec, exec_mode=ota.EXEC_FUSED)
    assert s.step({}) == ota.KYN_OK
    want = s.get("q")
    try:
        assert hip.hipSetDevice(1) == 0
        assert kyn.L.kyn_save_state(s.h) == ota.KYN_OK
        assert hip.hipGetDevice(C.byref(current)) == 0 and current.value == 1
        assert hip.hipSetDevice(0) == 0
        assert s.step({}) == ota.KYN_OK
        assert hip.hipSetDevice(1) == 0
        assert kyn.L.kyn_restore_state(s.h) == ota.KYN_OK
    finally:
        assert hip.hipSetDevice(0) == 0
    assert np.array_equal(s.get("q"), want)
