"""Saving and restoring the state work on the system's device also while another one is current, as
the other state transfers do."""

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_save_and_restore_with_another_device_current():
    torch = pytest.importorskip("torch")
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    kyn = ota.KynLib()
    spec = W.rotor_config_spec(num_nodes=6, num_qps=10, num_steps=2)
    with torch.cuda.device(0):
        s = ota.KynSystem(kyn, spec, exec_mode=ota.EXEC_FUSED)
        assert s.step({}) == ota.KYN_OK
    want = s.get("q")
    with torch.cuda.device(1):
        assert kyn.L.kyn_save_state(s.h) == ota.KYN_OK
        assert torch.cuda.current_device() == 1
    with torch.cuda.device(0):
        assert s.step({}) == ota.KYN_OK
    with torch.cuda.device(1):
        assert kyn.L.kyn_restore_state(s.h) == ota.KYN_OK
    assert np.array_equal(s.get("q"), want)
