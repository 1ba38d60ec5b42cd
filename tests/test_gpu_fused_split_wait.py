"""The split fused step's wait between workgroups has a bound: a step in which it is reached (here at
the first wait, by a negative bound) ends with an error, alone and among the steps of one call, with
and without a graph, and after a restore the same system steps on with the bits it has without."""

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("x", "q", "q_delta", "v", "vd", "a")


@pytest.mark.parametrize("precision", [ota.TANGENT_FP64, ota.TANGENT_FP32], ids=["fp64", "fp32"])
def test_peer_wait_bound_gives_up_and_reports(precision):
    kyn = ota.KynLib()
    # mixed blade sizes: the small blades' workgroups wait for the large ones'
    specs = W.ensemble_config_specs(num_rotors=6, num_steps=8)
    cd, tips, loads = W.ensemble_schedule(specs, 8)
    s, ref = (ota.KynSystem(kyn, specs, exec_mode=ota.EXEC_FUSED, precision=precision) for _ in range(2))
    for x in (s, ref):
        x.set_schedule(8, cd, tips, loads)
        assert kyn.L.kyn_step_many(x.h, 2, 1) == ota.KYN_OK
        assert kyn.L.kyn_save_state(x.h) == ota.KYN_OK
        assert kyn.L.kyn_step_many(x.h, 2, 1) == ota.KYN_OK
    assert kyn.L.kyn_debug_set_peer_wait_limit(s.h, -1) == ota.KYN_OK
    for call in (lambda: kyn.L.kyn_step(s.h), lambda: kyn.L.kyn_step_many(s.h, 3, 0),
                 lambda: kyn.L.kyn_step_many(s.h, 3, 1)):
        assert call() == ota.KYN_ERR_HIP
        assert "other blocks of its model" in kyn.error()
    assert kyn.L.kyn_debug_set_peer_wait_limit(s.h, 1 << 24) == ota.KYN_OK
    for x in (s, ref):
        assert kyn.L.kyn_restore_state(x.h) == ota.KYN_OK
        assert kyn.L.kyn_step(x.h) == ota.KYN_OK
        assert kyn.L.kyn_step_many(x.h, 3, 1) == ota.KYN_OK
    for f in FIELDS:
        assert np.array_equal(s.get(f), ref.get(f)), f
    for m in range(len(specs)):
        assert np.array_equal(s.convergence(m), ref.convergence(m))
