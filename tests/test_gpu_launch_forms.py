"""Which launch a system takes: one workgroup per block of the fused step, and three per element of the
plain form, up to the sizes that fill the chip, and not one model or element beyond."""

import ctypes as C

import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kyn():
    return ota.KynLib()


def _launch(kyn, specs, **kw):
    s = ota.KynSystem(kyn, specs, **kw)
    out = [C.c_int() for _ in range(3)]
    assert kyn.L.kyn_debug_get_launch(s.h, *map(C.byref, out)) == ota.KYN_OK
    s.close()
    return [v.value for v in out]


@pytest.fixture(scope="module")
def cus(kyn):
    return _launch(kyn, W.cantilever_config_spec(num_steps=1))[2]


@pytest.mark.parametrize("precision,per_cu", [(ota.TANGENT_FP64, 1), (ota.TANGENT_FP32, 2)], ids=["fp64", "fp32"])
def test_fused_step_is_split_while_models_fit_the_chip(kyn, cus, precision, per_cu):
    spec = W.rotor_config_spec(num_nodes=3, num_qps=4)  # three blocks
    for models, workgroups in ((1, 3), (per_cu * cus, 3 * per_cu * cus), (per_cu * cus + 1, per_cu * cus + 1)):
        got = _launch(kyn, [spec] * models, exec_mode=ota.EXEC_FUSED, precision=precision)[0]
        assert got == workgroups, models


def test_plain_elements_are_split_while_they_fit_the_chip(kyn, cus):
    spec = W.cantilever_config_spec(num_steps=1)  # one element
    for elements, workgroups in ((1, 3), (cus // 3, 3), (cus // 3 + 1, 1)):
        assert _launch(kyn, [spec] * elements, exec_mode=ota.EXEC_PLAIN)[1] == workgroups, elements
    assert _launch(kyn, [spec], exec_mode=ota.EXEC_PLAIN, precision=ota.TANGENT_FP32)[1] == 1
