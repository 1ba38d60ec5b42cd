"""The blocked LU at the sizes where its tiling can go wrong, against the oracle's solve of the same
matrix: blocks of one panel (12, 18 dofs), a last panel of 2 to 16 columns, one, two and three
candidate rows per lane (to 64, 128 and 143), up to seven column tiles (the largest blocks), in the fused
and the plain form.  One Newton iteration, so that the increment is one solve; the bounds are the ones
the parity tests hold final states to (of the largest value): q 1e-12, v 1e-10, vd 1e-9, the rates
carrying the increment times gamma' and beta' (1.8e2 and 3.6e4 at this step size)."""

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W
from oracle_lib import OracleLib, OracleSystem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kyn():
    return ota.KynLib()


@pytest.fixture(scope="module")
def orc():
    return OracleLib()


@pytest.mark.parametrize("mode", [ota.EXEC_FUSED, ota.EXEC_PLAIN], ids=["fused", "plain"])
@pytest.mark.parametrize("nodes", [2, 3, 4, 7, 9, 10, 12, 15, 17, 18, 20, 21])
def test_one_newton_iteration_solves_as_the_oracle(kyn, orc, nodes, mode):
    spec = W.rotor_config_spec(num_nodes=nodes, num_qps=max(2, 2 * nodes - 2), num_steps=1, max_iter=1, seed=nodes)
    g, o = ota.KynSystem(kyn, spec, exec_mode=mode), OracleSystem(orc, spec)
    inputs = spec.step_inputs(0)
    g.step(inputs)
    o.step(inputs)
    for f, bar in (("q", 1e-12), ("v", 1e-10), ("vd", 1e-9)):
        a, b = g.get(f), o.get(f)
        assert np.max(np.abs(a - b)) <= bar * max(np.max(np.abs(b)), 1.0), f
