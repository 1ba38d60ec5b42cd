"""The fused launch's list: one workgroup per block while the models leave the chip idle, one per
model beyond that.  Both give a model the same bits, so a model of a small ensemble (split) is
compared with the same model inside one too large to split; models of one, two and three blocks
(rotors with blades taken off) likewise."""

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("x", "q", "q_delta", "v", "vd", "a")


@pytest.fixture(scope="module")
def kyn():
    return ota.KynLib()


def _run(kyn, specs, steps, precision):
    sweeps = 1 if precision == ota.TANGENT_FP32 else 0
    s = ota.KynSystem(kyn, specs, exec_mode=ota.EXEC_FUSED, precision=precision, refine_sweeps=sweeps)
    cd, tips, loads = W.ensemble_schedule(specs, steps)
    s.set_schedule(steps, cd, tips, loads)
    assert s.step_many(1, use_graph=False) == ota.KYN_OK
    assert s.step_many(steps - 1, use_graph=True) == ota.KYN_OK
    return s


@pytest.mark.parametrize("precision,many", [(ota.TANGENT_FP64, 260), (ota.TANGENT_FP32, 520)], ids=["fp64", "fp32"])
def test_split_and_unsplit_launches_agree_bit_for_bit(kyn, precision, many):
    steps = 3
    specs = W.ensemble_config_specs(num_rotors=many, num_steps=steps)
    few = 4
    a, b = _run(kyn, specs[:few], steps, precision), _run(kyn, specs, steps, precision)
    nodes = sum(sp.num_nodes for sp in specs[:few])
    for f in FIELDS:
        assert np.array_equal(a.get(f), b.get(f)[:nodes]), f
    assert np.array_equal(a.totals()[0], b.totals()[0][:few])
    for m in range(few):
        assert np.array_equal(a.convergence(m), b.convergence(m))


def _without_blades(spec, keep):
    """The rotor with its first `keep` blades (their nodes come first, one constraint each)."""
    n = sum(len(b.nodes) for b in spec.beams[:keep])
    return W.ModelSpec(spec.name, spec.x0[:n], spec.u[:n], spec.v[:n], spec.vd[:n], spec.s[:n], spec.beams[:keep],
                       spec.constraints[:keep], spec.gravity)


def test_models_of_one_two_and_three_blocks(kyn):
    rotors = [W.rotor_config_spec(num_nodes=n, num_qps=2 * n - 2, num_steps=3, seed=n) for n in (5, 21, 8)]
    specs = [_without_blades(rotors[0], 1), rotors[1], _without_blades(rotors[2], 2)]
    filler = [_without_blades(rotors[0], 1)] * 260
    out = []
    for sp in (specs, specs + filler):
        s = ota.KynSystem(kyn, sp, exec_mode=ota.EXEC_FUSED)
        for k in range(3):
            assert s.step() == ota.KYN_OK
        out.append(s)
    nodes = sum(sp.num_nodes for sp in specs)
    for f in FIELDS:
        assert np.array_equal(out[0].get(f), out[1].get(f)[:nodes]), f
    for m in range(len(specs)):
        assert np.array_equal(out[0].convergence(m), out[1].convergence(m))
