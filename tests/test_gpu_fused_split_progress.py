"""A split model's step ends, with the same bits, whatever share of its workgroups finds room on the
GPU: launched with all of them, with one of each model (it then runs every block of the model) and
with numbers between; with more blocks than the rotors' three; past the 64 blocks and the 1024 iterations
a split model may have (one workgroup then); and with two systems stepping at once from threads."""

import ctypes as C
import threading

import numpy as np
import pytest

import openturbine_amd as ota
from openturbine_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("x", "q", "q_delta", "v", "vd", "a")
PRECISIONS = pytest.mark.parametrize("precision", [ota.TANGENT_FP64, ota.TANGENT_FP32], ids=["fp64", "fp32"])


@pytest.fixture(scope="module")
def kyn():
    return ota.KynLib()


def _joined(specs):
    """One model holding the given models' blades (blocks) and constraints."""
    beams, cons, off = [], [], 0
    for sp in specs:
        for b in sp.beams:
            beams.append(W.BeamSpec(np.asarray(b.nodes) + off, b.section_s, b.section_M, b.section_C, b.quad))
        for c in sp.constraints:
            cons.append(W.ConstraintSpec(c.type, c.base + off, c.target + off, c.axis, c.init))
        off += sp.num_nodes
    cat = [np.concatenate([getattr(sp, f) for sp in specs]) for f in ("x0", "u", "v", "vd", "s")]
    one = specs[0]
    return W.ModelSpec("joined", *cat, beams, cons, one.gravity, max_iter=one.max_iter, atol=one.atol, rtol=one.rtol)


def _rotors(sizes):
    return [W.rotor_config_spec(num_nodes=n, num_qps=max(3, 2 * n - 2), num_steps=3, seed=n) for n in sizes]


def _system(kyn, specs, precision):
    sweeps = 1 if precision == ota.TANGENT_FP32 else 0
    return ota.KynSystem(kyn, specs, exec_mode=ota.EXEC_FUSED, precision=precision, refine_sweeps=sweeps)


def _launched(kyn, s):
    fused = C.c_int()
    assert kyn.L.kyn_debug_get_launch(s.h, C.byref(fused), None, None) == ota.KYN_OK
    return fused.value


def _state(s):
    return [s.get(f) for f in FIELDS] + [s.totals()[0]] + [s.convergence(m) for m in range(s.num_models)]


@PRECISIONS
def test_any_number_of_started_workgroups_gives_the_same_bits(kyn, precision):
    # blocks: 3 + 9 + 3; the nine are of three sizes
    specs = [_rotors([4])[0], _joined(_rotors([3, 11, 6])), _rotors([8])[0]]
    want = None
    for per_model, groups in ((9, 15), (1, 3), (2, 6), (5, 11)):
        s = _system(kyn, specs, precision)
        assert _launched(kyn, s) == 15
        assert kyn.L.kyn_debug_set_fused_workgroups(s.h, per_model) == ota.KYN_OK
        assert _launched(kyn, s) == groups
        for k in range(2):
            assert s.step({}) == ota.KYN_OK
        assert kyn.L.kyn_step_many(s.h, 2, 1) == ota.KYN_OK
        got = _state(s)
        want = want or got
        for a, b in zip(got, want):
            assert np.array_equal(a, b), per_model
        s.close()


def test_a_model_needs_a_workgroup(kyn):
    s = _system(kyn, _rotors([3, 4]), ota.TANGENT_FP64)
    assert kyn.L.kyn_debug_set_fused_workgroups(s.h, 0) == ota.KYN_ERR_INVALID


def test_models_past_the_split_limit_keep_one_workgroup(kyn):
    few, many = _joined(_rotors([2] * 21)), _joined(_rotors([2] * 22))  # 63 and 66 blocks
    for spec, groups in ((few, 63), (many, 1)):
        s = _system(kyn, spec, ota.TANGENT_FP64)
        assert _launched(kyn, s) == groups
        assert s.step({}) == ota.KYN_OK
    q = [_system(kyn, sp, ota.TANGENT_FP64) for sp in (few, _rotors([2])[0])]
    for s in q:
        assert s.step({}) == ota.KYN_OK
    # 21 copies of one rotor converge as one (the error is a mean over the degrees of freedom)
    one = q[1].get("q")
    assert np.max(np.abs(q[0].get("q").reshape(21, -1) - one.reshape(1, -1))) <= 1e-12 * np.max(np.abs(one))


@pytest.mark.parametrize("max_iter,groups", [(1024, 3), (1025, 1), (1 << 24, 1)])
def test_an_iteration_limit_past_the_exchange_is_taken_unsplit(kyn, max_iter, groups):
    spec = _rotors([4])[0]
    s = ota.KynSystem(kyn, spec, exec_mode=ota.EXEC_FUSED, max_iter=max_iter)
    ref = ota.KynSystem(kyn, spec, exec_mode=ota.EXEC_FUSED)
    assert (_launched(kyn, s), _launched(kyn, ref)) == (groups, 3)
    for x in (s, ref):
        assert x.step({}) == ota.KYN_OK
    for a, b in zip(_state(s), _state(ref)):
        assert np.array_equal(a, b)


@PRECISIONS
def test_two_systems_stepping_at_once(kyn, precision):
    specs = [W.ensemble_config_specs(num_rotors=60, num_steps=3), [_joined(_rotors([3, 11, 6])), *_rotors([21, 5])]]
    want = []
    for sp in specs:
        s = _system(kyn, sp, precision)
        assert _launched(kyn, s) > s.num_models
        assert kyn.L.kyn_step_many(s.h, 3, 0) == ota.KYN_OK
        want.append(_state(s))
        s.close()
    both, rcs = [_system(kyn, sp, precision) for sp in specs], [None, None]

    def run(i):
        rcs[i] = kyn.L.kyn_step_many(both[i].h, 3, 0)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert rcs == [ota.KYN_OK, ota.KYN_OK]
    for s, w in zip(both, want):
        for a, b in zip(_state(s), w):
            assert np.array_equal(a, b)
