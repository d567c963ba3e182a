"""Golden-section line search on the device against the host search.

DeviceGoldenSearch runs the search of core/petsc/minimizers.py:14-64 as a device state
machine (fne_golden_trial / fne_energy / fne_golden_step).  With the energies of the same
trial points it must choose the same alpha after the same number of energies as
minimizers.golden_section_search, including a bracket narrower than the tolerance; and a
Newton solve must follow the same path with either search.
"""

import numpy as np
import pytest
import torch

from fenics_nonlinear_energies_amd.drivers import DeviceGoldenSearch, solve_newton
from fenics_nonlinear_energies_amd.minimizers import golden_section_search
from fenics_nonlinear_energies_amd.problems.plaplace import PLaplaceReorderedElementAssembler, build_plaplace_problem

pytestmark = pytest.mark.gpu


def _asm():
    p, adj, _ = build_plaplace_problem(32)
    return PLaplaceReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="jacobi")


@pytest.mark.parametrize("lo,hi,tol", [(-0.5, 2.0, 1e-3), (-0.5, 2.0, 1e-6), (0.1, 0.1005, 1e-3), (0.0, 1.0, 1e-2)])
def test_device_golden_matches_host(require_gpu, lo, hi, tol):
    asm = _asm()
    rng = np.random.default_rng(11)
    x = asm.create_vec(rng.random(asm.layout.n_free))
    d = asm.create_vec(-0.5 * rng.random(asm.layout.n_free))
    trial = torch.empty_like(x.t)

    def f(a):
        torch.add(x.t, d.t, alpha=a, out=trial)
        return float(asm.energy_device(trial).item())

    a_h, n_h = golden_section_search(f, lo, hi, tol)
    a_d, f_d, n_d = DeviceGoldenSearch(asm)(x, d, lo, hi, tol)
    assert n_d == n_h
    assert abs(a_d - a_h) <= 1e-12 * max(1.0, abs(a_h))
    assert f_d == pytest.approx(f(a_d), rel=1e-13)
    asm.cleanup()


def test_newton_same_path_with_device_linesearch(require_gpu):
    res = {}
    for dev in (False, True):
        asm = _asm()
        x = asm.create_vec(np.zeros(asm.layout.n_free))
        r = solve_newton(asm, x, ksp_rtol=1e-6, device_linesearch=dev, first_step_laplacian=True, tolg=1e-8,
                         tolf=0.0, maxit=60)
        res[dev] = (r["nit"], r["fun"])
        asm.cleanup()
    assert res[True][0] == res[False][0]
    assert res[True][1] == pytest.approx(res[False][1], rel=1e-13)


def _he_asm():
    from fenics_nonlinear_energies_amd.problems.hyperelasticity import HEReorderedElementAssembler, build_beam_problem

    p, adj, u0 = build_beam_problem(6, 2, 2)
    asm = HEReorderedElementAssembler(p, None, adj)
    return asm, np.asarray(u0)[asm.layout.perm], 1e-4


def _mc_asm():
    from fenics_nonlinear_energies_amd.problems.slope_stability import SlopeStabilityReorderedElementAssembler
    from tests.test_oracle_mc import mc_params

    p, adj = mc_params(h=4.0, degree=2, lam=1.2)
    asm = SlopeStabilityReorderedElementAssembler(p, None, adj)
    return asm, np.zeros(asm.layout.n_free), 1e-2


def _p1_asm():
    asm = _asm()
    return asm, np.random.default_rng(1).random(asm.layout.n_free), 0.5


@pytest.mark.parametrize("make", [_p1_asm, _he_asm, _mc_asm])
def test_search_in_one_call_equals_point_by_point(require_gpu, make):
    """fne_golden_search against fne_golden_trial / fne_energy / fne_golden_step per point, and resumed two points at a
    time: the same energies up to the order of their sums, so the same points."""
    asm, x0, amp = make()
    x = asm.create_vec(x0)
    d = asm.create_vec(amp * np.random.default_rng(3).standard_normal(x0.size))
    one, each = DeviceGoldenSearch(asm), DeviceGoldenSearch(asm)
    assert one._native
    each._native = False
    got, ref = one(x, d, -0.5, 2.0, 1e-4), each(x, d, -0.5, 2.0, 1e-4)
    assert got[2] == ref[2]
    assert abs(got[0] - ref[0]) <= 1e-12 and got[1] == pytest.approx(ref[1], rel=1e-13)
    steps = DeviceGoldenSearch(asm)
    steps._points(x.t, d.t, (-0.5, 2.0, 1e-4), 2, False)
    for _ in range(40):
        steps._points(x.t, d.t, (-0.5, 2.0, 1e-4), 2, True)
    st = steps.state.cpu().numpy()
    assert st[11] == 7.0 and (float(st[8]), float(st[9]), int(st[12])) == got
    asm.cleanup()


def test_search_calls_an_energy_set_on_the_instance(require_gpu):
    """A counter put over one assembler's energy_device sees every point, also when it is put there after
    the search was made, and the search is the same."""
    asm, x0, amp = _p1_asm()
    x = asm.create_vec(x0)
    d = asm.create_vec(amp * np.random.default_rng(3).standard_normal(x0.size))
    search = DeviceGoldenSearch(asm)
    ref = search(x, d, -0.5, 2.0, 1e-3)
    plain, calls = asm.energy_device, []

    def counted(*args, **kw):
        calls.append(1)
        return plain(*args, **kw)

    asm.energy_device = counted
    for s in (search, DeviceGoldenSearch(asm)):
        calls.clear()
        got = s(x, d, -0.5, 2.0, 1e-3)
        assert len(calls) >= got[2] == ref[2]
        assert abs(got[0] - ref[0]) <= 1e-12 and got[1] == pytest.approx(ref[1], rel=1e-13)
    del asm.energy_device
    calls.clear()
    assert search(x, d, -0.5, 2.0, 1e-3) == ref and not calls
    asm.cleanup()
