"""GPU parity of the Neo-Hookean tetrahedron kernels (A3) against the CPU oracle."""

import numpy as np
import pytest
import torch

from fenics_nonlinear_energies_amd.problems.hyperelasticity import (
    HEReorderedElementAssembler,
    build_beam_problem,
    problem_from_mesh,
    rotate_right_face_from_reference,
)
from oracle import assembly
from tests import fixtures

pytestmark = pytest.mark.gpu


def _state(p, u0, seed, amp=2e-4):
    return u0 + amp * np.random.default_rng(seed).standard_normal(u0.size)


@pytest.mark.parametrize("amode", ["staged", "rowgather"])
@pytest.mark.parametrize("absdet", [False, True])
def test_he_energy_gradient_hessian_fp64(require_gpu, absdet, amode):
    p, adj, u0 = build_beam_problem(16, 3, 3)
    asm = HEReorderedElementAssembler(p, None, adj, use_abs_det=absdet, assembly_mode=amode)
    u = _state(p, u0, 1)
    lay = asm.layout
    x = asm.create_vec(u[lay.perm])
    ref = assembly.assemble("he", p, u, dirichlet_key="u_0_ref", use_abs_det=absdet)
    assert abs(asm.energy_fn(x) - ref["e"]) <= 1e-12 * abs(ref["e"])
    g = x.duplicate()
    asm.gradient_fn(x, g)
    assert np.max(np.abs(g.array[lay.iperm] - ref["g"])) <= 1e-10 * np.max(np.abs(ref["g"]))
    asm.assemble_hessian(x)
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    assert abs(H - ref["h"]).max() <= 1e-11 * abs(ref["h"]).max()
    asm.cleanup()


@pytest.mark.parametrize("amode", ["staged", "rowgather"])
def test_he_fp32_hessian_and_rotated_face(require_gpu, amode):
    p, adj, u0 = build_beam_problem(20, 2, 2)
    asm = HEReorderedElementAssembler(p, None, adj, hessian_precision="fp32", assembly_mode=amode)
    u0_rot = rotate_right_face_from_reference(p["u_0_ref"], p["nodes2coord"], 0.3, p["right_nodes"])
    asm.update_dirichlet(u0_rot)
    pr = dict(p)
    pr["u_0_ref"] = u0_rot
    u = _state(p, u0, 2)
    x = asm.create_vec(u[asm.layout.perm])
    ref = assembly.assemble("he", pr, u, dirichlet_key="u_0_ref")
    assert abs(asm.energy_fn(x) - ref["e"]) <= 1e-12 * abs(ref["e"])
    asm.assemble_hessian(x)
    H = asm.A.to_scipy()[asm.layout.iperm][:, asm.layout.iperm]
    assert abs(H - ref["h"]).max() <= 2e-6 * abs(ref["h"]).max()
    h1 = asm.A.data.clone()
    asm.assemble_hessian(x)
    assert torch.equal(h1, asm.A.data)


def test_he_reference_mesh_element_eval(require_gpu):
    raw, adj = fixtures.he(1)
    from fenics_nonlinear_energies_amd.problems.hyperelasticity import problem_from_mesh

    p, a2, u0 = problem_from_mesh(raw["nodes2coord"], raw["elems2nodes"], float(raw["C1"]), float(raw["D1"]),
                                  dphi=(raw["dphix"], raw["dphiy"], raw["dphiz"], raw["vol"]))
    asm = HEReorderedElementAssembler(p, None, adj)
    u = _state(p, u0, 3)
    e, g, h = asm.element_eval(asm.create_vec(u[asm.layout.perm]))
    q = assembly.element_eval("he", p, assembly.local_state(p, u, "u_0_ref"))
    assert np.allclose(e.cpu().numpy(), q["e"], rtol=1e-11, atol=1e-12 * np.abs(q["e"]).max())
    assert np.allclose(g.cpu().numpy(), q["g"], rtol=1e-10, atol=1e-10 * np.abs(q["g"]).max())
    assert np.allclose(h.cpu().numpy(), q["h"], rtol=1e-10, atol=1e-10 * np.abs(q["h"]).max())


def test_he_nonpositive_jacobian_gives_nan_energy(require_gpu):
    """J <= 0 makes ln J non-finite; the energy is NaN/inf, never an error (line search repairs)."""
    p, adj, u0 = build_beam_problem(6, 1, 1)
    asm = HEReorderedElementAssembler(p, None, adj)
    u = u0.copy()
    u[0::3] *= -1.0  # mirror x: inverts every free-node element orientation
    E = asm.energy_fn(asm.create_vec(u[asm.layout.perm]))
    assert not np.isfinite(E)


class _RowGather(HEReorderedElementAssembler):
    node_patches = False


def _node_permutation(p, seed):
    """Free nodes in random order, components together: patches whose nodes share few elements."""
    n = p["freedofs"].size // 3
    return (3 * np.random.default_rng(seed).permutation(n)[:, None] + np.arange(3)).ravel()


def _fan(n):
    """Three axis edges joined to a ring of n vertices: edges with n tetrahedra (more than one
    block of items), axis nodes with 2 n."""
    t = 2 * np.pi * np.arange(n) / n
    axis = np.stack((np.zeros(4), np.zeros(4), np.arange(4.0)), 1)
    nodes = np.concatenate((axis, np.stack((np.cos(t), np.sin(t), 1.5 + 0 * t), 1)))
    k = np.arange(n)
    tets = [np.stack((0 * k + j, 0 * k + j + 1, 4 + k, 4 + (k + 1) % n), 1) for j in range(3)]
    return problem_from_mesh(nodes, np.concatenate(tets), 1.0, 2.0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,order,absdet", [
    ("fan", "block_morton", False),
    ((2, 1, 1), "block_morton", False),  # four free nodes, one patch
    ((6, 1, 1), "none", True),
    ((16, 3, 3), "random", False),
    ((30, 5, 4), "block_xyz", False),
    ((40, 9, 7), "block_morton", True),  # patches cut by their elements and by their nodes
])
def test_node_patches_match_row_gather(require_gpu, dims, order, absdet, precision):
    """The node-patch schedule against the row gather on the same plan arrays.  Both evaluate the same
    FP64 element formulas: a CSR value sums at most ~30 element values, so 1e-12 of the largest entry
    (2e-6 where the row gather sums in FP32); the energy 1e-12; the gradient's terms cancel, 1e-10 of
    its largest entry as against the oracle."""
    p, adj, u0 = _fan(30) if dims == "fan" else build_beam_problem(*dims)
    kw = dict(use_abs_det=absdet, hessian_precision=precision)
    kw.update({"perm_override": _node_permutation(p, 3)} if order == "random" else {"reorder_mode": order})
    u = _state(p, u0, 5, amp=0.05 if dims == "fan" else 2e-3 / max(dims[1:]))
    out = []
    for cls in (HEReorderedElementAssembler, _RowGather):
        asm = cls(p, None, adj, **kw)
        x = asm.create_vec(u[asm.layout.perm])
        asm._f_dev = torch.as_tensor(np.random.default_rng(7).standard_normal(u.size)).cuda()  # a load
        g, g2 = x.duplicate(), x.duplicate()
        asm.A.data.fill_(float("nan"))  # every entry is written
        e = float(asm.energy_grad_hessian_device(x.t, g.t).item())
        h = asm.A.data.clone()
        asm.gradient_fn(x, g2)
        assert torch.equal(g.t, g2.t)
        asm.A.data.fill_(float("nan"))
        asm.assemble_hessian(x)
        assert torch.equal(asm.A.data, h)
        out.append((e, g.t.cpu().numpy(), h.double().cpu().numpy()))
        asm.cleanup()
    (e, g, h), (e0, g0, h0) = out
    # an inverted element's energy is NaN (ln J) in either form
    assert abs(e - e0) <= 1e-12 * abs(e0) if np.isfinite(e0) else np.isnan(e) == np.isnan(e0)
    assert np.abs(g - g0).max() <= 1e-10 * np.abs(g0).max()
    assert np.abs(h - h0).max() <= (1e-12 if precision == "fp64" else 2e-6) * np.abs(h0).max()


def test_node_patches_leave_mixed_orders_to_the_row_gather(require_gpu):
    """Components of one node apart: no 3x3 blocks in the CSR rows, the plan keeps the row gather."""
    p, adj, u0 = build_beam_problem(8, 2, 2)
    perm = np.random.default_rng(2).permutation(u0.size)
    out = []
    for cls in (HEReorderedElementAssembler, _RowGather):
        asm = cls(p, None, adj, perm_override=perm)
        x = asm.create_vec(_state(p, u0, 4)[perm])
        asm.assemble_hessian(x)
        out.append(asm.A.data.clone())
        asm.cleanup()
    assert torch.equal(*out)


@pytest.mark.parametrize("dims,amp", [((6, 2, 2), 1e-4), ((6, 2, 2), 1e-7), ((40, 9, 7), 1e-6)])
def test_fused_energy_is_the_separate_one_near_rest(require_gpu, dims, amp):
    """Near rest an element's energy is the difference of terms of size C1, so its rounding is relative
    to those and not to the energy.  The fused call and fne_energy round every element alike and add
    up with compensation: equal to the last two bits each, 4 eps."""
    p, adj, u0 = build_beam_problem(*dims)
    asm = HEReorderedElementAssembler(p, None, adj)
    rest = np.asarray(p["nodes2coord"]).reshape(-1)[np.asarray(p["freedofs"])]
    u = rest + amp * np.random.default_rng(1).standard_normal(rest.size) / max(dims[1:])
    x = asm.create_vec(u[asm.layout.perm])
    asm.dvals.copy_(torch.as_tensor(np.asarray(p["nodes2coord"]).reshape(-1)))
    e = float(asm.energy_device(x.t).item())
    g = x.duplicate()
    fused = float(asm.energy_grad_hessian_device(x.t, g.t).item())
    print("near rest", dims, amp, e, fused - e, flush=True)
    assert np.isfinite(e) and abs(fused - e) <= 4 * np.finfo(float).eps * abs(e)
    asm.cleanup()


@pytest.mark.parametrize("cls", [HEReorderedElementAssembler, _RowGather])
def test_energy_of_a_beam_with_an_inverted_element(require_gpu, cls):
    """Admissible states have a finite energy, the same in the fused and the separate call; with det F < 0
    in one element it is NaN (ln J) without |det F| and finite with it."""
    p, adj, u0 = build_beam_problem(12, 3, 3)
    u = _state(p, u0, 5, amp=2e-4)
    for turned in (False, True):
        v = u.copy()
        if turned:  # one node moved through its neighbours' faces
            v[3 * (u.size // 6):][:3] += [0.2, 0.0, 0.0]
        for absdet in (False, True):
            asm = cls(p, None, adj, use_abs_det=absdet)
            x = asm.create_vec(v[asm.layout.perm])
            g = x.duplicate()
            both = [float(asm.energy_device(x.t).item()), float(asm.energy_grad_hessian_device(x.t, g.t).item())]
            if turned and not absdet:
                assert np.isnan(both).all()
            else:
                assert np.isfinite(both).all() and abs(both[0] - both[1]) <= 4 * np.finfo(float).eps * abs(both[0])
            asm.cleanup()
