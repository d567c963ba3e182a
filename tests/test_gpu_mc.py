"""GPU parity of the Mohr-Coulomb P2/P4 kernels against the CPU oracle.

Tolerances: FP64 mode -- energy 1e-12 relative, gradient 1e-11 and Hessian 1e-10 of their
largest entry (MFMA FP64 sums in another order than numpy).  FP32 Hessian -- 3e-5 of the
largest entry (FP32 MFMA accumulation over 2 n_q = 38 products).
"""

import numpy as np
import pytest
import scipy.sparse as sp
import torch

from fenics_nonlinear_energies_amd.problems.slope_stability import SlopeStabilityReorderedElementAssembler
from oracle import assembly
from tests.test_oracle_mc import mc_params

pytestmark = pytest.mark.gpu


def _state(p, lay, seed, scale=2e-3):
    rng = np.random.default_rng(seed)
    X = p["nodes"]
    v = np.zeros(2 * X.shape[0])
    v[0::2] = scale * X[:, 1] + 0.05 * scale * rng.standard_normal(X.shape[0])
    v[1::2] = -0.5 * scale * X[:, 1] + 0.05 * scale * rng.standard_normal(X.shape[0])
    return v[p["freedofs"]]


@pytest.mark.parametrize("degree", [4, 2])
def test_element_eval_matches_oracle(require_gpu, degree):
    p, adj = mc_params(h=4.0, degree=degree, lam=1.5)
    asm = SlopeStabilityReorderedElementAssembler(p, None, adj, hessian_precision="fp64")
    u = _state(p, asm.layout, 1)
    e, g, h = asm.element_eval(asm.create_vec(u[asm.layout.perm]))
    v = assembly.local_state(p, u)
    q = assembly.element_eval("mc", p, v)
    e, g, h = e.cpu().numpy(), g.cpu().numpy(), h.cpu().numpy()  # original element order
    assert np.allclose(e, q["e"], rtol=1e-12, atol=1e-12 * np.abs(q["e"]).max())
    assert np.abs(g - q["g"]).max() <= 1e-11 * np.abs(q["g"]).max()
    assert np.abs(h - q["h"]).max() <= 1e-10 * np.abs(q["h"]).max()
    asm.cleanup()


@pytest.mark.parametrize("degree", [4, 2])
def test_assembly_fp64_matches_oracle(require_gpu, degree):
    p, adj = mc_params(h=4.0, degree=degree, lam=1.5)
    asm = SlopeStabilityReorderedElementAssembler(p, None, adj, hessian_precision="fp64")
    lay = asm.layout
    u = _state(p, lay, 2)
    ref = assembly.assemble("mc", p, u)
    x = asm.create_vec(u[lay.perm])
    E = asm.energy_fn(x)
    assert abs(E - ref["e"]) <= 1e-12 * abs(ref["e"])
    g = x.duplicate()
    asm.gradient_fn(x, g)
    assert np.abs(g.array[lay.iperm] - ref["g"]).max() <= 1e-11 * np.abs(ref["g"]).max()
    asm.assemble_hessian(x)
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    assert abs(H - ref["h"]).max() <= 1e-10 * abs(ref["h"]).max()
    # deterministic: bitwise identical on a second assembly
    v1 = asm.A.data.clone()
    asm.assemble_hessian(x)
    assert torch.equal(v1, asm.A.data)
    asm.cleanup()


def test_fp32_hessian_and_fused_call(require_gpu):
    p, adj = mc_params(h=4.0, degree=4, lam=1.5)
    asm = SlopeStabilityReorderedElementAssembler(p, None, adj, hessian_precision="fp32")
    lay = asm.layout
    u = _state(p, lay, 3)
    ref = assembly.assemble("mc", p, u)
    x = asm.create_vec(u[lay.perm])
    g1, g2 = x.duplicate(), x.duplicate()
    e_sep = float(asm.energy_device(x.t).item())
    asm.gradient_device(x.t, g1.t)
    asm.hessian_device(x.t)
    h_sep = asm.A.data.clone()
    e_f = float(asm.energy_grad_hessian_device(x.t, g2.t).item())
    assert e_f == e_sep
    assert torch.equal(g1.t, g2.t) and torch.equal(h_sep, asm.A.data)
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    assert abs(H - ref["h"]).max() <= 3e-5 * abs(ref["h"]).max()
    assert np.abs(g1.array[lay.iperm] - ref["g"]).max() <= 1e-11 * np.abs(ref["g"]).max()
    asm.cleanup()


def test_elastic_mode_matches_elastic_stiffness(require_gpu):
    p, adj = mc_params(h=4.0, degree=4, lam=1.0)
    asm = SlopeStabilityReorderedElementAssembler(p, None, adj, hessian_precision="fp64")
    lay = asm.layout
    u = _state(p, lay, 4, scale=5e-3)
    asm.assemble_hessian_with_mode(asm.create_vec(u[lay.perm]), constitutive_mode="elastic")
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    ref = assembly.assemble("mc", p, u, want=("h",), elastic_only=True)
    assert abs(H - ref["h"]).max() <= 1e-10 * abs(ref["h"]).max()
    # the mode switch is scoped to the call: the energy afterwards is the full Mohr-Coulomb one
    Ee = asm.energy_fn(asm.create_vec(u[lay.perm]))
    Eref = assembly.assemble("mc", p, u, want=("e",))["e"]
    assert abs(Ee - Eref) <= 1e-12 * abs(Eref)
    asm.cleanup()


class _SingleRows(SlopeStabilityReorderedElementAssembler):
    row_units = False


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("degree,h,order", [
    (4, 10.0, "odd"),  # a y component constrained by itself: the last batch has one row
    (4, 3.0, "block_xyz"),
    (4, 3.0, "apart"),  # the x rows, then the y rows
    (2, 1.3, "block_morton"),
    (2, 1.6, "apart"),
])
def test_rows_without_units_match_the_oracle(require_gpu, degree, h, order, precision):
    """The row-by-row form: plans without row units, and orderings that leave no pairs to list.  Tolerances
    of the tests above."""
    p, adj = mc_params(h=h, degree=degree, lam=1.5)
    kw = {"reorder_mode": order}
    if order == "odd":
        keep = np.delete(np.arange(p["freedofs"].size), 101)
        p, adj, kw = dict(p, freedofs=np.asarray(p["freedofs"])[keep]), adj.tocsr()[keep][:, keep], {}
    free = np.asarray(p["freedofs"])
    assert (free.size % 2 == 1) == (order == "odd")
    if order == "apart":
        kw = {"perm_override": np.argsort(free % 2, kind="stable")}
    cls = SlopeStabilityReorderedElementAssembler if order == "apart" else _SingleRows
    asm = cls(p, None, adj, hessian_precision=precision, **kw)
    lay = asm.layout
    u = _state(p, lay, 6)
    ref = assembly.assemble("mc", p, u)
    x = asm.create_vec(u[lay.perm])
    g, y = x.duplicate(), x.duplicate()
    asm.A.data.fill_(float("nan"))  # every entry is written
    e = float(asm.energy_grad_hessian_device(x.t, g.t).item())
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    assert abs(e - ref["e"]) <= 1e-12 * abs(ref["e"])
    assert np.abs(g.array[lay.iperm] - ref["g"]).max() <= 1e-11 * np.abs(ref["g"]).max()
    assert abs(H - ref["h"]).max() <= (1e-10 if precision == "fp64" else 3e-5) * abs(ref["h"]).max()
    v = asm.A.data.clone()
    asm.A.data.fill_(float("nan"))
    asm.hessian_device(x.t)
    assert torch.equal(asm.A.data, v)
    asm.hvp_device(x.t, x.t, y.t)
    want = ref["h"] @ u
    assert np.abs(y.array[lay.iperm] - want).max() <= 1e-10 * np.abs(want).max()
    asm.cleanup()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", [4, 2])
@pytest.mark.parametrize("points", [20, 21])  # the last of the shorter K range, and the longer one
def test_quadrature_of_20_and_21_points(require_gpu, points, degree, precision):
    """The 19-point rule with its last points split in two halves of their weight integrates the same:
    the oracle's results, within the tolerances of the tests above."""
    p, adj = mc_params(h=4.0, degree=degree, lam=1.5)
    nq = p["wq"].size
    split = np.arange(nq - (points - nq), nq)
    take = np.append(np.arange(nq), split)
    w = p["wq"].copy()
    w[split] *= 0.5
    q = dict(p, xq=p["xq"][take], wq=w[take], phi=p["phi"][:, take], dhat=p["dhat"][take])
    assert q["wq"].size == points
    asm = SlopeStabilityReorderedElementAssembler(q, None, adj, hessian_precision=precision)
    lay = asm.layout
    u = _state(p, lay, 7)
    ref = assembly.assemble("mc", p, u)
    x = asm.create_vec(u[lay.perm])
    g, y = x.duplicate(), x.duplicate()
    e = float(asm.energy_grad_hessian_device(x.t, g.t).item())
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm]
    assert abs(e - ref["e"]) <= 1e-12 * abs(ref["e"])
    assert np.abs(g.array[lay.iperm] - ref["g"]).max() <= 1e-11 * np.abs(ref["g"]).max()
    assert abs(H - ref["h"]).max() <= (1e-10 if precision == "fp64" else 3e-5) * abs(ref["h"]).max()
    asm.hvp_device(x.t, x.t, y.t)
    want = ref["h"] @ u
    assert np.abs(y.array[lay.iperm] - want).max() <= 1e-10 * np.abs(want).max()
    asm.cleanup()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", [4, 2])
@pytest.mark.parametrize("cls", [SlopeStabilityReorderedElementAssembler, _SingleRows])
def test_free_node_without_elements(require_gpu, cls, degree, precision):
    """A free node that no element names has CSR rows without entries: nothing is read or stored for them,
    the other rows are those of the mesh without it, and its gradient is minus its load."""
    p, adj = mc_params(h=5.0, degree=degree, lam=1.2)
    n, nt = p["freedofs"].size, p["nodes"].shape[0]
    q = dict(p, nodes=np.vstack((p["nodes"], [[60.0, 60.0]])), freedofs=np.append(p["freedofs"], [2 * nt, 2 * nt + 1]),
             force=np.append(p["force"], [3.0, -2.0]), u_0=np.append(p["u_0"], [0.0, 0.0]))
    adj2 = sp.block_diag((adj, sp.coo_matrix((2, 2))))
    asm = cls(q, None, adj2, hessian_precision=precision)
    lay = asm.layout
    lens = np.diff(lay.indptr)[lay.iperm]
    assert np.all(lens[n:] == 0) and np.all(lens[:n] > 0)
    ref_asm = cls(p, None, adj)
    u = _state(p, ref_asm.layout, 3)
    ref = assembly.assemble("mc", p, u)
    x = asm.create_vec(np.append(u, [0.3, -0.1])[lay.perm])
    g = x.duplicate()
    asm.A.data.fill_(float("nan"))
    asm.energy_grad_hessian_device(x.t, g.t)
    H = asm.A.to_scipy()[lay.iperm][:, lay.iperm][:n, :n]
    assert abs(H - ref["h"]).max() <= (1e-10 if precision == "fp64" else 3e-5) * abs(ref["h"]).max()
    got = g.array[lay.iperm]
    assert np.abs(got[:n] - ref["g"]).max() <= 1e-11 * np.abs(ref["g"]).max()
    assert got[n:].tolist() == [-3.0, 2.0]
    asm.cleanup()
    ref_asm.cleanup()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("degree,h,order", [
    (4, 10.0, "block_morton"),  # fewer elements than a block's wavefronts take
    (4, 4.0, "block_morton"),
    (4, 2.2, "block_xyz"),  # rows of a node together
    (4, 3.0, "random"),  # components of a node apart: single-row units
    (2, 1.1, "block_morton"),
    (2, 1.6, "random"),
])
def test_row_units_match_single_rows(require_gpu, degree, h, order, precision):
    """Node rows assembled together against every row by itself on the same plan arrays, with a load and
    the tolerances of the tests above (an FP32 entry: both forms within 3e-5 of the largest)."""
    p, adj = mc_params(h=h, degree=degree, lam=1.5)
    n = p["freedofs"].size
    kw = {"perm_override": np.random.default_rng(4).permutation(n)} if order == "random" else {"reorder_mode": order}
    out = []
    for cls in (SlopeStabilityReorderedElementAssembler, _SingleRows):
        asm = cls(p, None, adj, hessian_precision=precision, **kw)
        x = asm.create_vec(_state(p, asm.layout, 5)[asm.layout.perm])
        g, g2 = x.duplicate(), x.duplicate()
        asm.A.data.fill_(float("nan"))  # every entry is written
        e = float(asm.energy_grad_hessian_device(x.t, g.t).item())
        v = asm.A.data.clone()
        asm.gradient_device(x.t, g2.t)
        assert float(asm.energy_device(x.t).item()) == e and torch.equal(g.t, g2.t)
        asm.A.data.fill_(float("nan"))
        asm.hessian_device(x.t)
        assert torch.equal(asm.A.data, v)
        out.append((e, g.t.cpu().numpy(), v.double().cpu().numpy()))
        asm.cleanup()
    (e, g, v), (e0, g0, v0) = out
    assert abs(e - e0) <= 1e-12 * abs(e0)
    assert np.abs(g - g0).max() <= 1e-11 * np.abs(g0).max()
    assert np.abs(v - v0).max() <= (1e-10 if precision == "fp64" else 3e-5) * np.abs(v0).max()
