"""Smoothed-aggregation AMG preconditioner (pc_type "gamg") on the GPU.

CG with the V-cycle reaches the solution of a direct solve (rel. 1e-6 at rtol 1e-10) in far
fewer iterations than point Jacobi, for an elasticity Hessian (rigid-body near-nullspace)
and a scalar p-Laplace Hessian (constant near-nullspace).
"""

import numpy as np
import pytest
import scipy.sparse.linalg as spla

from fenics_nonlinear_energies_amd.problems.hyperelasticity import (
    HEReorderedElementAssembler,
    build_beam_problem,
    rigid_modes,
)
from fenics_nonlinear_energies_amd.problems.plaplace import PLaplaceReorderedElementAssembler, build_plaplace_problem

pytestmark = pytest.mark.gpu


def _solve(asm, pc, rtol, b):
    ksp = asm.ksp
    ksp.pc_type = pc
    ksp._amg = None
    ksp._inv_diag = None
    ksp.setOperators(asm.A)
    ksp.setTolerances(rtol=rtol, max_it=20000)
    ksp.setUp()
    x = b.duplicate()
    ksp.solve(b, x)
    return x, ksp.getIterationNumber()


@pytest.mark.parametrize("coarse", ["host", "device"])
@pytest.mark.parametrize("kind", ["he", "plaplace"])
def test_gamg_cg_matches_direct_solve(require_gpu, kind, coarse):
    """Multigrid-preconditioned CG reaches the direct solution in far fewer iterations than
    Jacobi, with the coarsest level factorised on the host (LAPACK) or on the GPU."""
    opts = {"mg_coarse_factor": coarse}
    if kind == "he":
        p, adj, u0 = build_beam_problem(40, 4, 4)
        asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg", pc_options=opts)
        u = u0 + 1e-5 * np.random.default_rng(0).standard_normal(u0.size)
        x0 = asm.create_vec(u[asm.layout.perm])
    else:
        p, adj, _ = build_plaplace_problem(96)
        asm = PLaplaceReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg", pc_options=opts)
        x0 = asm.create_vec(np.random.default_rng(0).random(asm.layout.n_free))
    asm.assemble_hessian(x0)
    b = asm.create_vec(np.random.default_rng(1).standard_normal(asm.layout.n_free))
    xg, its_g = _solve(asm, "gamg", 1e-10, b)
    _, its_j = _solve(asm, "jacobi", 1e-10, b)
    ref = spla.spsolve(asm.A.to_scipy().tocsc(), b.array)
    assert np.linalg.norm(xg.array - ref) <= 1e-6 * np.linalg.norm(ref)
    assert its_g * 4 < its_j, (its_g, its_j)
    asm.cleanup()


def test_vcycle_graph_replays_match_eager(require_gpu):
    """The V-cycle recorded as a HIP graph gives bitwise the eager result on every replay
    (several replays, with unrelated eager work in between)."""
    import torch

    p, adj, _ = build_plaplace_problem(64)
    asm = PLaplaceReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg")
    asm.assemble_hessian(asm.create_vec(np.random.default_rng(0).random(asm.layout.n_free)))
    ksp = asm.ksp
    ksp.setOperators(asm.A)
    ksp.setUp()
    pc = ksp._amg
    assert pc._graph is not None
    rng = np.random.default_rng(5)
    for k in range(4):
        r = torch.as_tensor(rng.standard_normal(asm.layout.n_free)).cuda()
        eager = pc._cycle(0, r.clone())
        junk = torch.randn(10000, device="cuda").cumsum(0)  # unrelated eager work
        z = torch.empty_like(r)
        pc.apply(r, z)
        torch.cuda.synchronize()
        assert torch.equal(z, eager), k
        assert torch.isfinite(junk).all()
    asm.cleanup()


@pytest.mark.parametrize("a_prec", ["fp64", "fp32"])
def test_spgemm_numeric_matches_scipy(require_gpu, a_prec):
    """fne_spgemm_numeric against scipy's product, with result rows longer than one LDS chunk
    (512 entries) and A rows longer than one staging chunk (256), with signed values (cancelled entries of the fixed pattern come out 0)."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg

    A = sp.random(70, 3000, density=0.1, random_state=3, format="csr")
    B = sp.random(3000, 4000, density=0.003, random_state=4, format="csr")
    A.data -= 0.5
    B.data -= 0.5
    if a_prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
    C_pat = amg._pattern_product(A, B)
    assert np.diff(C_pat.indptr).max() > 1024  # more than two LDS chunks of result columns
    assert np.diff(A.indptr).max() > 256  # more than one staging chunk of A's row
    dev = torch.device("cuda")
    Bd = amg._DevMat(B.indptr, B.indices, B.shape[1], dev, "fp64")
    Bd.data.copy_(torch.as_tensor(B.data))
    Cd = amg._DevMat(C_pat.indptr, C_pat.indices, C_pat.shape[1], dev, "fp64")
    a_ptr = torch.as_tensor(A.indptr.astype(np.int32)).to(dev)
    a_idx = torch.as_tensor(A.indices.astype(np.int32)).to(dev)
    a_dat = torch.as_tensor(A.data).to(dev, torch.float32 if a_prec == "fp32" else torch.float64)
    Cd.data.fill_(np.nan)
    amg._spgemm(a_ptr, a_idx, a_dat, Bd, Bd.data, Cd, Cd.data)
    got = sp.csr_matrix((Cd.data.cpu().numpy(), C_pat.indices, C_pat.indptr), shape=C_pat.shape).toarray()
    ref = (A @ B).toarray()
    assert np.all(np.isfinite(got))
    np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-14 * np.abs(ref).max())
    # deterministic: a second product is bitwise the same
    first = Cd.data.clone()
    amg._spgemm(a_ptr, a_idx, a_dat, Bd, Bd.data, Cd, Cd.data)
    assert torch.equal(first, Cd.data)


@pytest.mark.parametrize("a_prec", ["fp64", "fp32"])
@pytest.mark.parametrize("lanes", [0, 8, 16, 32, 64])
def test_spgemm_lane_groups_match_scipy(require_gpu, lanes, a_prec):
    """Every lane-group width on rows at its edges: empty rows of A, B and C, rows of A and B one
    shorter, as long and one longer than the group, result rows longer than its 8 x lanes staged
    columns; sums in the order of A's row, so all widths agree bitwise."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg, native

    rng = np.random.default_rng(11)

    def rows_of(lengths, n_cols):
        cols = [np.sort(rng.choice(n_cols, size=m, replace=False)) for m in lengths]
        ptr = np.concatenate(([0], np.cumsum(lengths)))
        return sp.csr_matrix((rng.standard_normal(ptr[-1]), np.concatenate(cols), ptr), shape=(len(lengths), n_cols))

    edges = [m for g in (8, 16, 32, 64) for m in (g - 1, g, g + 1)]
    A = rows_of([0, 1, 3, 4, 5, *edges, 0, 1], 97)
    B = rows_of(([0, 1, 2, *edges] * 7)[:97], 1500)
    if a_prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
    C_pat = amg._pattern_product(A, B)
    assert np.diff(C_pat.indptr).max() > 8 * 64
    dev = torch.device("cuda")
    i32 = lambda a: torch.as_tensor(a.astype(np.int32)).to(dev)  # noqa: E731
    a = [i32(A.indptr), i32(A.indices), torch.as_tensor(A.data).to(dev, torch.float32 if a_prec == "fp32" else torch.float64)]
    b = [i32(B.indptr), i32(B.indices), torch.as_tensor(B.data).to(dev)]
    c = [i32(C_pat.indptr), i32(C_pat.indices)]
    prec = native.FNE_FP32 if a_prec == "fp32" else native.FNE_FP64
    out = []
    for g in (lanes, 64):
        val = torch.full((C_pat.nnz,), float("nan"), dtype=torch.float64, device=dev)
        native.check(native.lib().fne_spgemm_numeric(
            A.shape[0], *(native.ptr(t) for t in a), prec | g << 8, *(native.ptr(t) for t in b),
            *(native.ptr(t) for t in c), native.ptr(val), native.stream_ptr()), "fne_spgemm_numeric")
        out.append(val.cpu().numpy())
    assert np.array_equal(out[0], out[1])
    # a sum of at most 65 products in another order
    bound = 2 * 65 * 2.0**-53 * (abs(A) @ abs(B)).toarray()
    got = sp.csr_matrix((out[0], C_pat.indices, C_pat.indptr), shape=C_pat.shape).toarray()
    assert np.all(np.abs(got - (A @ B).toarray()) <= bound)


@pytest.mark.parametrize("a_prec", ["fp64", "fp32"])
def test_spgemm_split_rows_match_scipy(require_gpu, a_prec):
    """Four lane groups per row: rows of A shorter than four, with and without a remainder, result rows
    longer than the staged columns; a sum of at most 300 products in another order."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg, native

    rng = np.random.default_rng(5)
    lengths = [0, 1, 2, 3, 4, 5, 63, 64, 65, 255, 256, 257, 300]
    ptr = np.concatenate(([0], np.cumsum(lengths)))
    cols = np.concatenate([np.sort(rng.choice(301, size=m, replace=False)) for m in lengths]).astype(int)
    A = sp.csr_matrix((rng.standard_normal(ptr[-1]), cols, ptr), shape=(len(lengths), 301))
    B = sp.random(301, 900, density=0.08, random_state=9, format="csr")
    if a_prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
    C_pat = amg._pattern_product(A, B)
    assert np.diff(C_pat.indptr).max() > 512 and np.diff(B.indptr).max() > 64
    dev = torch.device("cuda")
    i32 = lambda a: torch.as_tensor(a.astype(np.int32)).to(dev)  # noqa: E731
    prec = native.FNE_FP32 if a_prec == "fp32" else native.FNE_FP64
    args = [i32(A.indptr), i32(A.indices), torch.as_tensor(A.data).to(dev, torch.float32 if prec == native.FNE_FP32
                                                                      else torch.float64)]
    rest = [i32(B.indptr), i32(B.indices), torch.as_tensor(B.data).to(dev), i32(C_pat.indptr), i32(C_pat.indices)]
    val = torch.full((C_pat.nnz,), float("nan"), dtype=torch.float64, device=dev)

    def run(code):
        return native.lib().fne_spgemm_numeric(A.shape[0], *(native.ptr(t) for t in args), code,
                                               *(native.ptr(t) for t in rest), native.ptr(val), native.stream_ptr())

    assert run(prec | 32 << 8 | 1 << 16) != 0 and run(prec | 64 << 8 | 2 << 16) != 0
    native.check(run(prec | 64 << 8 | 1 << 16), "fne_spgemm_numeric")
    got = sp.csr_matrix((val.cpu().numpy(), C_pat.indices, C_pat.indptr), shape=C_pat.shape).toarray()
    bound = 2 * 304 * 2.0**-53 * (abs(A) @ abs(B)).toarray()
    assert np.all(np.abs(got - (A @ B).toarray()) <= bound)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,width", [(1, 1), (255, 7), (257, 60), (4097, 20)])
def test_first_two_chebyshev_steps_equal_the_steps_one_by_one(require_gpu, n, width, prec):
    """fne_vcycle_cheb_first against w_0 r and fne_vcycle_cheb with a zero vector before it, in the forms of the row
    kernels: the same sums, and one more or one less fused multiply-add per entry."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg, linalg, native

    rng = np.random.default_rng(n)
    A = (sp.random(n, n, density=min(1.0, width / n), random_state=2) + sp.identity(n)).tocsr()
    A.sort_indices()
    dev = torch.device("cuda")
    M = amg._DevMat(A.indptr, A.indices, n, dev, prec)
    M.data.copy_(torch.as_tensor(A.data))
    r, w0, w1 = (torch.as_tensor(rng.uniform(0.5, 1.5, n)).to(dev) for _ in range(3))
    for code in (linalg.spmv_code(M.prec, A.nnz / n), M.prec, M.prec | 64 << 8, M.prec | 1 << 8):
        M.code = code
        y, ref = torch.full_like(r, float("nan")), torch.empty_like(r)
        M.cheb_first(r, w0, w1, 0.3, y)
        M.cheb(w0 * r, torch.zeros_like(r), r, w1, 0.3, ref)
        # |A| x_1 is at most 2.25 (nnz of the row); a few roundings of each product
        assert (y - ref).abs().max().item() <= 8 * 2.0**-53 * 1.5 * 2.25 * (2 + np.diff(A.indptr).max())
    assert native.lib().fne_vcycle_cheb_first(n, native.ptr(M.indptr), native.ptr(M.indices), native.ptr(M.data),
                                              M.code, native.ptr(r), native.ptr(w0), native.ptr(w1), 0.3,
                                              native.ptr(r), native.stream_ptr()) != 0


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,width", [(1, 1), (2, 2), (13, 3), (255, 7), (257, 30), (4097, 60), (150_000, 7)])
def test_lanczos_and_smoothed_product_match_host(require_gpu, n, width, prec):
    """fne_lanczos_max in both forms of its product against the host recurrence (the same Krylov
    space in other roundings: 1e-9 of the eigenvalue), its inverse diagonal with a zero entry, and
    fne_spgemm_smoothed; sizes around a block, above the partial sums one block adds up, and below
    the number of steps."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg, linalg, native

    rng = np.random.default_rng(n)
    off = [sp.diags(rng.uniform(-1.0, 0.0, n - k), k) for k in sorted({int(j) for j in np.linspace(1, n - 1, width)})
           if 0 < k < n] if n > 1 else []
    U = sum(off, sp.csr_matrix((n, n)))
    A = (U + U.T + sp.diags(np.asarray(abs(U + U.T).sum(axis=1)).ravel() + rng.uniform(0.5, 1.0, n))).tocsr()
    A.sort_indices()
    if prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
    diag = amg._positions(A, np.arange(n), np.arange(n))
    dev = torch.device("cuda")
    ptr, idx = (torch.as_tensor(a.astype(np.int32)).to(dev) for a in (A.indptr, A.indices))
    val = torch.as_tensor(A.data).to(dev, torch.float32 if prec == "fp32" else torch.float64)
    dg, v0 = torch.as_tensor(diag).to(dev), torch.as_tensor(rng.standard_normal(n)).to(dev)
    dinv, out = torch.empty(n, dtype=torch.float64, device=dev), torch.empty(2, dtype=torch.float64, device=dev)
    base = native.FNE_FP32 if prec == "fp32" else native.FNE_FP64

    class _Host:
        @staticmethod
        def mult_tensor(x, y):
            y.copy_(torch.as_tensor(A @ x.numpy()))

    ref = amg.SmoothedAggregationPC()._lanczos_lambda_max(0, _Host, torch.as_tensor(1.0 / A.diagonal()), v0.cpu())

    def run(code, values):
        m = int(native.lib().fne_lanczos_work_len(n, code))
        assert m == amg._lanczos_work_len(n, code)
        work = torch.full((m,), float("nan"), dtype=torch.float64, device=dev)
        native.check(native.lib().fne_lanczos_max(n, native.ptr(ptr), native.ptr(idx), native.ptr(values), code,
                                                  native.ptr(dg), native.ptr(v0), 12, native.ptr(dinv),
                                                  native.ptr(work), m, native.ptr(out), native.stream_ptr()), "lanczos")
        return out.cpu().numpy()

    for code in (linalg.spmv_code(base, A.nnz / n), base, base | 64 << 8):
        lam, ok = run(code, val)
        assert ok == 1.0 and abs(lam - ref) <= 1e-9 * ref
        np.testing.assert_array_equal(dinv.cpu().numpy(), 1.0 / A.diagonal())
    holes = val.clone()
    holes[diag[0]] = 0.0
    assert np.isfinite(run(base, holes)).all() and dinv[0].item() == 1.0
    holes[diag[n // 2]] = float("nan")
    assert run(base, holes)[1] == 0.0

    # P = P_tent - diag(w) A P_tent with aggregates of three
    Pt, _ = amg.tentative_prolongator(rng.standard_normal((n, 1)), 3)
    w = rng.uniform(0.1, 1.0, n)
    C_pat = amg._pattern(amg._pattern_product(A, Pt) + amg._pattern(Pt))
    B = amg._DevMat(Pt.indptr, Pt.indices, Pt.shape[1], dev, "fp64")
    B.data.copy_(torch.as_tensor(Pt.data))
    C = amg._DevMat(C_pat.indptr, C_pat.indices, C_pat.shape[1], dev, "fp64")
    C.data.fill_(float("nan"))
    amg._spgemm_smoothed(ptr, idx, val, B, C, torch.as_tensor(w).to(dev))
    got = sp.csr_matrix((C.data.cpu().numpy(), C_pat.indices, C_pat.indptr), shape=C_pat.shape)
    want = (Pt - sp.diags(w) @ (A @ Pt)).tocsr()
    scale = abs(Pt) + sp.diags(w) @ (abs(A) @ abs(Pt))
    # at most 61 products, the scaling and the addition
    assert abs(got - want).max() <= 2 * 64 * 2.0**-53 * scale.max()


@pytest.mark.parametrize("steps", [12, 64, 65, 90])
def test_setup_takes_any_number_of_lanczos_steps(require_gpu, steps):
    """LANCZOS_STEPS beyond the 64 that fne_lanczos_max takes: the Jacobi weights of the finest level hold a
    Ritz value, between 0.9 (12 steps; 0.99 from 64 on) and all of the largest eigenvalue of D^-1 A."""
    import torch

    from fenics_nonlinear_energies_amd import amg
    from fenics_nonlinear_energies_amd.linalg import DeviceCSR

    p, adj, _ = build_plaplace_problem(16)
    asm = PLaplaceReorderedElementAssembler(p, None, adj)
    asm.assemble_hessian(asm.create_vec(np.random.default_rng(2).random(asm.layout.n_free)))
    pc = amg.SmoothedAggregationPC(max_coarse=20)
    pc.LANCZOS_STEPS = steps
    pc.setup(asm.A)
    H = asm.A.to_scipy().toarray()
    s = 1.0 / np.sqrt(H.diagonal())
    top = np.linalg.eigvalsh(s[:, None] * H * s).max()
    L = pc.levels[0]
    lam = 4.0 / (3.0 * pc.RHO_SAFETY) * (L["dinv"] / L["wd"]).cpu().numpy()
    assert np.ptp(lam) <= 1e-13 * lam.max()
    assert (0.9 if steps < 64 else 0.99) * top <= lam[0] <= (1 + 1e-12) * top
    r = torch.ones(asm.layout.n_free, dtype=torch.float64, device="cuda")
    z = torch.empty_like(r)
    pc.apply(r, z)
    assert torch.isfinite(z).all()
    asm.cleanup()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 97, 287])
def test_spd_inverse_matches_numpy(require_gpu, n):
    """fne_spd_inverse at the edges of its 32-column blocks: a matrix of condition 1e4 (n eps cond is
    6e-10 at most of the inverse's largest entry), the symmetric part of an unsymmetric one, and the
    status of an indefinite one and of a NaN."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import native

    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    S = (Q * np.geomspace(1.0, 1e-4, n)) @ Q.T
    S = 0.5 * (S + S.T)
    K = rng.standard_normal((n, n)) * 1e-3
    dev = torch.device("cuda")
    m = int(native.lib().fne_spd_inverse_work_len(n))
    work, inv = (torch.full((k,), float("nan"), dtype=torch.float64, device=dev) for k in (m, n * n))
    status = torch.full((1,), 7.0, dtype=torch.float64, device=dev)

    def run(M):
        C = sp.csr_matrix(M)
        ptr, idx = (torch.as_tensor(a.astype(np.int32)).to(dev) for a in (C.indptr, C.indices))
        val = torch.as_tensor(C.data).to(dev)
        native.check(native.lib().fne_spd_inverse(n, native.ptr(ptr), native.ptr(idx), native.ptr(val),
                                                  native.ptr(work), m, native.ptr(inv), native.ptr(status),
                                                  native.stream_ptr()), "fne_spd_inverse")
        return inv.cpu().numpy().reshape(n, n), status.item()

    X, st = run(S + (K - K.T))
    ref = np.linalg.inv(S)
    assert st == 0.0 and np.array_equal(X, X.T)
    assert np.abs(X - ref).max() <= 1e-9 * np.abs(ref).max()
    flip = np.geomspace(1.0, 1e-4, n)
    flip[-1] = -0.5
    assert run((Q * flip) @ Q.T)[1] == 1.0
    bad = S.copy()
    bad[n // 2, n // 2] = np.nan
    assert run(bad)[1] == 1.0


@pytest.mark.parametrize("n,cond", [(32, 1e8), (33, 1e8), (33, 1e11), (65, 1e10), (97, 1e12), (287, 1e11), (1200, 1e8)])
def test_spd_inverse_is_as_accurate_as_lapack(require_gpu, n, cond):
    """fne_spd_inverse of ill-conditioned operators, up to the default coarse size, against coarse_inverse
    (potrf, potri).  The factor's inverse is within n eps cond of the inverse's largest entry in either."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import native
    from fenics_nonlinear_energies_amd.amg import coarse_inverse

    rng = np.random.default_rng(n)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    S = (Q * np.geomspace(1.0, 1.0 / cond, n)) @ Q.T
    S = 0.5 * (S + S.T)
    dev = torch.device("cuda")
    C = sp.csr_matrix(S)
    ptr, idx = (torch.as_tensor(a.astype(np.int32)).to(dev) for a in (C.indptr, C.indices))
    val = torch.as_tensor(C.data).to(dev)
    m = int(native.lib().fne_spd_inverse_work_len(n))
    work, inv, status = (torch.full((k,), float("nan"), dtype=torch.float64, device=dev) for k in (m, n * n, 1))
    native.check(native.lib().fne_spd_inverse(n, native.ptr(ptr), native.ptr(idx), native.ptr(val), native.ptr(work), m,
                                              native.ptr(inv), native.ptr(status), native.stream_ptr()),
                 "fne_spd_inverse")
    ref, fallback = coarse_inverse(S)
    assert not fallback and status.item() == 0.0
    X = inv.cpu().numpy().reshape(n, n)
    err = np.abs(X - ref).max() / np.abs(ref).max()
    print("spd inverse", n, cond, err, flush=True)
    assert err <= 2.0 * n * np.finfo(float).eps * cond


@pytest.mark.parametrize("coarse", ["host", "device"])
def test_setup_after_a_failed_one(require_gpu, coarse):
    """A set-up on an operator with a NaN raises; the next one, on the same object with finite values, leaves
    the hierarchy and the cycle of a new object bit for bit."""
    import torch

    from fenics_nonlinear_energies_amd import amg

    p, adj, _ = build_plaplace_problem(24)
    asm = PLaplaceReorderedElementAssembler(p, None, adj)
    asm.assemble_hessian(asm.create_vec(np.random.default_rng(2).random(asm.layout.n_free)))
    r = torch.as_tensor(np.random.default_rng(3).standard_normal(asm.layout.n_free)).cuda()

    def result(pc):
        pc.setup(asm.A)
        z = torch.empty_like(r)
        pc.apply(r, z)
        return [z] + [t for L in pc.levels for t in (L["P64"].data, L["Ac64"].data, L["wd"], L["wcheb"])]

    pc = amg.SmoothedAggregationPC(max_coarse=30, coarse_factor=coarse)
    good = asm.A.data.clone()
    asm.A.data[asm.A.nnz // 2] = float("nan")
    with pytest.raises(FloatingPointError):
        pc.setup(asm.A)
    asm.A.data.copy_(good)
    got, ref = result(pc), result(amg.SmoothedAggregationPC(max_coarse=30, coarse_factor=coarse))
    assert all(torch.equal(a, b) and torch.isfinite(a).all() for a, b in zip(got, ref))
    asm.cleanup()


def _host_levels(pc, A0):
    """Operators of every level read back from the device (FP64 masters)."""
    import scipy.sparse as sp

    out = []
    A = A0
    for L in pc.levels:
        P = L["P64"]
        Pm = sp.csr_matrix((P.data.cpu().numpy(), P.indices.cpu().numpy(), P.indptr.cpu().numpy()),
                           shape=(L["n"], L["nc"]))
        Ac = L["Ac64"]
        Acm = sp.csr_matrix((Ac.data.cpu().numpy(), Ac.indices.cpu().numpy(), Ac.indptr.cpu().numpy()),
                            shape=(L["nc"], L["nc"]))
        out.append((A, Pm, Acm, L["wd"].cpu().numpy()))
        A = Acm
    return out


@pytest.mark.parametrize("smoother", ["jacobi", "chebyshev"])
def test_device_galerkin_setup_matches_host_products(require_gpu, smoother):
    """Every level of the device set-up: P = P_tent - omega D^-1 A P_tent with P_tent from the
    host QR of the (current-configuration) rigid modes, A_c = P^T A P, omega within 15 % of the
    host power-iteration value of 4 / (3 rho(D^-1 A)) (60 steps); and the V-cycle equals a host cycle
    on the same operators, with either smoother (Chebyshev in the textbook form of Saad,
    Iterative Methods, Alg. 12.1, on [0.1, 1.1] lambda_max with Jacobi scaling)."""
    import torch

    from fenics_nonlinear_energies_amd import amg

    p, adj, u0 = build_beam_problem(40, 4, 4)
    asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg")
    u = u0 + 1e-4 * np.random.default_rng(0).standard_normal(u0.size)
    x = asm.create_vec(u[asm.layout.perm])
    asm.assemble_hessian(x)
    B = asm._rigid_modes_current().cpu().numpy()
    np.testing.assert_array_equal(B, rigid_modes(x.t.cpu().numpy().reshape(-1, 3)))
    pc = amg.SmoothedAggregationPC(B, precision="fp64", max_coarse=100, smoother=smoother)
    pc.setup(asm.A)
    assert len(pc.levels) >= 2
    Bl = B
    for lvl, (A, P, Ac, wd) in enumerate(_host_levels(pc, asm.A.to_scipy())):
        Pt, Bc = amg.tentative_prolongator(Bl, pc.levels[lvl]["agg"])
        d = A.diagonal()
        omega = wd[0] * d[0]
        np.testing.assert_allclose(wd, omega / d, rtol=1e-12)
        amg_rho = None  # host estimate of rho(D^-1 A)
        v = np.random.default_rng(1).standard_normal(A.shape[0])
        for _ in range(60):
            y = (A @ v) / d
            amg_rho = np.linalg.norm(y) / np.linalg.norm(v)
            v = y / np.linalg.norm(y)
        rho = amg_rho
        # omega from a 12-step device Lanczos estimate x 1.1: near 4 / (3 rho), convergent smoother
        assert 0.85 <= omega * 3.0 * rho / 4.0 <= 1.15 and omega * rho < 2.0, (omega, rho)
        Pdev = pc.levels[lvl]["Pt"].data.cpu().numpy()  # device QR (fne_aggregate_qr)
        np.testing.assert_allclose(Pdev, Pt.data, rtol=0, atol=1e-12)
        np.testing.assert_allclose(pc.levels[lvl]["Bc"].cpu().numpy(), Bc, rtol=0, atol=1e-12 * np.abs(Bc).max())
        Pref = (Pt - omega * (A @ Pt).multiply(1.0 / d[:, None])).toarray()
        np.testing.assert_allclose(P.toarray(), Pref, rtol=0, atol=1e-12 * np.abs(Pref).max())
        Acref = (P.T @ A @ P).toarray()
        Acref = 0.5 * (Acref + Acref.T)
        np.testing.assert_allclose(Ac.toarray(), Acref, rtol=0, atol=1e-12 * np.abs(Acref).max())
        Bl = Bc
    # V-cycle against the host restatement on the read-back operators
    levels = _host_levels(pc, asm.A.to_scipy())
    Ainv = pc.coarse_op.data.cpu().numpy().reshape(pc._coarse_n, pc._coarse_n)

    def cheb(lvl, A, r, x):
        # Saad Alg. 12.1 with M = D: d_0 = M^-1 r_0 / theta, d_k = rho_k rho_{k-1} d_{k-1}
        # + (2 rho_k / delta) M^-1 r_k, x_{k+1} = x_k + d_k
        dinv = 1.0 / A.diagonal()
        lam = 1.0 / (0.6 * float(pc.levels[lvl]["wcheb"][0, 0].cpu()) / dinv[0])
        a, b = 0.1 * lam, 1.1 * lam
        theta, delta = 0.5 * (b + a), 0.5 * (b - a)
        sigma = theta / delta
        rho = 1.0 / sigma
        dk = dinv * (r - A @ x) / theta
        x = x + dk
        for _ in range(pc.sweeps - 1):
            rho_new = 1.0 / (2.0 * sigma - rho)
            dk = rho_new * rho * dk + (2.0 * rho_new / delta) * dinv * (r - A @ x)
            x = x + dk
            rho = rho_new
        return x

    def cycle(lvl, r):
        if lvl == len(levels):
            return Ainv @ r
        A, P, _, wd = levels[lvl]
        if smoother == "chebyshev":
            xx = cheb(lvl, A, r, np.zeros_like(r))
        else:
            xx = wd * r
            for _ in range(pc.sweeps - 1):
                xx = xx + wd * (r - A @ xx)
        xx = xx + P @ cycle(lvl + 1, P.T @ (r - A @ xx))
        if smoother == "chebyshev":
            return cheb(lvl, A, r, xx)
        for _ in range(pc.sweeps):
            xx = xx + wd * (r - A @ xx)
        return xx

    r = np.random.default_rng(2).standard_normal(asm.layout.n_free)
    z = torch.empty(r.size, dtype=torch.float64, device="cuda")
    pc.apply(torch.as_tensor(r).cuda(), z)
    ref = cycle(0, r)
    np.testing.assert_allclose(z.cpu().numpy(), ref, rtol=0, atol=1e-10 * np.abs(ref).max())
    asm.cleanup()


def test_resetup_reuses_graph_and_follows_the_hessian(require_gpu):
    """A second set-up at another state rewrites the recorded cycle's buffers in place: the
    graph object is kept and its replays equal the eager cycle on the new operators."""
    import torch

    p, adj, u0 = build_beam_problem(40, 4, 4)
    asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg")
    ksp = asm.ksp
    rng = np.random.default_rng(3)
    graph = None
    for k, scale in enumerate((1e-5, 3e-3)):
        x = asm.create_vec((u0 + scale * rng.standard_normal(u0.size))[asm.layout.perm])
        asm.assemble_hessian(x)
        ksp.setOperators(asm.A)
        ksp.setUp()
        pc = ksp._amg
        if graph is None:
            graph = pc._graph
        assert pc._graph is graph and pc.setup_count == k + 1
        r = torch.as_tensor(rng.standard_normal(asm.layout.n_free)).cuda()
        eager = pc._cycle(0, r.clone())
        z = torch.empty_like(r)
        pc.apply(r, z)
        torch.cuda.synchronize()
        assert torch.equal(z, eager), k
    asm.cleanup()


def test_device_cg_with_graph_preconditioner_matches_host_cg(require_gpu):
    """fne_pcg_graph (device iteration launching the recorded V-cycle) against the host-driven
    KSPCG restatement with the same preconditioner: same iteration count and reason, and the
    same solution to 1e-10."""
    import torch

    p, adj, u0 = build_beam_problem(40, 4, 4)
    asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg")
    x = asm.create_vec((u0 + 1e-5 * np.random.default_rng(4).standard_normal(u0.size))[asm.layout.perm])
    asm.assemble_hessian(x)
    ksp = asm.ksp
    ksp.setOperators(asm.A)
    ksp.setUp()
    assert ksp._amg._graph is not None
    b = asm.create_vec(np.random.default_rng(5).standard_normal(asm.layout.n_free))
    for rtol in (1e-1, 1e-8):
        ksp.setTolerances(rtol=rtol, max_it=500)
        xd = b.duplicate()
        ksp.solve(b, xd)
        its_d, reason_d = ksp.getIterationNumber(), ksp.getConvergedReason()
        xh = torch.empty_like(b.t)
        ksp._solve_cg_host(b.t, xh)
        assert (its_d, reason_d) == (ksp.getIterationNumber(), ksp.getConvergedReason()), (its_d, reason_d)
        assert reason_d > 0
        torch.testing.assert_close(xd.t, xh, rtol=1e-10, atol=1e-10 * float(xh.abs().max()))
    asm.cleanup()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_fused_vcycle_ops_match_numpy(require_gpu, prec):
    """fne_vcycle_op: first sweep, sweep, residual and in-place prolongation-add against numpy
    on a random CSR operator (FP32 values are compared with their FP32-rounded numpy twin)."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg

    rng = np.random.default_rng(7)
    A = sp.random(500, 500, density=0.03, random_state=8, format="csr") + sp.eye(500, format="csr")
    A.sort_indices()
    P = sp.random(500, 80, density=0.05, random_state=9, format="csr")
    P.sort_indices()
    if prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
        P.data = P.data.astype(np.float32).astype(np.float64)
    dev = torch.device("cuda")
    Ad = amg._DevMat(A.indptr, A.indices, 500, dev, prec)
    Ad.data.copy_(torch.as_tensor(A.data))
    Pd = amg._DevMat(P.indptr, P.indices, 80, dev, prec)
    Pd.data.copy_(torch.as_tensor(P.data))
    x, r, w = (rng.standard_normal(500) for _ in range(3))
    xc = rng.standard_normal(80)
    T = lambda v: torch.as_tensor(v).to(dev)  # noqa: E731
    y = torch.empty(500, dtype=torch.float64, device=dev)
    tol = dict(rtol=1e-12, atol=1e-12)
    Ad.op(amg._SWEEP_FIRST, None, T(r), T(w), None, y)
    x1 = w * r
    np.testing.assert_allclose(y.cpu().numpy(), x1 + w * (r - A @ x1), **tol)
    Ad.op(amg._SWEEP, T(x), T(r), T(w), None, y)
    np.testing.assert_allclose(y.cpu().numpy(), x + w * (r - A @ x), **tol)
    Ad.op(amg._RESIDUAL, T(x), T(r), None, None, y)
    np.testing.assert_allclose(y.cpu().numpy(), r - A @ x, **tol)
    yy = T(x)
    Pd.op(amg._ADD_PRODUCT, T(xc), None, None, yy, yy)
    np.testing.assert_allclose(yy.cpu().numpy(), x + P @ xc, **tol)
    from fenics_nonlinear_energies_amd.native import FneError

    with pytest.raises(FneError):
        Ad.op(amg._SWEEP, yy, T(r), T(w), None, yy)  # in-place sweep is rejected


def test_fp32_multigrid_with_fp64_operator(require_gpu):
    """pc_precision="fp32" with an FP64 Hessian: the hierarchy (finest copy included) is stored
    in FP32 while CG runs on the FP64 operator, and still reaches the direct solution."""
    import torch

    p, adj, u0 = build_beam_problem(40, 4, 4)
    asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg", pc_precision="fp32")
    u = u0 + 1e-5 * np.random.default_rng(0).standard_normal(u0.size)
    asm.assemble_hessian(asm.create_vec(u[asm.layout.perm]))
    assert asm.A.precision == "fp64"
    b = asm.create_vec(np.random.default_rng(1).standard_normal(asm.layout.n_free))
    xg, its = _solve(asm, "gamg", 1e-10, b)
    pc = asm.ksp._amg
    assert pc.precision == "fp32" and pc.levels[0]["A"].data.dtype == torch.float32
    assert asm.ksp.getConvergedReason() > 0 and its < 200
    ref = spla.spsolve(asm.A.to_scipy().tocsc(), b.array)
    assert np.linalg.norm(xg.array - ref) <= 1e-6 * np.linalg.norm(ref)
    asm.cleanup()


@pytest.mark.parametrize("prec,density", [("fp64", 0.03), ("fp32", 0.03), ("fp64", 0.12)])
def test_chebyshev_step_matches_numpy(require_gpu, prec, density):
    """fne_vcycle_cheb: y = x + c (x - x_prev) + w.(r - A x) against numpy (the 0.12 density gives
    60-entry rows, the grouped-load path), in place over x_prev, and with x_prev absent for
    c = 0; an output aliasing x is rejected."""
    import scipy.sparse as sp
    import torch

    from fenics_nonlinear_energies_amd import amg
    from fenics_nonlinear_energies_amd.native import FneError

    rng = np.random.default_rng(11)
    A = sp.random(500, 500, density=density, random_state=12, format="csr") + sp.eye(500, format="csr")
    A.sort_indices()
    if prec == "fp32":
        A.data = A.data.astype(np.float32).astype(np.float64)
    dev = torch.device("cuda")
    Ad = amg._DevMat(A.indptr, A.indices, 500, dev, prec)
    Ad.data.copy_(torch.as_tensor(A.data))
    x, xp, r, w = (rng.standard_normal(500) for _ in range(4))
    T = lambda v: torch.as_tensor(v).to(dev)  # noqa: E731
    tol = dict(rtol=1e-12, atol=1e-12)
    y = torch.empty(500, dtype=torch.float64, device=dev)
    Ad.cheb(T(x), T(xp), T(r), T(w), 0.7, y)
    np.testing.assert_allclose(y.cpu().numpy(), x + 0.7 * (x - xp) + w * (r - A @ x), **tol)
    Ad.cheb(T(x), None, T(r), T(w), 0.0, y)
    np.testing.assert_allclose(y.cpu().numpy(), x + w * (r - A @ x), **tol)
    yp = T(xp)
    Ad.cheb(T(x), yp, T(r), T(w), 0.3, yp)  # in place over x_prev
    np.testing.assert_allclose(yp.cpu().numpy(), x + 0.3 * (x - xp) + w * (r - A @ x), **tol)
    xx = T(x)
    with pytest.raises(FneError):
        Ad.cheb(xx, T(xp), T(r), T(w), 0.5, xx)


@pytest.mark.parametrize("kind", ["he", "slope"])
def test_chebyshev_smoothed_multigrid_cg(require_gpu, kind):
    """CG with the Chebyshev-smoothed multigrid (mg_levels_ksp_type chebyshev, 2 steps) reaches
    the direct solution; its graph replays equal the eager cycle; iteration counts of both
    smoothers are printed."""
    import torch

    from fenics_nonlinear_energies_amd.problems.slope_stability import SlopeStabilityReorderedElementAssembler
    from tests.test_gpu_mc import _state
    from tests.test_oracle_mc import mc_params

    its = {}
    for smoother in ("richardson", "chebyshev"):
        opts = {"mg_levels_ksp_type": smoother, "mg_levels_ksp_max_it": 2}
        if kind == "he":
            p, adj, u0 = build_beam_problem(40, 4, 4)
            asm = HEReorderedElementAssembler(p, None, adj, ksp_type="cg", pc_type="gamg", pc_options=opts)
            x0 = asm.create_vec((u0 + 1e-5 * np.random.default_rng(0).standard_normal(u0.size))[asm.layout.perm])
        else:
            p, adj = mc_params(h=1.0, degree=4, lam=1.0)
            asm = SlopeStabilityReorderedElementAssembler(p, None, adj, hessian_precision="fp64", ksp_type="cg",
                                                          pc_type="mg", pc_options=opts)
            x0 = asm.create_vec(_state(p, asm.layout, 11)[asm.layout.perm])
        asm.assemble_hessian(x0)
        b = asm.create_vec(np.random.default_rng(1).standard_normal(asm.layout.n_free))
        ksp = asm.ksp
        ksp.setOperators(asm.A)
        ksp.setTolerances(rtol=1e-10, max_it=5000)
        ksp.setUp()
        assert ksp._amg.smoother == ("chebyshev" if smoother == "chebyshev" else "jacobi")
        x = b.duplicate()
        ksp.solve(b, x)
        assert ksp.getConvergedReason() > 0
        its[smoother] = ksp.getIterationNumber()
        ref = spla.spsolve(asm.A.to_scipy().tocsc(), b.array)
        assert np.linalg.norm(x.array - ref) <= 1e-6 * np.linalg.norm(ref)
        pc = ksp._amg
        r = torch.as_tensor(np.random.default_rng(2).standard_normal(asm.layout.n_free)).cuda()
        eager = pc._cycle(0, r.clone())
        z = torch.empty_like(r)
        pc.apply(r, z)
        torch.cuda.synchronize()
        assert torch.equal(z, eager)
        asm.cleanup()
    print(kind, "CG iterations", its, flush=True)
